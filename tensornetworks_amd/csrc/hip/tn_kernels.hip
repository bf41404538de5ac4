// tn_kernels.hip -- CDNA4 (gfx950) kernels for the variational MPS sweep.
//
// * wmix_k     : applies the sparse MPO tensor W[w][w'][m][n] between the GEMMs
//                (coalesced along the trailing bond index).
// * mdot/gemv  : Lanczos re-orthogonalisation (fp64, deterministic reductions).
// * jacobi_k   : one block pair of a one-sided block-Jacobi SVD (fp64).
#include "tn_device.h"

#include <algorithm>
#include <cstring>

namespace tn {

// ---------------------------------------------------------------------------
// MPO mixing.  Bound by HBM for large bonds (D = 1024 FP64: 250 MB in 51 us) and
// by latency below: every entry is a chain offset / value / selector, then the
// data.  The table is staged in LDS first (one latency instead of one per
// entry), and the outputs are spread over the grid's z until about three
// workgroups per CU exist.  Before (one workgroup walking all outputs with the
// table in global memory) and after: transposed FP64 form, D = 8: 11.5 and
// 4.1 us; 320 x 224, d = 2: 15.5 and 7.5 us; D = 256, d = 3: 21.7 and 6.9 us;
// FP32 512 x 448, d = 3: 16.5 and 8.9 us; plain FP64 form, D = 256, d = 2: 6.9
// and 6.4 us.  What comes from LDS is the same for every lane.  In the transposed
// FP32 form, with eight reads per entry, it goes back to scalar registers, so that
// the eight addresses are one scalar sum each (with the offsets left in vector
// registers D = 2048, d = 3 took 160 us, D = 1500 78; now 114 and 63).  In FP64 the
// memory hides the sums and small bonds lose (D = 256, d = 3: 7.0 -> 8.0 us); with one
// read per entry it only lengthens the chain (batched form 48 -> 55 us).  Sums keep
// the table's order.
#define MIX_MAXO 64
#define MIX_MAXE 512
template <typename V> struct MixLds {
    int optr[MIX_MAXO + 1], osel[MIX_MAXO], esel[MIX_MAXE];
    long ooff[MIX_MAXO], eoff[MIX_MAXE];
    V eval[MIX_MAXE];
};
// STG: the table's copy in LDS (nout <= MIX_MAXO, nnz <= MIX_MAXE), else global.
// SCALAR: what comes from LDS goes back to scalar registers
template <typename V, bool STG, bool SCALAR> struct MixView {
    const int *optr_, *osel_, *esel_;
    const long *ooff_, *eoff_;
    const V* eval_;
    static __device__ __forceinline__ int uni(int v)
    {
        if constexpr (STG && SCALAR) return __builtin_amdgcn_readfirstlane(v);
        else return v;
    }
    static __device__ __forceinline__ long uni(long v)
    {
        if constexpr (STG && SCALAR)
            return (long)(uint32_t)uni((int)v) | ((long)uni((int)(v >> 32)) << 32);
        else return v;
    }
    __device__ __forceinline__ int optr(int o) const { return uni(optr_[o]); }
    __device__ __forceinline__ int osel(int o) const { return uni(osel_[o]); }
    __device__ __forceinline__ int esel(int e) const { return uni(esel_[e]); }
    __device__ __forceinline__ long ooff(int o) const { return uni(ooff_[o]); }
    __device__ __forceinline__ long eoff(int e) const { return uni(eoff_[e]); }
    __device__ __forceinline__ V eval(int e) const { return eval_[e]; }
};
template <typename V>
__device__ __forceinline__ const V* mix_values(const MixTable& t)
{
    if constexpr (std::is_same<V, double>::value) return t.eval;
    else return t.evalf;
}
template <typename V, bool STG, bool SCALAR = false>
__device__ __forceinline__ MixView<V, STG, SCALAR> mix_view(const MixTable& t, MixLds<V>* l)
{
    if constexpr (!STG) {
        return MixView<V, STG, SCALAR>{t.optr, t.osel, t.esel, t.ooff, t.eoff, mix_values<V>(t)};
    } else {
        const V* v = mix_values<V>(t);
        const bool idt = t.esel != nullptr;
        for (int i = threadIdx.x; i <= t.nout; i += 256) l->optr[i] = t.optr[i];
        for (int i = threadIdx.x; i < t.nout; i += 256) {
            l->ooff[i] = t.ooff[i];
            l->osel[i] = idt ? t.osel[i] : 0;
        }
        for (int i = threadIdx.x; i < t.nnz; i += 256) {
            l->eoff[i] = t.eoff[i];
            l->eval[i] = v[i];
            l->esel[i] = idt ? t.esel[i] : 0;
        }
        __syncthreads();
        return MixView<V, STG, SCALAR>{l->optr, l->osel, l->esel, l->ooff, l->eoff, l->eval};
    }
}
// grid z for nout outputs over xy workgroups
static int mix_groups(long xy, int nout)
{
    const long z = (768 + xy - 1) / xy;
    return (int)(z < nout ? z : nout);
}

// 64 b times 4 x per workgroup
template <typename TI, typename TO, bool STG>
__global__ void __launch_bounds__(256) wmix_k(const TI* __restrict__ in, long isx, TO* __restrict__ out, long osx,
                                              int X, int Bn, MixTable t)
{
    typedef typename std::conditional<std::is_same<TI, double>::value, double, float>::type acc_t;
    __shared__ typename std::conditional<STG, MixLds<acc_t>, int>::type lds;
    const MixView<acc_t, STG, false> m = mix_view<acc_t, STG>(t, (MixLds<acc_t>*)&lds);
    const int b = blockIdx.x * 64 + (threadIdx.x & 63);
    const long x = (long)blockIdx.y * 4 + (threadIdx.x >> 6);
    if (b >= Bn || x >= X) return;
    const TI* ip = in + x * isx + b;
    TO* op = out + x * osx + b;
    for (int o = blockIdx.z; o < t.nout; o += gridDim.z) {
        const int e0 = m.optr(o), e1 = m.optr(o + 1);
        acc_t acc = 0;
#pragma unroll 4
        for (int e = e0; e < e1; e++) acc += m.eval(e) * to_acc<acc_t>(ip[m.eoff(e)]);
        if constexpr (std::is_same<TI, double>::value) op[m.ooff(o)] = cvt_from_d<TO>(acc);
        else op[m.ooff(o)] = cvt_from_f<TO>(acc);
    }
}

hipError_t wmix(int tin, int tout, const void* in, long isx, void* out, long osx, int X, int Bn,
                const MixTable& t, hipStream_t s)
{
    dim3 grid((Bn + 63) / 64, (X + 3) / 4);
    grid.z = mix_groups((long)grid.x * grid.y, t.nout);
    const bool stg = t.nout <= MIX_MAXO && t.nnz <= MIX_MAXE;
#define WM_CASE(TIc, TOc, TIt, TOt)                                                                             \
    if (tin == TIc && tout == TOc) {                                                                            \
        if (stg) wmix_k<TIt, TOt, true><<<grid, 256, 0, s>>>((const TIt*)in, isx, (TOt*)out, osx, X, Bn, t);    \
        else wmix_k<TIt, TOt, false><<<grid, 256, 0, s>>>((const TIt*)in, isx, (TOt*)out, osx, X, Bn, t);       \
        return hipGetLastError();                                                                               \
    }
    WM_CASE(T_F64, T_F64, double, double)
    WM_CASE(T_F32, T_F32, float, float)
    WM_CASE(T_F32, T_BF16, float, bf16)
    WM_CASE(T_F32, T_F64, float, double)
#undef WM_CASE
    return hipErrorInvalidValue;
}

template <typename TI, typename TX, typename TO, bool X3, bool STG>
__global__ void __launch_bounds__(256) wmix_idt_k(const TI* __restrict__ in, long isx, const TX* __restrict__ in2,
                                                  long isx2, TO* __restrict__ out, long ldo, long ops,
                                                  double* __restrict__ out2, long osx2, int Bn, MixTable t)
{
    typedef typename std::conditional<std::is_same<TI, double>::value, double, float>::type acc_t;
    __shared__ acc_t tile[64][33];
    __shared__ typename std::conditional<STG, MixLds<acc_t>, int>::type lds;
    constexpr bool SCALAR = !std::is_same<TI, double>::value;
    const MixView<acc_t, STG, SCALAR> m = mix_view<acc_t, STG, SCALAR>(t, (MixLds<acc_t>*)&lds);
    const int tb = threadIdx.x & 63, tr = threadIdx.x >> 6;  // b within the tile, row group of 8
    const int b = blockIdx.x * 64 + tb;
    const long x0 = (long)blockIdx.y * 32 + tr * 8;
    const bool bok = b < Bn;
    // writer role: row wb of the tile (b), columns wc..wc+7 (x)
    const int wb = threadIdx.x >> 2, wc = (threadIdx.x & 3) * 8;
    const bool wok = blockIdx.x * 64 + wb < Bn;
    for (int o = blockIdx.z; o < t.nout; o += gridDim.z) {
        const int e0 = m.optr(o), e1 = m.optr(o + 1);
        acc_t acc[8];
#pragma unroll
        for (int r = 0; r < 8; r++) acc[r] = 0;
        if (bok) {
#pragma unroll 2
            for (int e = e0; e < e1; e++) {
                const acc_t v = m.eval(e);
                const long off = m.eoff(e) + b;
                if (m.esel(e)) {
#pragma unroll
                    for (int r = 0; r < 8; r++) acc[r] += v * to_acc<acc_t>(in2[(x0 + r) * isx2 + off]);
                } else {
#pragma unroll
                    for (int r = 0; r < 8; r++) acc[r] += v * to_acc<acc_t>(in[(x0 + r) * isx + off]);
                }
            }
        }
        if (m.osel(o)) {  // identity channel of L: straight into y[x][m][b]
            if (bok) {
#pragma unroll
                for (int r = 0; r < 8; r++) out2[(x0 + r) * osx2 + m.ooff(o) + b] = (double)acc[r];
            }
            continue;
        }
        __syncthreads();  // the previous output's tile has been written out
#pragma unroll
        for (int r = 0; r < 8; r++) tile[tb][tr * 8 + r] = acc[r];
        __syncthreads();
        if (wok) {
            TO* dst = out + m.ooff(o) + (long)(blockIdx.x * 64 + wb) * ldo + (long)blockIdx.y * 32 + wc;
            if constexpr (X3) {
                // three bfloat16 planes, one 16-byte store per plane (8 values;
                // every offset here is a multiple of 8 elements)
                uint32_t h[3][8];
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    bf16 h0, h1, h2;
                    split3_val((float)tile[wb][wc + c], h0, h1, h2);
                    h[0][c] = h0;
                    h[1][c] = h1;
                    h[2][c] = h2;
                }
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    u32x4 w;
                    w.x = h[q][0] | (h[q][1] << 16);
                    w.y = h[q][2] | (h[q][3] << 16);
                    w.z = h[q][4] | (h[q][5] << 16);
                    w.w = h[q][6] | (h[q][7] << 16);
                    *(u32x4*)(dst + q * ops) = w;
                }
            } else {
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    if constexpr (std::is_same<TO, double>::value) dst[c] = (double)tile[wb][wc + c];
                    else dst[c] = cvt_from_f<TO>((float)tile[wb][wc + c]);
                }
            }
        }
    }
}

hipError_t wmix_idt(int tin, int tx, int tout, const void* in, long isx, const void* in2, long isx2, void* out,
                    long ldo, double* out2, long osx2, int X, int Bn, const MixTable& t, hipStream_t s, long ops)
{
    if (!t.esel || !t.osel || X % 32) return hipErrorInvalidValue;
    dim3 grid((Bn + 63) / 64, X / 32);
    grid.z = mix_groups((long)grid.x * grid.y, t.nout);
    const bool stg = t.nout <= MIX_MAXO && t.nnz <= MIX_MAXE;
    if (tout == T_BF16X3 && (tin != T_F32 || tx != T_F64 || ops <= 0 || ops % 8 || ldo % 8)) return hipErrorInvalidValue;
#define WT_CASE(TIc, TXc, TOc, TIt, TXt, TOt, X3)                                                               \
    if (tin == TIc && tx == TXc && tout == TOc) {                                                               \
        if (stg)                                                                                                \
            wmix_idt_k<TIt, TXt, TOt, X3, true><<<grid, 256, 0, s>>>(                                           \
                (const TIt*)in, isx, (const TXt*)in2, isx2, (TOt*)out, ldo, ops, out2, osx2, Bn, t);            \
        else                                                                                                    \
            wmix_idt_k<TIt, TXt, TOt, X3, false><<<grid, 256, 0, s>>>(                                          \
                (const TIt*)in, isx, (const TXt*)in2, isx2, (TOt*)out, ldo, ops, out2, osx2, Bn, t);            \
        return hipGetLastError();                                                                               \
    }
    WT_CASE(T_F32, T_F64, T_BF16X3, float, double, bf16, true)
    WT_CASE(T_F64, T_F64, T_F64, double, double, double, false)
    WT_CASE(T_F32, T_F32, T_F32, float, float, float, false)
    WT_CASE(T_F32, T_BF16, T_BF16, float, bf16, bf16, false)
#undef WT_CASE
    return hipErrorInvalidValue;
}

__global__ void __launch_bounds__(256) publish_k(const double* __restrict__ src, int n, double* host_dst,
                                                 unsigned long long* host_flag, unsigned long long seq)
{
    for (int t = threadIdx.x; t < n; t += 256) host_dst[t] = src[t];
    // every wave orders its own stores at system scope before the barrier;
    // the barrier alone is a workgroup-scope fence, so without this the host
    // could see the flag before the values of waves 1-3
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence_system();
        *(volatile unsigned long long*)host_flag = seq;
    }
}

hipError_t publish(const double* src, int n, double* host_dst, unsigned long long* host_flag,
                   unsigned long long seq, hipStream_t s)
{
    if (n < 0 || n > TN_PUBLISH_MAX) return hipErrorInvalidValue;
    publish_k<<<1, 256, 0, s>>>(src, n, host_dst, host_flag, seq);
    return hipGetLastError();
}

// Words carried in the kernel's arguments: they are copied when the launch is
// queued, so nothing has to wait for the stream (a pageable copy of 256 bytes
// and the wait for it take about 20 us, this launch about 5).
struct Words {
    unsigned w[512];
};
__global__ void __launch_bounds__(256) upload_k(unsigned* __restrict__ dst, Words a, int n)
{
    for (int t = threadIdx.x; t < n; t += 256) dst[t] = a.w[t];
}
hipError_t upload(void* dst, const void* src, long bytes, hipStream_t s)
{
    if (bytes % 4 != 0) return hipErrorInvalidValue;
    Words a;
    for (long off = 0; off < bytes; off += (long)sizeof(a)) {
        const int n = (int)std::min((long)sizeof(a), bytes - off);
        memcpy(a.w, (const char*)src + off, n);
        upload_k<<<1, 256, 0, s>>>((unsigned*)((char*)dst + off), a, n / 4);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// ---------------------------------------------------------------------------
// elementwise
template <typename TI, typename TO>
__global__ void convert_k(const TI* __restrict__ in, TO* __restrict__ out, long n)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256)
        out[i] = cvt_from_d<TO>(to_d(in[i]));
}

hipError_t convert(int tin, const void* in, int tout, void* out, long n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
#define CV_CASE(TIc, TOc, TIt, TOt)                                                           \
    if (tin == TIc && tout == TOc) {                                                          \
        convert_k<TIt, TOt><<<blocks, 256, 0, s>>>((const TIt*)in, (TOt*)out, n);             \
        return hipGetLastError();                                                             \
    }
    CV_CASE(T_F64, T_F32, double, float)
    CV_CASE(T_F64, T_BF16, double, bf16)
    CV_CASE(T_F32, T_F64, float, double)
    CV_CASE(T_BF16, T_F64, bf16, double)
    CV_CASE(T_F64, T_F64, double, double)
#undef CV_CASE
    return hipErrorInvalidValue;
}

template <typename TI>
__global__ void split3_k(const TI* __restrict__ in, bf16* __restrict__ out, long n, long ps)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        bf16 h0, h1, h2;
        split3_val(in[i], h0, h1, h2);
        out[i] = h0;
        out[ps + i] = h1;
        out[2 * ps + i] = h2;
    }
}

hipError_t split3(int tin, const void* in, void* out, long n, long ps, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    if (ps < n) return hipErrorInvalidValue;
    long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    if (tin == T_F64) split3_k<double><<<blocks, 256, 0, s>>>((const double*)in, (bf16*)out, n, ps);
    else if (tin == T_F32) split3_k<float><<<blocks, 256, 0, s>>>((const float*)in, (bf16*)out, n, ps);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// x <- a x in place, and the three bfloat16 planes of the scaled values
// (the Lanczos scaling of the next basis vector fused into the apply's first
// pass over it; a x rounds exactly as the separate scaling would)
__global__ void split3_scale_k(double* __restrict__ x, double a, bf16* __restrict__ out, long n, long ps)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        const double v = a * x[i];
        x[i] = v;
        bf16 h0, h1, h2;
        split3_val(v, h0, h1, h2);
        out[i] = h0;
        out[ps + i] = h1;
        out[2 * ps + i] = h2;
    }
}
hipError_t split3_scale(double* x, double a, void* out, long n, long ps, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    if (ps < n) return hipErrorInvalidValue;
    long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    split3_scale_k<<<blocks, 256, 0, s>>>(x, a, (bf16*)out, n, ps);
    return hipGetLastError();
}
// x <- a x in place, and the scaled values converted to TO
template <typename TO>
__global__ void convert_scale_k(double* __restrict__ x, double a, TO* __restrict__ out, long n)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        const double v = a * x[i];
        x[i] = v;
        out[i] = cvt_from_d<TO>(v);
    }
}
hipError_t convert_scale(double* x, double a, int tout, void* out, long n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    if (tout == T_F32) convert_scale_k<float><<<blocks, 256, 0, s>>>(x, a, (float*)out, n);
    else if (tout == T_BF16) convert_scale_k<bf16><<<blocks, 256, 0, s>>>(x, a, (bf16*)out, n);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

__global__ void fill_zero_k(uint32_t* p, long n)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256) p[i] = 0u;
}
hipError_t fill_zero(void* p, long bytes, hipStream_t s)
{
    if (bytes <= 0) return hipSuccess;
    long n = bytes / 4;
    long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    fill_zero_k<<<blocks, 256, 0, s>>>((uint32_t*)p, n);
    return hipGetLastError();
}
__global__ void fill_value_k(double* p, double v, long n)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256) p[i] = v;
}
hipError_t fill_value(double* p, double v, long n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    fill_value_k<<<blocks, 256, 0, s>>>(p, v, n);
    return hipGetLastError();
}

// out[c*ldo + r] = (r < R && c < C) ? in[r*ldi + c] : 0, for r < Ro, c < Co,
// through a 32 x 32 LDS tile so that reads and writes are both coalesced
// (D = 1024, d = 3, 50 MB moved: 23 and 17 us, read or written with a stride,
// against 10.6 us tiled)
__global__ void __launch_bounds__(256) transpose_k(const double* __restrict__ in, long ldi, int R, int C,
                                                   double* __restrict__ out, long ldo, int Ro, int Co)
{
    __shared__ double tile[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
#pragma unroll
    for (int i = 0; i < 32; i += 8) {
        const int r = r0 + ty + i, c = c0 + tx;
        tile[ty + i][tx] = (r < R && c < C) ? in[(long)r * ldi + c] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 32; i += 8) {
        const int c = c0 + ty + i, r = r0 + tx;
        if (r < Ro && c < Co) out[(long)c * ldo + r] = tile[tx][ty + i];
    }
}
static hipError_t transpose(const double* in, long ldi, int R, int C, double* out, long ldo, int Ro, int Co,
                            hipStream_t s)
{
    transpose_k<<<dim3((Co + 31) / 32, (Ro + 31) / 32), 256, 0, s>>>(in, ldi, R, C, out, ldo, Ro, Co);
    return hipGetLastError();
}

// site tensor layouts: reference psi[m + d*(a + D1*b)] is the matrix (b, (a, m)),
// internal [D1p][d][D2p] the matrix ((a, m), b): transposes of each other, with
// zero padding on the internal side
hipError_t psi_ref_to_int(const double* ref, double* out, int d, int D1, int D2, int D1p, int D2p, hipStream_t s)
{
    if (d <= 0 || D1 <= 0 || D2 <= 0 || D1p < D1 || D2p < D2) return hipErrorInvalidValue;
    return transpose(ref, (long)d * D1, D2, d * D1, out, D2p, D2p, d * D1p, s);
}

// psi_ref_to_int with the operand of a reduced-precision apply formed in the same
// pass: lo (FP32, BF16, or three BF16 planes ps apart, the values of convert and
// split3) and, for the planes, whose MPO stage reads x itself, the FP64 copy.  One
// launch instead of two (about 2 us of 33 at D = 42) and one pass over x less
// (D = 1024, d = 3: 5 + 10 us as two kernels).
template <typename TO, bool X3>
__global__ void __launch_bounds__(256) transpose_lo_k(const double* __restrict__ in, long ldi, int R, int C,
                                                      double* __restrict__ out, TO* __restrict__ lo, long ps, long ldo,
                                                      int Ro, int Co)
{
    __shared__ double tile[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
#pragma unroll
    for (int i = 0; i < 32; i += 8) {
        const int r = r0 + ty + i, c = c0 + tx;
        tile[ty + i][tx] = (r < R && c < C) ? in[(long)r * ldi + c] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 32; i += 8) {
        const int c = c0 + ty + i, r = r0 + tx;
        if (r >= Ro || c >= Co) continue;
        const long o = (long)c * ldo + r;
        const double v = tile[tx][ty + i];
        if constexpr (X3) {
            bf16 h0, h1, h2;
            split3_val(v, h0, h1, h2);
            out[o] = v;
            lo[o] = h0;
            lo[ps + o] = h1;
            lo[2 * ps + o] = h2;
        } else {
            lo[o] = cvt_from_d<TO>(v);
        }
    }
}
hipError_t psi_ref_to_int_lo(const double* ref, int tlo, double* out, void* lo, int d, int D1, int D2, int D1p, int D2p,
                             hipStream_t s)
{
    if (d <= 0 || D1 <= 0 || D2 <= 0 || D1p < D1 || D2p < D2) return hipErrorInvalidValue;
    const int R = D2, C = d * D1, Ro = D2p, Co = d * D1p;
    const long ps = (long)Ro * Co;
    const dim3 grid((Co + 31) / 32, (Ro + 31) / 32);
    if (tlo == T_BF16X3) transpose_lo_k<bf16, true><<<grid, 256, 0, s>>>(ref, C, R, C, out, (bf16*)lo, ps, D2p, Ro, Co);
    else if (tlo == T_BF16) transpose_lo_k<bf16, false><<<grid, 256, 0, s>>>(ref, C, R, C, out, (bf16*)lo, ps, D2p, Ro, Co);
    else if (tlo == T_F32) transpose_lo_k<float, false><<<grid, 256, 0, s>>>(ref, C, R, C, out, (float*)lo, ps, D2p, Ro, Co);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
hipError_t psi_int_to_ref(const double* in, double* ref, int d, int D1, int D2, int D2p, hipStream_t s)
{
    if (d <= 0 || D1 <= 0 || D2 <= 0 || D2p < D2) return hipErrorInvalidValue;
    return transpose(in, D2p, d * D1, D2, ref, (long)d * D1, d * D1, D2, s);
}

__global__ void copy3_k(const double* __restrict__ in, long si, long sj, long sk,
                        double* __restrict__ out, int n1, int n2, int n2o)
{
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n2o) return;
    const int j = blockIdx.y, i = blockIdx.z;
    out[((long)i * n1 + j) * n2o + k] = (k < n2) ? in[i * si + j * sj + k * sk] : 0.0;
}
hipError_t copy3(const double* in, long si, long sj, long sk, double* out, int n0, int n1,
                 int n2, int n2o, hipStream_t s)
{
    if (n0 <= 0 || n1 <= 0 || n2o <= 0) return hipSuccess;
    dim3 grid((n2o + 255) / 256, n1, n0);
    copy3_k<<<grid, 256, 0, s>>>(in, si, sj, sk, out, n1, n2, n2o);
    return hipGetLastError();
}

__global__ void copy2_k(const double* __restrict__ in, long si0, long si1, int r, int c,
                        double* __restrict__ out, long so0, long so1, int co)
{
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= co) return;
    const int i = blockIdx.y;
    out[i * so0 + j * so1] = (i < r && j < c) ? in[i * si0 + j * si1] : 0.0;
}
hipError_t copy2(const double* in, long si0, long si1, int r, int c, double* out, long so0,
                 long so1, int ro, int co, hipStream_t s)
{
    if (ro <= 0 || co <= 0) return hipSuccess;
    if (si1 == 1 && so0 == 1 && so1 != 1) return transpose(in, si0, r, c, out, so1, ro, co, s);
    if (si0 == 1 && so1 == 1 && si1 != 1) return transpose(in, si1, c, r, out, so0, co, ro, s);
    dim3 grid((co + 255) / 256, ro);
    copy2_k<<<grid, 256, 0, s>>>(in, si0, si1, r, c, out, so0, so1, co);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Lanczos vector kernels
#define MD_BLOCK 256
#define MD_EPT 8
#define MD_MAXK 512

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

long mdot_part_size(long n, int k)
{
    long blocks = (n + MD_BLOCK * MD_EPT - 1) / (MD_BLOCK * MD_EPT);
    return blocks * (long)k;
}

// stage 1: part[i*G + blk] = sum over the block's chunk of V[i]*w
__global__ void __launch_bounds__(MD_BLOCK) mdot1_k(const double* __restrict__ V, long ldv, int k,
                                                    const double* __restrict__ w, long n,
                                                    double* __restrict__ part)
{
    __shared__ double red[MD_MAXK][MD_BLOCK / 64];
    const long base = (long)blockIdx.x * MD_BLOCK * MD_EPT + threadIdx.x;
    double wr[MD_EPT];
#pragma unroll
    for (int e = 0; e < MD_EPT; e++) {
        long idx = base + (long)e * MD_BLOCK;
        wr[e] = idx < n ? w[idx] : 0.0;
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int i = 0; i < k; i++) {
        const double* vi = V + (long)i * ldv;
        double acc = 0.0;
#pragma unroll
        for (int e = 0; e < MD_EPT; e++) {
            long idx = base + (long)e * MD_BLOCK;
            if (idx < n) acc += vi[idx] * wr[e];
        }
        acc = wave_sum(acc);
        if (lane == 0) red[i][wid] = acc;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < k; i += MD_BLOCK) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < MD_BLOCK / 64; q++) s += red[i][q];
        part[(long)i * gridDim.x + blockIdx.x] = s;
    }
}

// stage 2: out[i] = sum_b part[i*G + b]  (one block per i, fixed order)
__global__ void __launch_bounds__(256) mdot2_k(const double* __restrict__ part, int G,
                                               double* __restrict__ out)
{
    __shared__ double red[4];
    const int i = blockIdx.x;
    double acc = 0.0;
    for (int b = threadIdx.x; b < G; b += 256) acc += part[(long)i * G + b];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) out[i] = red[0] + red[1] + red[2] + red[3];
}

hipError_t mdot(const double* V, long ldv, int k, const double* w, long n, double* out,
                double* part, int part_cap, hipStream_t s)
{
    if (k <= 0) return hipSuccess;
    long G = (n + MD_BLOCK * MD_EPT - 1) / (MD_BLOCK * MD_EPT);
    for (int i0 = 0; i0 < k; i0 += MD_MAXK) {
        const int kc = (k - i0) < MD_MAXK ? (k - i0) : MD_MAXK;
        if (G * kc > part_cap) return hipErrorInvalidValue;
        mdot1_k<<<G, MD_BLOCK, 0, s>>>(V + (long)i0 * ldv, ldv, kc, w, n, part);
        mdot2_k<<<kc, 256, 0, s>>>(part, (int)G, out + i0);
    }
    return hipGetLastError();
}

// One Lanczos step is four launches (lz_dot, lz_step, lz_update, lz_publish):
// each kernel sums the partial results of the one before it in its own
// prologue, in a fixed order, so no reduction has a launch of its own.  Bound
// by launches and load latency up to n ~ 1e5, by the last-level cache or HBM
// beyond; the grid of lz_step splits the basis vectors as well as the entries
// (one workgroup per 2048 entries, taking the vectors one after the other,
// left 45 of 256 CUs busy at n = 92160).  Measured for the vector part of an
// iteration with a pass against k vectors, that form (with a second launch per
// reduction) and this one: n = 2048, k ~ 28: 58 and 15 us; n = 92160, k ~ 84:
// 224 and 43 us (the 62 MB basis read twice: 2.9 TB/s); n = 196608, k = 2
// (partial re-orthogonalisation): 33 and 22 us.  lz_step has its first eight
// vectors in flight while it sums alpha: 25 -> 19 us at n = 92160, k ~ 84, 9.5 ->
// 5.9 us at n = 18432, k ~ 12.
#define LZ_SMALL 131072  // entries up to which chunks are sized for latency

// entry pairs per thread of lz_step: one while the vectors are short or few (a
// workgroup per 512 entries), else four (2048 entries; up to LZ_SMALL at most
// 64 partial sums per coefficient, which lz_update sums by one thread each)
static inline int lz_step_pairs(long n, int k) { return n <= 8192 || (n <= LZ_SMALL && k <= 8) ? 1 : 4; }
static inline long lz_step_blocks(long n, int k)
{
    const long c = 2L * MD_BLOCK * lz_step_pairs(n, k);
    return (n + c - 1) / c;
}
static inline long lz_dot_blocks(long n)
{
    const long c = n <= LZ_SMALL ? 2L * MD_BLOCK : 8L * MD_BLOCK;
    return (n + c - 1) / c;
}
static inline long lz_norm_blocks(long n)
{
    const long c = n <= LZ_SMALL ? 128 : 8L * MD_BLOCK;
    return (n + c - 1) / c;
}
long lz_part_size(long n, int k)
{
    const long few = lz_step_blocks(n, 1) * (k < 8 ? k : 8), all = lz_step_blocks(n, k) * (long)k;
    return lz_dot_blocks(n) + lz_norm_blocks(n) + (few > all ? few : all);
}

// sum of acc, or of v[0..n), over the workgroup (MD_BLOCK threads), the same on every
// thread
__device__ __forceinline__ double block_total(double acc, double* red)
{
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}
__device__ __forceinline__ double block_sum(const double* __restrict__ v, int n, double* red)
{
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += MD_BLOCK) acc += v[i];
    return block_total(acc, red);
}

template <int P>
__global__ void __launch_bounds__(MD_BLOCK) lz_dot_k(const double* __restrict__ v, const double* __restrict__ w,
                                                     long n, double* __restrict__ part)
{
    __shared__ double red[4];
    double acc = 0.0;
#pragma unroll
    for (int e = 0; e < P; e++) {
        const long idx = 2 * ((long)(blockIdx.x * P + e) * MD_BLOCK + threadIdx.x);
        if (idx < n) {
            const double2 a = *(const double2*)(v + idx), b = *(const double2*)(w + idx);
            acc += a.x * b.x + a.y * b.y;
        }
    }
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// na > 0: alpha = sum apart[0..na), w <- y - alpha V_{k-1} - beta V_{k-2} (the
// latter when k >= 2), alpha to aout[0]; na = 0: w is read as it is.  Then
// part[i*gridDim.x + block] = V_i . w over the block's entries, for the ng
// vectors i of block row blockIdx.y (w is formed by every block row, written
// by the first: y and w are different buffers).
template <int P, int U>
__global__ void __launch_bounds__(MD_BLOCK) lz_step_k(const double* __restrict__ y, double* __restrict__ w,
                                                      const double* __restrict__ V, long ldv, int k,
                                                      const double* __restrict__ apart, int na,
                                                      double* __restrict__ aout, double beta, long n, int ng,
                                                      double* __restrict__ part)
{
    __shared__ double ared[4];
    __shared__ double red[2][U][4];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const long c0 = (long)blockIdx.x * 2 * MD_BLOCK * P;
    const int i1 = min(k, (int)(blockIdx.y + 1) * ng);
    // U vectors at a time: their loads and their lane reductions are independent
    double2 v[U][P];
    auto load = [&](int i0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const double* vi = V + (long)(i0 + u) * ldv;
#pragma unroll
            for (int e = 0; e < P; e++) {
                const long idx = c0 + 2 * (e * MD_BLOCK + tid);
                v[u][e] = i0 + u < i1 && idx < n ? *(const double2*)(vi + idx) : make_double2(0.0, 0.0);
            }
        }
    };
    double2 x[P];
    if (na > 0) {
        double asum = 0.0;
        for (int i = tid; i < na; i += MD_BLOCK) asum += apart[i];
        const double* vj = V + (long)(k - 1) * ldv;
        const double* vm = k >= 2 ? V + (long)(k - 2) * ldv : vj;
        const double b = k >= 2 ? beta : 0.0;
        double2 p[P], q[P];
#pragma unroll
        for (int e = 0; e < P; e++) {
            const long idx = c0 + 2 * (e * MD_BLOCK + tid);
            const bool in = idx < n;
            x[e] = in ? *(const double2*)(y + idx) : make_double2(0.0, 0.0);
            p[e] = in ? *(const double2*)(vj + idx) : make_double2(0.0, 0.0);
            q[e] = in ? *(const double2*)(vm + idx) : make_double2(0.0, 0.0);
        }
        load(blockIdx.y * ng);  // in flight while alpha is summed
        const double a = block_total(asum, ared);
        if (blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) aout[0] = a;
#pragma unroll
        for (int e = 0; e < P; e++) {
            x[e].x -= a * p[e].x;
            x[e].y -= a * p[e].y;
            x[e].x -= b * q[e].x;
            x[e].y -= b * q[e].y;
            const long idx = c0 + 2 * (e * MD_BLOCK + tid);
            if (blockIdx.y == 0 && idx < n) *(double2*)(w + idx) = x[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < P; e++) {
            const long idx = c0 + 2 * (e * MD_BLOCK + tid);
            x[e] = idx < n ? *(const double2*)(w + idx) : make_double2(0.0, 0.0);
        }
        load(blockIdx.y * ng);
    }
    int par = 0;
    for (int i0 = blockIdx.y * ng; i0 < i1; i0 += U, par ^= 1) {
        double acc[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            double s = 0.0;
#pragma unroll
            for (int e = 0; e < P; e++) s += v[u][e].x * x[e].x + v[u][e].y * x[e].y;
            acc[u] = s;
        }
        if (i0 + U < i1) load(i0 + U);
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1)
#pragma unroll
            for (int u = 0; u < U; u++) acc[u] += __shfl_xor(acc[u], o, 64);
        if (lane == 0) {
#pragma unroll
            for (int u = 0; u < U; u++) red[par][u][wid] = acc[u];
        }
        __syncthreads();  // the other slot of red is read before the next round's barrier
        if (tid < U && i0 + tid < i1)
            part[(long)(i0 + tid) * gridDim.x + blockIdx.x] =
                (red[par][tid][0] + red[par][tid][1]) + (red[par][tid][2] + red[par][tid][3]);
    }
}

// c_i = sum_b part[i*G + b] (G > 0; written to coef by the first workgroup) or
// coef[i] (G = 0); w <- w - sum_{i<k} c_i V_i; npart[block] = |w|^2 over the
// block's entries.  KG groups of MD_BLOCK / KG threads take every KG-th
// vector, each thread P pairs of entries: (4, 1) for short vectors (128
// entries per workgroup), (1, 4) for long ones.  Workgroups walk the entries in
// the reverse order of lz_step, whose last reads of the basis are still in the
// last-level cache when the basis exceeds it.
template <int KG, int P>
__global__ void __launch_bounds__(MD_BLOCK) lz_update_k(double* __restrict__ w, const double* __restrict__ V,
                                                        long ldv, int k, const double* __restrict__ part, int G,
                                                        double* __restrict__ coef, long n,
                                                        double* __restrict__ npart)
{
    constexpr int TG = MD_BLOCK / KG;
    __shared__ double c[MD_MAXK];
    __shared__ double2 sub[KG][TG * P];
    __shared__ double red[4];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int t = tid % TG, kg = tid / TG;
    if (G == 0) {
        for (int i = tid; i < k; i += MD_BLOCK) c[i] = coef[i];
    } else if (G <= 64) {
        for (int i = tid; i < k; i += MD_BLOCK) {
            double s = 0.0;
#pragma unroll 8
            for (int b = 0; b < G; b++) s += part[(long)i * G + b];
            c[i] = s;
        }
    } else {
        for (int i = wid; i < k; i += 4) {
            double s = 0.0;
            for (int b = lane; b < G; b += 64) s += part[(long)i * G + b];
            s = wave_sum(s);
            if (lane == 0) c[i] = s;
        }
    }
    __syncthreads();
    if (G > 0 && blockIdx.x == 0)
        for (int i = tid; i < k; i += MD_BLOCK) coef[i] = c[i];
    const int blk = gridDim.x - 1 - blockIdx.x;
    const long c0 = (long)blk * 2 * TG * P;
    double2 acc[P];
#pragma unroll
    for (int e = 0; e < P; e++) acc[e] = make_double2(0.0, 0.0);
#pragma unroll 4
    for (int i = kg; i < k; i += KG) {
        const double* vi = V + (long)i * ldv;
        const double ci = c[i];
#pragma unroll
        for (int e = 0; e < P; e++) {
            const long idx = c0 + 2 * ((long)e * TG + t);
            if (idx < n) {
                const double2 p = *(const double2*)(vi + idx);
                acc[e].x += ci * p.x;
                acc[e].y += ci * p.y;
            }
        }
    }
    if constexpr (KG > 1) {
#pragma unroll
        for (int e = 0; e < P; e++) sub[kg][e * TG + t] = acc[e];
        __syncthreads();
    }
    double sq = 0.0;
    if (kg == 0) {
#pragma unroll
        for (int e = 0; e < P; e++) {
            const long idx = c0 + 2 * ((long)e * TG + t);
            if (idx < n) {
                double2 x = *(const double2*)(w + idx);
                double2 s = acc[e];
                if constexpr (KG > 1) {
#pragma unroll
                    for (int g = 1; g < KG; g++) {
                        const double2 o = sub[g][e * TG + t];
                        s.x += o.x;
                        s.y += o.y;
                    }
                }
                x.x -= s.x;
                x.y -= s.y;
                *(double2*)(w + idx) = x;
                sq += x.x * x.x + x.y * x.y;
            }
        }
    }
    sq = wave_sum(sq);
    if (lane == 0) red[wid] = sq;
    __syncthreads();
    if (tid == 0) npart[blk] = (red[0] + red[1]) + (red[2] + red[3]);
}

hipError_t lz_dot(const double* v, const double* w, long n, double* part, hipStream_t s)
{
    if (n <= 0 || (n & 1)) return hipErrorInvalidValue;
    const int G = (int)lz_dot_blocks(n);
    if (n <= LZ_SMALL) lz_dot_k<1><<<G, MD_BLOCK, 0, s>>>(v, w, n, part);
    else lz_dot_k<4><<<G, MD_BLOCK, 0, s>>>(v, w, n, part);
    return hipGetLastError();
}

hipError_t lz_step(const double* y, double* w, const double* V, long ldv, int k, bool three, double beta, long n,
                   double* h, double* part, hipStream_t s)
{
    if (k < 1 || k > MD_MAXK || n <= 0 || (n & 1) || (three && y == w)) return hipErrorInvalidValue;
    const long G = lz_step_blocks(n, k), na = lz_dot_blocks(n);
    double* dots = part + na + lz_norm_blocks(n);
    // block rows of eight or more vectors each until the chip is full
    const int groups = (k + 7) / 8;
    const int S = (int)(G >= 512 ? 1 : (512 / G < groups ? 512 / G : groups));
    const int ng = 8 * ((groups + S - 1) / S);
    const dim3 grid(G, (k + ng - 1) / ng);
    const int nap = three ? (int)na : 0;
    // one or two vectors (partial re-orthogonalisation): room for two only, so that
    // more workgroups of the long streams fit on a CU (with room for eight a sweep at
    // D = 1024, n = 3.1e6, took 2.15 s, with two 2.07 s)
    if (lz_step_pairs(n, k) == 1) lz_step_k<1, 8><<<grid, MD_BLOCK, 0, s>>>(y, w, V, ldv, k, part, nap, h, beta, n, ng, dots);
    else if (k <= 2) lz_step_k<4, 2><<<grid, MD_BLOCK, 0, s>>>(y, w, V, ldv, k, part, nap, h, beta, n, ng, dots);
    else lz_step_k<4, 8><<<grid, MD_BLOCK, 0, s>>>(y, w, V, ldv, k, part, nap, h, beta, n, ng, dots);
    return hipGetLastError();
}

hipError_t lz_update(double* w, const double* V, long ldv, int k, long n, double* coef, double* part, hipStream_t s)
{
    if (k < 1 || k > MD_MAXK || n <= 0 || (n & 1)) return hipErrorInvalidValue;
    int G = (int)lz_step_blocks(n, k);
    double* npart = part + lz_dot_blocks(n);
    double* dots = npart + lz_norm_blocks(n);
    // summing the partial dots in every workgroup costs k*G reads each: for
    // long vectors and more than a few coefficients a launch of its own is
    // cheaper
    if (G > 64 && k > 8) {
        mdot2_k<<<k, 256, 0, s>>>(dots, G, coef);
        G = 0;
    }
    const int Gn = (int)lz_norm_blocks(n);
    if (n <= LZ_SMALL) lz_update_k<4, 1><<<Gn, MD_BLOCK, 0, s>>>(w, V, ldv, k, dots, G, coef, n, npart);
    else lz_update_k<1, 4><<<Gn, MD_BLOCK, 0, s>>>(w, V, ldv, k, dots, G, coef, n, npart);
    return hipGetLastError();
}

// The whole step of a short vector in one workgroup: scales v_j = V_{k-1} by
// vscale first when that is not 1 (in place), then alpha, the three-term step,
// the pass against V_0 .. V_{k-1}, |w|^2, and the publication of (alpha,
// coefficients, |w|^2).
// w goes to V_k, divided by |w| when `unit`.  w stays in registers (PP pairs
// per thread) and in LDS, where every wave takes whole vectors of the basis:
// one lane reduction per vector instead of one per vector and wave.  Bound by
// the one CU's reads of the basis (two passes), so it pays while that is small
// (lz_small_ok).  This launch and the four of the split step, launch after launch:
// n = 1024: 9.0 and 12.3 us at k = 1, 14.1 and 13.8 at 32, 17.3 and 14.3 at 48;
// n = 2048: 9.0 and 12.5 at 1, 12.5 and 13.7 at 16, 16.3 and 14.1 at 32;
// n = 4096: 10.3 and 13.2 at 1, 13.3 and 13.6 at 8, 17.2 and 13.8 at 16;
// n = 6144: 11.8 and 13.7 at 1, 13.4 and 13.9 at 4, 16.2 and 14.2 at 8 (12288: 23 at 2).
// They cross near n k = 32768.
#define LZ_TINY_T 1024
#define LZ_TINY_K 64
#define LZ_TINY_N (6 * LZ_TINY_T)
bool lz_small_ok(long n, int k) { return n > 0 && n % 128 == 0 && n <= LZ_TINY_N && k >= 1 && k <= LZ_TINY_K && n * k <= 32768; }

template <int PP>
__global__ void __launch_bounds__(LZ_TINY_T) lz_small_k(const double* __restrict__ y, double* __restrict__ V, long ldv,
                                                        int k, double vscale, double beta, int unit, int n,
                                                        double* host_dst, unsigned long long* host_flag,
                                                        unsigned long long seq)
{
    constexpr int NW = LZ_TINY_T / 64;
    __shared__ __attribute__((aligned(16))) double ws[2 * PP * LZ_TINY_T];
    __shared__ double one[2][NW];
    __shared__ double c[LZ_TINY_K];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    double* vj = V + (long)(k - 1) * ldv;
    const double* vm = k >= 2 ? vj - ldv : vj;
    const double b = k >= 2 ? beta : 0.0;
    auto total = [&](double v, double* buf) {  // sum over the workgroup
        v = wave_sum(v);
        if (lane == 0) buf[wid] = v;
        __syncthreads();
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < NW; q++) s += buf[q];
        return s;
    };
    double2 x[PP], p[PP], q[PP];
#pragma unroll
    for (int e = 0; e < PP; e++) {
        const int idx = 2 * (e * LZ_TINY_T + tid);
        const bool in = idx < n;
        x[e] = in ? *(const double2*)(y + idx) : make_double2(0.0, 0.0);
        p[e] = in ? *(const double2*)(vj + idx) : make_double2(0.0, 0.0);
        q[e] = in ? *(const double2*)(vm + idx) : make_double2(0.0, 0.0);
    }
    double dot = 0.0;
#pragma unroll
    for (int e = 0; e < PP; e++) {
        const int idx = 2 * (e * LZ_TINY_T + tid);
        if (vscale != 1.0) {
            p[e].x *= vscale;
            p[e].y *= vscale;
            if (idx < n) *(double2*)(vj + idx) = p[e];
        }
        dot += x[e].x * p[e].x + x[e].y * p[e].y;
    }
    const double alpha = total(dot, one[0]);
#pragma unroll
    for (int e = 0; e < PP; e++) {
        x[e].x -= alpha * p[e].x;
        x[e].y -= alpha * p[e].y;
        x[e].x -= b * q[e].x;
        x[e].y -= b * q[e].y;
        *(double2*)(ws + 2 * (e * LZ_TINY_T + tid)) = x[e];
    }
    __syncthreads();  // w in LDS; the scaled v_j is visible to every wave
    for (int i = wid; i < k; i += NW) {
        const double* vi = V + (long)i * ldv;
        double s = 0.0;
#pragma unroll 16
        for (int e = 0; e < n / 128; e++) {
            const int idx = 2 * (e * 64 + lane);
            const double2 v = *(const double2*)(vi + idx), w = *(const double2*)(ws + idx);
            s += v.x * w.x + v.y * w.y;
        }
        s = wave_sum(s);
        if (lane == 0) {
            c[i] = s;
            host_dst[1 + i] = s;
        }
    }
    __syncthreads();
#pragma unroll 8
    for (int i = 0; i < k; i++) {
        const double* vi = V + (long)i * ldv;
        const double ci = c[i];
#pragma unroll
        for (int e = 0; e < PP; e++) {
            const int idx = 2 * (e * LZ_TINY_T + tid);
            if (idx < n) {
                const double2 v = *(const double2*)(vi + idx);
                x[e].x -= ci * v.x;
                x[e].y -= ci * v.y;
            }
        }
    }
    double sq = 0.0;
#pragma unroll
    for (int e = 0; e < PP; e++) sq += x[e].x * x[e].x + x[e].y * x[e].y;
    const double nn = total(sq, one[1]);
    const double f = unit ? 1.0 / sqrt(nn) : 1.0;  // infinite when the Krylov space is complete: w is not used then
    double* w = vj + ldv;
#pragma unroll
    for (int e = 0; e < PP; e++) {
        const int idx = 2 * (e * LZ_TINY_T + tid);
        if (idx < n) *(double2*)(w + idx) = make_double2(f * x[e].x, f * x[e].y);
    }
    if (tid == 0) {
        host_dst[0] = alpha;
        host_dst[k + 1] = nn;
    }
    // the published values (each written by lane 0 of a wave) before the flag
    __threadfence_system();
    __syncthreads();
    if (tid == 0) {
        __threadfence_system();
        *(volatile unsigned long long*)host_flag = seq;
    }
}

hipError_t lz_small(const double* y, double* V, long ldv, int k, double vscale, double beta, bool unit, long n,
                    double* host_dst, unsigned long long* host_flag, unsigned long long seq, hipStream_t s)
{
    if (!lz_small_ok(n, k)) return hipErrorInvalidValue;
    const int pp = (int)((n + 2 * LZ_TINY_T - 1) / (2 * LZ_TINY_T));
#define LZ_CASE(P)                                                                                             \
    if (pp <= P) {                                                                                             \
        lz_small_k<P><<<1, LZ_TINY_T, 0, s>>>(y, V, ldv, k, vscale, beta, unit, (int)n, host_dst, host_flag,   \
                                              seq);                                                            \
        return hipGetLastError();                                                                              \
    }
    LZ_CASE(1) LZ_CASE(2) LZ_CASE(3)
#undef LZ_CASE
    return hipErrorInvalidValue;
}

// h[0..nh) and then sum npart[0..G) (|w|^2) to the host, as publish does
__global__ void __launch_bounds__(MD_BLOCK) lz_publish_k(const double* __restrict__ h, int nh,
                                                         const double* __restrict__ npart, int G, double* host_dst,
                                                         unsigned long long* host_flag, unsigned long long seq)
{
    __shared__ double red[4];
    const double nn = block_sum(npart, G, red);
    for (int t = threadIdx.x; t < nh; t += MD_BLOCK) host_dst[t] = h[t];
    if (threadIdx.x == 0) host_dst[nh] = nn;
    __threadfence_system();  // every wave's stores before the flag (see publish_k)
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence_system();
        *(volatile unsigned long long*)host_flag = seq;
    }
}

// The same with w <- w / |w|: every workgroup forms |w|^2 from npart as the first
// one does for the host, so the next apply can be queued on w before the host has
// seen |w| (one launch for the publication and the scaling: 4.8 us at n = 92160,
// 6.8 us for the two; no wait between this step and the next apply).
__global__ void __launch_bounds__(MD_BLOCK) lz_publish_unit_k(const double* __restrict__ h, int nh,
                                                              const double* __restrict__ npart, int G,
                                                              double* __restrict__ w, long n, double* host_dst,
                                                              unsigned long long* host_flag, unsigned long long seq)
{
    __shared__ double red[4];
    const long i = 2 * (blockIdx.x * (long)MD_BLOCK + threadIdx.x);
    double2 x = i < n ? *(const double2*)(w + i) : make_double2(0.0, 0.0);
    const double nn = block_sum(npart, G, red);
    if (blockIdx.x == 0) {
        for (int t = threadIdx.x; t < nh; t += MD_BLOCK) host_dst[t] = h[t];
        if (threadIdx.x == 0) host_dst[nh] = nn;
        __threadfence_system();  // every wave's stores before the flag (see publish_k)
        __syncthreads();
        if (threadIdx.x == 0) {
            __threadfence_system();
            *(volatile unsigned long long*)host_flag = seq;
        }
    }
    const double f = 1.0 / sqrt(nn);  // infinite when the Krylov space is complete: w is not used then
    x.x *= f;
    x.y *= f;
    if (i < n) *(double2*)(w + i) = x;
}

hipError_t lz_publish_unit(const double* h, int nh, double* w, long n, const double* part, double* host_dst,
                           unsigned long long* host_flag, unsigned long long seq, hipStream_t s)
{
    if (nh < 0 || nh >= TN_PUBLISH_MAX || n <= 0 || (n & 1)) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)((n + 2 * MD_BLOCK - 1) / (2 * MD_BLOCK));
    lz_publish_unit_k<<<grid, MD_BLOCK, 0, s>>>(h, nh, part + lz_dot_blocks(n), (int)lz_norm_blocks(n), w, n, host_dst,
                                                host_flag, seq);
    return hipGetLastError();
}

hipError_t lz_publish(const double* h, int nh, long n, const double* part, double* host_dst,
                      unsigned long long* host_flag, unsigned long long seq, hipStream_t s)
{
    if (nh < 0 || nh >= TN_PUBLISH_MAX) return hipErrorInvalidValue;
    lz_publish_k<<<1, MD_BLOCK, 0, s>>>(h, nh, part + lz_dot_blocks(n), (int)lz_norm_blocks(n), host_dst, host_flag,
                                        seq);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256) gemv_acc_k(const double* __restrict__ V, long ldv, int k,
                                                  const double* __restrict__ coef,
                                                  double coef_scale, double beta_w,
                                                  double* __restrict__ w, long n)
{
    __shared__ double c[MD_MAXK];
    for (int i = threadIdx.x; i < k; i += 256) c[i] = coef[i] * coef_scale;
    __syncthreads();
    for (long idx = blockIdx.x * 256L + threadIdx.x; idx < n; idx += (long)gridDim.x * 256) {
        double acc = (beta_w == 0.0) ? 0.0 : beta_w * w[idx];
        for (int i = 0; i < k; i++) acc += c[i] * V[(long)i * ldv + idx];
        w[idx] = acc;
    }
}
hipError_t gemv_acc(const double* V, long ldv, int k, const double* coef, double coef_scale,
                    double beta_w, double* w, long n, hipStream_t s)
{
    long blocks = (n + 255) / 256;
    if (blocks > 16384) blocks = 16384;
    if (k <= 0) {
        if (beta_w != 1.0) gemv_acc_k<<<blocks, 256, 0, s>>>(V, ldv, 0, coef, coef_scale, beta_w, w, n);
        return hipGetLastError();
    }
    for (int i0 = 0; i0 < k; i0 += MD_MAXK) {
        const int kc = (k - i0) < MD_MAXK ? (k - i0) : MD_MAXK;
        gemv_acc_k<<<blocks, 256, 0, s>>>(V + (long)i0 * ldv, ldv, kc, coef + i0, coef_scale,
                                          i0 == 0 ? beta_w : 1.0, w, n);
    }
    return hipGetLastError();
}

// max |x| over n entries: stage 1 per block, stage 2 one block; out[0] = max
__global__ void __launch_bounds__(256) absmax1_k(const double* __restrict__ x, long n,
                                                 double* __restrict__ part)
{
    __shared__ double red[4];
    double m = 0.0;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256) m = fmax(m, fabs(x[i]));
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}
__global__ void __launch_bounds__(256) absmax2_k(const double* __restrict__ part, int G,
                                                 double* __restrict__ out)
{
    __shared__ double red[4];
    double m = 0.0;
    for (int i = threadIdx.x; i < G; i += 256) m = fmax(m, part[i]);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) out[0] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}
hipError_t absmax(const double* x, long n, double* out, double* part, int part_cap, hipStream_t s)
{
    if (n <= 0) return hipErrorInvalidValue;
    long G = (n + 255) / 256;
    if (G > 1024) G = 1024;
    if (G > part_cap) G = part_cap;
    if (G < 1) return hipErrorInvalidValue;
    absmax1_k<<<G, 256, 0, s>>>(x, n, part);
    absmax2_k<<<1, 256, 0, s>>>(part, (int)G, out);
    return hipGetLastError();
}

__global__ void scale_by_inv_k(double* v, const double* den, long n, bool keep_zero)
{
    const double f = keep_zero && den[0] == 0.0 ? 1.0 : 1.0 / den[0];
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256) v[i] *= f;
}
hipError_t scale_by_inv(double* v, const double* den, long n, hipStream_t s, bool keep_zero)
{
    long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    scale_by_inv_k<<<blocks, 256, 0, s>>>(v, den, n, keep_zero);
    return hipGetLastError();
}
__global__ void axpby_k(double a, const double* x, double b, double* y, long n)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256)
        y[i] = a * x[i] + b * y[i];
}
hipError_t axpby(double a, const double* x, double b, double* y, long n, hipStream_t s)
{
    long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    axpby_k<<<blocks, 256, 0, s>>>(a, x, b, y, n);
    return hipGetLastError();
}

__global__ void scale_copy_k(double a, const double* x, double* y, long n)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256) y[i] = a * x[i];
}
hipError_t scale_copy(double a, const double* x, double* y, long n, hipStream_t s)
{
    long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    scale_copy_k<<<blocks, 256, 0, s>>>(a, x, y, n);
    return hipGetLastError();
}

__global__ void dcopy_scalar_k(const double* src, double* dst)
{
    if (threadIdx.x == 0) dst[0] = src[0];
}
hipError_t dcopy_scalar(const double* src, double* dst, hipStream_t s)
{
    dcopy_scalar_k<<<1, 64, 0, s>>>(src, dst);
    return hipGetLastError();
}
__global__ void dsqrt_scalar_k(const double* src, double* dst)
{
    if (threadIdx.x == 0) dst[0] = sqrt(fmax(src[0], 0.0));
}
hipError_t dsqrt_scalar(const double* src, double* dst, hipStream_t s)
{
    dsqrt_scalar_k<<<1, 64, 0, s>>>(src, dst);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// one-sided block Jacobi SVD: gridDim.y workgroups per column-block pair (2 x
// 16 columns).  Each forms the pair's 32x32 Gram matrix from the source
// iterate Xs, diagonalises it in LDS by cyclic parallel Jacobi and applies the
// rotation to its own chunk of rows: Xs -> Xd, and V in place.  The Gram
// matrix and the rotation are computed the same way by every workgroup of the
// pair (same data, same order: bit-identical), so the q/32 pairs of a round
// spread over up to 16 times as many CUs; reading Xs and writing Xd keeps a
// workgroup from seeing rows another has already rotated.  A pair that is
// already orthogonal copies its rows to Xd.
//
// Bound by the latency of 31 dependent rotation rounds (three divisions and two
// square roots each).  A round has one barrier: every 16 lanes form the round's
// rotations themselves from the previous round's G (two buffers) instead of
// waiting for 16 threads to publish them.  Measured per launch, that form (with
// one thread per row in step 3) and this one: 45 and 31 us at p = q = 32, 50 and
// 34 us at 192, 53 and 41 us at 512; with FAST rotations 25, 29 and 34 us.
#define JB 16
#define JW 32
#define JR 128  // rows per Gram chunk

// the rotation that annihilates apq of [app apq; apq aqq] (no branch: the
// discarded values of a skipped rotation may be infinite).  FAST forms c and s
// from two reciprocal square roots instead of three divisions and two square
// roots: with d = aqq - app, o = 2 apq (scaled by a power of two so that the
// squares neither overflow nor vanish) and h = 1 / sqrt(d^2 + o^2),
// c^2 = (1 + |d| h) / 2, s = sign(d) o h / (2 c).
__device__ __forceinline__ double rsqrt_newton(double a)
{
    const double y = __builtin_amdgcn_rsq(a);  // to 2^-23
    const double e = fma(-a * y, y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

template <bool FAST>
__device__ __forceinline__ void jacobi_rot(double app, double aqq, double apq, double& c, double& s)
{
    if (FAST) {
        const double w = fabs(app * aqq);
        const bool rot = fabs(apq) > 1e-300 && !(fabs(apq) <= 1e-16 * (w * __builtin_amdgcn_rsq(w)));
        double d = aqq - app, o = 2.0 * apq;
        const int ex = -__builtin_amdgcn_frexp_exp(fmax(fabs(d), fabs(o)));
        d = __builtin_ldexp(d, ex);
        o = __builtin_ldexp(o, ex);
        const double h = rsqrt_newton(fma(d, d, o * o));
        const double c2 = fma(0.5 * fabs(d), h, 0.5);
        const double ic = rsqrt_newton(c2);
        c = rot ? c2 * ic : 1.0;
        s = rot ? copysign(0.5, d) * o * h * ic : 0.0;
        return;
    }
    const bool rot = fabs(apq) > 1e-300 && fabs(apq) > 1e-16 * sqrt(fabs(app * aqq));
    const double theta = (aqq - app) / (2.0 * apq);
    const double t = (theta >= 0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
    const double cr = 1.0 / sqrt(t * t + 1.0);
    c = rot ? cr : 1.0;
    s = rot ? t * cr : 0.0;
}

// One visit of a pair; false when it was orthogonal already (rows copied to Xd
// unless COPY is off).
template <bool FAST, bool COPY>
__device__ __forceinline__ bool jacobi_pair(const double* Xs, double* Xd, long ldx, int p, double* V, long ldv, int qv,
                                            int pb, int qb, double tol, int ch, int nch)
{
    __shared__ double G[2][JW][JW + 1];
    __shared__ __align__(16) double J[JW][JW + 2];  // even stride: column pairs are 16-byte aligned
    __shared__ double tile[JW][JR + 1];
    __shared__ int sh_off;
    const int tid = threadIdx.x;
    auto colidx = [&](int j) { return j < JB ? pb * JB + j : qb * JB + (j - JB); };
    // this workgroup's rows of the iterate and of V, 32 at a time: thread = row
    // ar of the 32 and columns 4 ac .. 4 ac + 3 of the product
    const int xrows = (p + nch - 1) / nch, vrows = (qv + nch - 1) / nch;
    const int xr0 = ch * xrows, xr1 = min(p, xr0 + xrows);
    const int vr0 = ch * vrows, vr1 = min(qv, vr0 + vrows);
    const int ar = tid & 31, ac = tid >> 5;

    // 1. Gram matrix over row chunks of JR rows staged in LDS, on the FP64
    // matrix cores: wave w forms the 16 x 16 block (w >> 1, w & 1) of G, one
    // v_mfma_f64_16x16x4 per 4 rows (lane l reads row l/16 of the step and
    // column l%16 of each of its two column blocks).
    const int lane = tid & 63, wv = tid >> 6;
    const int wi = wv >> 1, wj = wv & 1;
    v4d gacc = {0.0, 0.0, 0.0, 0.0};
    double ld[JR * JW / 256];
    auto load_chunk = [&](int r0) {  // rows past the last one read as zero
#pragma unroll
        for (int u = 0; u < JR * JW / 256; u++) {
            const int idx = tid + 256 * u;
            const int gr = r0 + idx % JR;
            const double w = Xs[(long)colidx(idx / JR) * ldx + min(gr, p - 1)];
            ld[u] = gr < p ? w : 0.0;
        }
    };
    load_chunk(0);
    for (int r0 = 0; r0 < p; r0 += JR) {
#pragma unroll
        for (int u = 0; u < JR * JW / 256; u++) {
            const int idx = tid + 256 * u;
            tile[idx / JR][idx % JR] = ld[u];
        }
        __syncthreads();
        if (r0 + JR < p) load_chunk(r0 + JR);
        const int kn = min(JR, (p - r0 + 3) & ~3);
#pragma unroll 8
        for (int k0 = 0; k0 < kn; k0 += 4) {
            const double a = tile[16 * wi + (lane & 15)][k0 + (lane >> 4)];
            const double b = tile[16 * wj + (lane & 15)][k0 + (lane >> 4)];
            gacc = mma(a, b, gacc);
        }
        __syncthreads();
    }
    // the first 32 rows of both products, in flight during the rotations (a row
    // that does not exist repeats the last one and is not stored)
    double x[JW], v[JW];
#pragma unroll
    for (int c = 0; c < JW; c++) {
        x[c] = Xs[(long)colidx(c) * ldx + min(xr0 + ar, p - 1)];
        v[c] = V[(long)colidx(c) * ldv + min(vr0 + ar, qv - 1)];
    }
#pragma unroll
    for (int r = 0; r < 4; r++) G[0][16 * wi + (lane >> 4) + 4 * r][16 * wj + (lane & 15)] = gacc[r];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int e = tid + 256 * u;
        J[e >> 5][e & 31] = ((e >> 5) == (e & 31)) ? 1.0 : 0.0;
    }
    if (tid == 0) sh_off = 0;
    __syncthreads();
    // convergence measure of this pair (full 32x32 off-diagonal)
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int e = tid + 256 * u;
        const int gi = e >> 5, gj = e & 31;
        if (gi < gj) {
            const double dd = G[0][gi][gi] * G[0][gj][gj];
            if (dd > 1e-300 && fabs(G[0][gi][gj]) > tol * sqrt(dd)) sh_off = 1;
        }
    }
    __syncthreads();
    if (sh_off == 0) {  // already orthogonal: nothing to rotate
        for (int e = tid; COPY && e < JW * (xr1 > xr0 ? xr1 - xr0 : 0); e += 256) {
            const long off = (long)colidx(e / (xr1 - xr0)) * ldx + xr0 + e % (xr1 - xr0);
            Xd[off] = Xs[off];
        }
        return false;
    }

    // 2. one sweep of cyclic parallel Jacobi on G (tournament ordering, 31
    // rounds).  The round's pairs are disjoint, so G <- R^T G R splits into
    // 16 x 16 independent 2 x 2 blocks (rows P1, Q1 of pair bi, columns P2, Q2
    // of pair bj), one per thread; J <- J R in place, rows 2 bi and 2 bi + 1 of
    // the columns P2, Q2.
    const int bi = tid >> 4, bj = tid & 15;
#pragma unroll 1
    for (int round = 0; round < JW - 1; round++) {
        auto elem = [&](int kpos) {
            const int k = kpos - 1 + round;
            return kpos == 0 ? 0 : (k >= JW - 1 ? k - (JW - 1) : k) + 1;
        };
        const int a1 = elem(bi), b1 = elem(JW - 1 - bi), a2 = elem(bj), b2 = elem(JW - 1 - bj);
        const int P1 = min(a1, b1), Q1 = max(a1, b1), P2 = min(a2, b2), Q2 = max(a2, b2);
        const double(*Gc)[JW + 1] = G[round & 1];
        double(*Gn)[JW + 1] = G[(round & 1) ^ 1];
        const double g00 = Gc[P1][P2], g01 = Gc[P1][Q2], g10 = Gc[Q1][P2], g11 = Gc[Q1][Q2];
        const double p2 = Gc[P2][P2], q2 = Gc[Q2][Q2], o2 = Gc[P2][Q2];
        const double j00 = J[2 * bi][P2], j01 = J[2 * bi][Q2], j10 = J[2 * bi + 1][P2], j11 = J[2 * bi + 1][Q2];
        // lanes bj of every 16 hold the rotation of pair bj; that of pair bi
        // comes from lane bi
        double c2, s2;
        jacobi_rot<FAST>(p2, q2, o2, c2, s2);
        const double c1 = __shfl(c2, bi, 64), s1 = __shfl(s2, bi, 64);
        const double h00 = c1 * g00 - s1 * g10, h01 = c1 * g01 - s1 * g11;
        const double h10 = s1 * g00 + c1 * g10, h11 = s1 * g01 + c1 * g11;
        Gn[P1][P2] = c2 * h00 - s2 * h01;
        Gn[P1][Q2] = s2 * h00 + c2 * h01;
        Gn[Q1][P2] = c2 * h10 - s2 * h11;
        Gn[Q1][Q2] = s2 * h10 + c2 * h11;
        J[2 * bi][P2] = c2 * j00 - s2 * j01;
        J[2 * bi][Q2] = s2 * j00 + c2 * j01;
        J[2 * bi + 1][P2] = c2 * j10 - s2 * j11;
        J[2 * bi + 1][Q2] = s2 * j10 + c2 * j11;
        __syncthreads();
    }

    // 3. X[:, cols] <- X[:, cols] J ; V[:, cols] <- V[:, cols] J
    auto product = [&](const double (&x)[JW], double (&y)[4]) {
#pragma unroll
        for (int u = 0; u < 4; u++) y[u] = 0.0;
#pragma unroll
        for (int c = 0; c < JW; c++) {
            const double2 ja = *(const double2*)&J[c][4 * ac], jb = *(const double2*)&J[c][4 * ac + 2];
            y[0] = fma(x[c], ja.x, y[0]);
            y[1] = fma(x[c], ja.y, y[1]);
            y[2] = fma(x[c], jb.x, y[2]);
            y[3] = fma(x[c], jb.y, y[3]);
        }
    };
    for (int r0 = xr0; r0 < xr1; r0 += 32) {
        const int row = r0 + ar;
        if (r0 > xr0) {
#pragma unroll
            for (int c = 0; c < JW; c++) x[c] = Xs[(long)colidx(c) * ldx + min(row, p - 1)];
        }
        double y[4];
        product(x, y);
        if (row < xr1) {
#pragma unroll
            for (int u = 0; u < 4; u++) Xd[(long)colidx(4 * ac + u) * ldx + row] = y[u];
        }
    }
    for (int r0 = vr0; r0 < vr1; r0 += 32) {
        const int row = r0 + ar;
        if (r0 > vr0) {
#pragma unroll
            for (int c = 0; c < JW; c++) v[c] = V[(long)colidx(c) * ldv + min(row, qv - 1)];
        }
        double y[4];
        product(v, y);
        __syncthreads();  // in place: every thread of these rows has read them
        if (row < vr1) {
#pragma unroll
            for (int u = 0; u < 4; u++) V[(long)colidx(4 * ac + u) * ldv + row] = y[u];
        }
    }
    return true;
}

// Round rd of the tournament of nb column blocks: gridDim.x = nb / 2 pairs,
// gridDim.y workgroups each.  flag[0] = tag when a pair rotated.
template <bool FAST>
__global__ void __launch_bounds__(256) jacobi_k(const double* __restrict__ Xs, double* __restrict__ Xd, long ldx, int p,
                                                double* __restrict__ V, long ldv, int qv, int nb, int rd, double tol,
                                                int* __restrict__ flag, int tag)
{
    auto elem = [&](int kp) { return kp == 0 ? 0 : (kp - 1 + rd) % (nb - 1) + 1; };
    const int i = blockIdx.x;
    if (jacobi_pair<FAST, true>(Xs, Xd, ldx, p, V, ldv, qv, elem(i), elem(nb - 1 - i), tol, blockIdx.y, gridDim.y) &&
        threadIdx.x == 0)
        flag[0] = tag;
}

// The whole iteration of two column blocks (one pair, so no round depends on
// another workgroup): sweeps until the pair is orthogonal, at most max_sweeps.
// The result is in X.  A sweep of this kernel costs what a launch of jacobi_k
// does (about 30 us at p = q = 32), without the launch, the flag's clearing and
// the host's look at it that followed each (about 30 us more); one workgroup
// takes every row, so the rule keeps to p <= 256, where the rows are a small
// part of the rotations' time.
__global__ void __launch_bounds__(256) jacobi_all_k(double* X, double* X2, long ldx, int p, double* V, long ldv, int qv,
                                                    double tol, int max_sweeps)
{
    double *a = X, *b = X2;
    for (int sweep = 0; sweep < max_sweeps; sweep++) {
        if (!jacobi_pair<false, false>(a, b, ldx, p, V, ldv, qv, 0, 1, tol, 0, 1)) break;
        double* t = a;
        a = b;
        b = t;
        __syncthreads();  // the rotated rows, before the next Gram matrix reads them
    }
    if (a != X)
        for (int e = threadIdx.x; e < JW * p; e += 256) {
            const long off = (long)(e / p) * ldx + e % p;
            X[off] = a[off];
        }
}

bool jacobi_all_ok(int p, int qv) { return qv == JW && p > 0 && p <= 256; }
hipError_t jacobi_all(double* X, double* X2, long ldx, int p, double* V, long ldv, int qv, double tol, int max_sweeps,
                      hipStream_t s)
{
    if (!jacobi_all_ok(p, qv) || X == X2) return hipErrorInvalidValue;
    jacobi_all_k<<<1, 256, 0, s>>>(X, X2, ldx, p, V, ldv, qv, tol, max_sweeps);
    return hipGetLastError();
}

hipError_t jacobi_step(const double* Xs, double* Xd, long ldx, int p, double* V, long ldv, int qv, int nb, int rd,
                       int nchunk, double tol, int* flag, int tag, bool fast, hipStream_t s)
{
    if (nb < 2) return hipSuccess;
    if (nb % 2 != 0 || rd < 0 || rd >= nb - 1 || nchunk < 1 || nchunk > 64 || Xs == Xd) return hipErrorInvalidValue;
    const dim3 grid(nb / 2, nchunk);
    if (fast) jacobi_k<true><<<grid, 256, 0, s>>>(Xs, Xd, ldx, p, V, ldv, qv, nb, rd, tol, flag, tag);
    else jacobi_k<false><<<grid, 256, 0, s>>>(Xs, Xd, ldx, p, V, ldv, qv, nb, rd, tol, flag, tag);
    return hipGetLastError();
}

// Householder QR of one 32-column panel (the column loop of LAPACK dgeqr2
// with the forward, columnwise T of dlarft).  A is column-major (column j at
// A + j*lda) with pp rows; the panel is columns c0..c0+31, rows c0..pp-1.
// Column c = c0 + j has its diagonal in row r = c0 + j: H_j = I - tau v v^T,
// v_r = 1, maps rows r.. of the column to beta e_r, so R(r, c) = beta and the
// rows below become zero (a column whose part below the diagonal is zero, or
// underflows to zero when squared, gets tau = 0).  v goes to column j of V
// (rows c0..pp-1, zero above r) and the upper-triangular T (32 x 32,
// row-major) satisfies H_0 H_1 ... H_31 = I - V T V^T.
//
// One workgroup.  Per column three phases, a barrier after each: (a) all 256
// threads form v and the reflected column; (b) the dot products of v with the
// 32 panel columns (the earlier v's for k < j, for T): 8 groups of 32 lanes,
// group g owns columns 4g..4g+3 and each lane every 32nd row, so a thread
// keeps 4 sums and its loads are all in flight together, and the 32 lanes
// reduce by shuffles; (c) H_j on the columns right of j (same layout; the
// others are stored back unchanged so the loads stay unconditional), the next
// column's squared norm below its diagonal, and column j of T.
__global__ void __launch_bounds__(256) hqr_panel_k(double* __restrict__ A, long lda, int pp, int c0,
                                                    double* __restrict__ V, long ldv, double* __restrict__ T)
{
    __shared__ double fin[34];  // [0, 32): dot products; [32]: norm^2 below the diagonal; [33]: diagonal
    __shared__ double Ts[32][33];
    __shared__ double red[4];
    const int tid = threadIdx.x;
    const int g = tid >> 5, rl = tid & 31;
    for (int e = tid; e < 32 * 33; e += 256) Ts[e / 33][e % 33] = 0.0;
    {
        const double* col = A + (long)c0 * lda;
        double s2 = 0.0;
        for (int i = c0 + 1 + tid; i < pp; i += 256) s2 += col[i] * col[i];
        s2 = wave_sum(s2);
        if ((tid & 63) == 0) red[tid >> 6] = s2;
        if (tid == 0) fin[33] = col[c0];
    }
    __syncthreads();
    if (tid == 0) fin[32] = red[0] + red[1] + red[2] + red[3];
    __syncthreads();
    for (int j = 0; j < 32; j++) {
        const int r = c0 + j;
        double* col = A + (long)r * lda;
        const double alpha = fin[33], sig2 = fin[32];
        double tau = 0.0, beta = alpha, scl = 0.0;
        if (sig2 > 0.0) {
            beta = -copysign(sqrt(alpha * alpha + sig2), alpha);
            tau = (beta - alpha) / beta;
            scl = 1.0 / (alpha - beta);
        }
        // (a) v and the reflected column
        double* vj = V + (long)j * ldv;
        for (int i = c0 + tid; i < pp; i += 256) {
            double vi = 0.0;
            if (i >= r) {
                vi = i == r ? 1.0 : col[i] * scl;
                col[i] = i == r ? beta : 0.0;
            }
            vj[i] = vi;
        }
        __syncthreads();
        // (b) d_k = src_k . v over rows >= r (src_k = v_k for k < j, column
        // c0 + k otherwise; d_j is not used)
        const double* src[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = 4 * g + e;
            src[e] = k < j ? V + (long)k * ldv : A + (long)(c0 + k) * lda;
        }
        const int i0 = c0 + rl + 32 * ((r - c0) >> 5);
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int i = i0; i < pp; i += 32) {
            const double vi = i >= r ? vj[i] : 0.0;
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] += src[e][i] * vi;
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
#pragma unroll
            for (int o = 16; o >= 1; o >>= 1) acc[e] += __shfl_xor(acc[e], o, 32);
        }
        if (rl == 0) {
#pragma unroll
            for (int e = 0; e < 4; e++) fin[4 * g + e] = acc[e];
        }
        __syncthreads();
        // (c) H_j on the columns right of j; the next column's norm; T
        double f[4];
#pragma unroll
        for (int e = 0; e < 4; e++) f[e] = 4 * g + e > j ? tau * fin[4 * g + e] : 0.0;
        double s2 = 0.0;
        const int kn = j + 1;
        const bool own_next = kn < 32 && g == (kn >> 2);
        // every lane has the same number of rows (pp - c0 is a multiple of
        // 32); rows above r keep their values (v is zero there).  Blocks of
        // four rows: all loads, then the updates, then all stores, since a
        // load cannot move above a store the compiler cannot tell apart.
        const int nrow = ((pp - c0) >> 5) - ((r - c0) >> 5);
        auto rows = [&](int t, int nu) {
            double x[4][4], w[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if (u >= nu) break;
                const int i = i0 + 32 * (t + u);
                w[u] = i >= r ? vj[i] : 0.0;
#pragma unroll
                for (int e = 0; e < 4; e++) x[u][e] = A[(long)(c0 + 4 * g + e) * lda + i];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if (u >= nu) break;
                const int i = i0 + 32 * (t + u);
                double y = 0.0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    x[u][e] -= f[e] * w[u];
                    A[(long)(c0 + 4 * g + e) * lda + i] = x[u][e];
                    y = 4 * g + e == kn ? x[u][e] : y;
                }
                s2 += i > r + 1 ? y * y : 0.0;
                if (own_next && i == r + 1) fin[33] = y;
            }
        };
        int t = 0;
        for (; t + 4 <= nrow; t += 4) rows(t, 4);
        for (; t < nrow; t++) rows(t, 1);
        if (own_next) {
#pragma unroll
            for (int o = 16; o >= 1; o >>= 1) s2 += __shfl_xor(s2, o, 32);
            if (rl == 0) fin[32] = s2;
        }
        if (tid < j) {
            double t = 0.0;
            for (int l = tid; l < j; l++) t += Ts[tid][l] * fin[l];
            Ts[tid][j] = -tau * t;
        } else if (tid == j) {
            Ts[j][j] = tau;
        }
        __syncthreads();
    }
    for (int e = tid; e < 32 * 32; e += 256) T[e] = Ts[e >> 5][e & 31];
}
hipError_t hqr_panel(double* A, long lda, int pp, int c0, double* V, long ldv, double* T, hipStream_t s)
{
    if (c0 < 0 || c0 + 32 > pp || lda < pp || ldv < pp) return hipErrorInvalidValue;
    hqr_panel_k<<<1, 256, 0, s>>>(A, lda, pp, c0, V, ldv, T);
    return hipGetLastError();
}

// m[i] = max over j != i (j < n) of |G_ij| / sqrt(G_ii G_jj), the largest
// cosine between column i and another column of the matrix whose Gram matrix
// G is (row-major, ld ldg); pairs with G_ii G_jj <= 1e-300 are skipped.
// One workgroup per row.
__global__ void __launch_bounds__(256) max_cos_k(const double* __restrict__ G, long ldg, int n,
                                                  double* __restrict__ m)
{
    __shared__ double red[4];
    const int i = blockIdx.x;
    const double gi = G[(long)i * ldg + i];
    double best = 0.0;
    for (int j = threadIdx.x; j < n; j += 256) {
        if (j == i) continue;
        const double d = gi * G[(long)j * ldg + j];
        if (d > 1e-300) best = fmax(best, fabs(G[(long)i * ldg + j]) / sqrt(d));
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) best = fmax(best, __shfl_xor(best, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) m[i] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}
hipError_t max_cos(const double* G, long ldg, int n, double* m, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    max_cos_k<<<n, 256, 0, s>>>(G, ldg, n, m);
    return hipGetLastError();
}

// out[j*ldo + i] = in[perm[j]*ldi + i] (i < rows, j < ncols): a column gather
__global__ void gather_cols_k(const double* __restrict__ in, long ldi, double* __restrict__ out, long ldo,
                              const int* __restrict__ perm, int rows)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int j = blockIdx.y;
    if (i < rows) out[(long)j * ldo + i] = in[(long)perm[j] * ldi + i];
}
hipError_t gather_cols(const double* in, long ldi, double* out, long ldo, const int* perm, int rows, int ncols,
                       hipStream_t s)
{
    if (rows <= 0 || ncols <= 0) return hipSuccess;
    gather_cols_k<<<dim3((rows + 255) / 256, ncols), 256, 0, s>>>(in, ldi, out, ldo, perm, rows);
    return hipGetLastError();
}
// X[j*ldx + perm[i]] = R[i*ldr + j] (i, j < n): R^T with its rows permuted
__global__ void tr_scatter_k(const double* __restrict__ R, long ldr, double* __restrict__ X, long ldx,
                             const int* __restrict__ perm, int n)
{
    const int j = blockIdx.x * 256 + threadIdx.x;
    const int i = blockIdx.y;
    if (j < n) X[(long)j * ldx + perm[i]] = R[(long)i * ldr + j];
}
hipError_t tr_scatter(const double* R, long ldr, double* X, long ldx, const int* perm, int n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    tr_scatter_k<<<dim3((n + 255) / 256, n), 256, 0, s>>>(R, ldr, X, ldx, perm, n);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256) col_norms_k(const double* __restrict__ X, long ldx, int p,
                                                   double* __restrict__ s)
{
    __shared__ double red[4];
    const double* x = X + (long)blockIdx.x * ldx;
    double acc = 0.0;
    for (int i = threadIdx.x; i < p; i += 256) acc += x[i] * x[i];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) s[blockIdx.x] = sqrt(red[0] + red[1] + red[2] + red[3]);
}
hipError_t col_norms(const double* X, long ldx, int p, int q, double* s, hipStream_t st)
{
    if (q <= 0) return hipSuccess;
    col_norms_k<<<q, 256, 0, st>>>(X, ldx, p, s);
    return hipGetLastError();
}

__global__ void set_int_k(int* p, int v)
{
    if (threadIdx.x == 0) p[0] = v;
}
hipError_t set_int(int* p, int v, hipStream_t s)
{
    set_int_k<<<1, 64, 0, s>>>(p, v);
    return hipGetLastError();
}

__global__ void set_identity_k(double* V, long ldv, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int j = blockIdx.y;
    if (i < n) V[(long)j * ldv + i] = (i == j) ? 1.0 : 0.0;
}
hipError_t set_identity(double* V, long ldv, int n, hipStream_t s)
{
    dim3 grid((n + 255) / 256, n);
    set_identity_k<<<grid, 256, 0, s>>>(V, ldv, n);
    return hipGetLastError();
}

__global__ void svd_gather1_k(const double* __restrict__ X, long ldx, int p,
                              const int* __restrict__ perm, double* __restrict__ out, long s0, long s1)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int j = blockIdx.y;
    if (i >= p) return;
    out[(long)i * s0 + (long)j * s1] = X[(long)perm[j] * ldx + i];
}
__global__ void svd_gather2_k(const double* __restrict__ V, long ldv, int q,
                              const int* __restrict__ perm, double* __restrict__ out, long s0,
                              long s1)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int j = blockIdx.y;
    if (i >= q) return;
    out[(long)j * s0 + (long)i * s1] = V[(long)perm[j] * ldv + i];
}
hipError_t svd_gather(const double* X, long ldx, int p, const double* V, long ldv, int q,
                      const int* perm, int k, double* out1, long s10, long s11,
                      double* out2, long s20, long s21, hipStream_t s)
{
    if (k <= 0) return hipSuccess;
    dim3 g1((p + 255) / 256, k), g2((q + 255) / 256, k);
    svd_gather1_k<<<g1, 256, 0, s>>>(X, ldx, p, perm, out1, s10, s11);
    svd_gather2_k<<<g2, 256, 0, s>>>(V, ldv, q, perm, out2, s20, s21);
    return hipGetLastError();
}

__global__ void set_unit_col_k(double* x, int p, int pos)
{
    for (int i = blockIdx.x * 256 + threadIdx.x; i < p; i += gridDim.x * 256) x[i] = (i == pos) ? 1.0 : 0.0;
}
hipError_t set_unit_col(double* x, int p, int pos, hipStream_t s)
{
    int blocks = (p + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    set_unit_col_k<<<blocks, 256, 0, s>>>(x, p, pos);
    return hipGetLastError();
}

__global__ void scale_cols_k(double* A, long lda, int r, int c, const double* sv)
{
    const int j = blockIdx.x * 256 + threadIdx.x;
    const int i = blockIdx.y;
    if (j < c && i < r) A[(long)i * lda + j] *= sv[j];
}
__global__ void scale_rows_k(double* A, long lda, int r, int c, const double* sv)
{
    const int j = blockIdx.x * 256 + threadIdx.x;
    const int i = blockIdx.y;
    if (j < c && i < r) A[(long)i * lda + j] *= sv[i];
}
hipError_t scale_cols(double* A, long lda, int r, int c, const double* sv, hipStream_t s)
{
    if (r <= 0 || c <= 0) return hipSuccess;
    dim3 grid((c + 255) / 256, r);
    scale_cols_k<<<grid, 256, 0, s>>>(A, lda, r, c, sv);
    return hipGetLastError();
}
hipError_t scale_rows(double* A, long lda, int r, int c, const double* sv, hipStream_t s)
{
    if (r <= 0 || c <= 0) return hipSuccess;
    dim3 grid((c + 255) / 256, r);
    scale_rows_k<<<grid, 256, 0, s>>>(A, lda, r, c, sv);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// CholeskyQR pieces.  chol_diag_k factors one CB x CB diagonal block of a
// symmetric positive definite G and writes L_kk (lower) and its inverse; a
// non-positive or non-finite pivot sets flag[0] = 1.
#define CB 64
#define CW 16  // columns of the trailing matrix (rows of the inverse) per wave
// v from lane `lane` (wave-uniform index) of the wavefront, as a register
// broadcast (two 32-bit readlanes)
__device__ __forceinline__ double wave_bcast(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Four wavefronts, lane r = row r.  Wave w keeps columns 16w .. 16w+15 of the
// not yet factored matrix, a[kk] = A[r][16w + kk], and rows 16w .. 16w+15 of
// the right-hand side of L X = I, b[kk] = B[16w + kk][r] (lane r = column r
// of X).  Right-looking step j, owned by wave j / 16 (register index j % 16 a
// compile-time constant: the 16 steps of a column block are unrolled):
//   owner: pivot A[j][j] from lane j, L[r][j] = A[r][j] / L[j][j] (the whole
//          column, zero above the diagonal) and X[j][r] = B[j][r] / L[j][j]
//          into LDS; X[j][:] is row j of L^-1;
//   all:   A[r][k] -= L[r][j] L[k][j] on their columns k and
//          B[i][r] -= L[i][j] X[j][r] on their rows i, L[k][j] read from LDS
//          as a broadcast.
// Entries above the diagonal of column j of L are zero, so the full-width
// updates need no guard; columns and rows already consumed take values that
// are never read again.  The column and row buffers alternate between two
// LDS slots by step parity, so one barrier per step orders them: a wave can
// only overwrite a slot after every wave has passed the next barrier, that
// is, after every wave has read it.  Columns past nbk are the identity's and
// are left out: a block of 32 takes 15 us, as one of 64 completed with the
// identity it took 27.  (A wave factoring its 16 columns alone in registers, the
// others updating theirs 16 columns at a time, took 29 us for 64 against 28: the
// chain of square root and division per column is the bound, not the barriers.)
__device__ __forceinline__ void chol_block(const double* __restrict__ G, long ldg, int k0, int nbk,
                                           double* __restrict__ L, long ldl, double* __restrict__ Linv, long ldi,
                                           int* __restrict__ flag, double (*Ls)[CB + 1], double (*col)[CB],
                                           double (*xrow)[CB])
{
    const int tid = threadIdx.x, r = tid & 63, wid = tid >> 6;
    // coalesced load (lane = column, one row per wave per round); a block
    // narrower than CB (the last one) is completed with the identity
#pragma unroll
    for (int i0 = 0; i0 < CB; i0 += 4 * 4) {
        double tmp[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = i0 + u * 4 + wid;
            tmp[u] = (i < nbk && r < nbk) ? G[(long)(k0 + i) * ldg + k0 + r] : (i == r ? 1.0 : 0.0);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) Ls[i0 + u * 4 + wid][r] = tmp[u];
    }
    __syncthreads();
    double a[CW], bv[CW];
#pragma unroll
    for (int kk = 0; kk < CW; kk++) {
        a[kk] = Ls[r][wid * CW + kk];
        bv[kk] = (wid * CW + kk == r) ? 1.0 : 0.0;
    }
    __syncthreads();  // every row is in registers before Ls takes L
    int bad = 0;
    for (int jb = 0; jb * CW < nbk; jb++) {
#pragma unroll
        for (int jj = 0; jj < CW; jj++) {
            const int j = jb * CW + jj, slot = jj & 1;
            if (wid == jb) {
                const double piv = wave_bcast(a[jj], j);
                const bool ok = piv > 0.0 && isfinite(piv);
                bad |= ok ? 0 : 1;
                const double d = ok ? sqrt(piv) : 1.0;
                const double inv = 1.0 / d;
                const double cj = r > j ? a[jj] * inv : (r == j ? d : 0.0);
                const double xj = bv[jj] * inv;
                col[slot][r] = cj;
                xrow[slot][r] = xj;
                Ls[r][j] = cj;
                if (j < nbk && r < nbk) Linv[(long)(k0 + j) * ldi + k0 + r] = xj;
            }
            __syncthreads();
            const double lr = col[slot][r];   // L[r][j]
            const double xr = xrow[slot][r];  // X[j][r]
#pragma unroll
            for (int kk = 0; kk < CW; kk += 2) {
                const double2 lk = *(const double2*)&col[slot][wid * CW + kk];  // L[k][j], L[k+1][j]
                a[kk] = fma(-lr, lk.x, a[kk]);
                a[kk + 1] = fma(-lr, lk.y, a[kk + 1]);
                bv[kk] = fma(-lk.x, xr, bv[kk]);
                bv[kk + 1] = fma(-lk.y, xr, bv[kk + 1]);
            }
        }
    }
    __syncthreads();
    // L (lower; Ls holds zeros above the diagonal), coalesced rows
    for (int i = wid; i < nbk; i += 4)
        if (r < nbk) L[(long)(k0 + i) * ldl + k0 + r] = Ls[i][r];
    if (r == 0 && bad) flag[0] = 1;
}

__global__ void __launch_bounds__(256) chol_diag_k(const double* __restrict__ G, long ldg, int k0, int nbk,
                                                   double* __restrict__ L, long ldl,
                                                   double* __restrict__ Linv, long ldi,
                                                   int* __restrict__ flag)
{
    __shared__ double Ls[CB][CB + 1];
    __shared__ __attribute__((aligned(16))) double col[2][CB];
    __shared__ double xrow[2][CB];
    chol_block(G, ldg, k0, nbk, L, ldl, Linv, ldi, flag, Ls, col, xrow);
}

// one diagonal block per workgroup, one job per chain
__global__ void __launch_bounds__(256) chol_diag_batch_k(const CholJob* __restrict__ jobs)
{
    __shared__ double Ls[CB][CB + 1];
    __shared__ __attribute__((aligned(16))) double col[2][CB];
    __shared__ double xrow[2][CB];
    const CholJob& j = jobs[blockIdx.x];
    chol_block(j.G, j.ldg, j.k0, j.nbk, j.L, j.ldl, j.Linv, j.ldi, j.flag, Ls, col, xrow);
}

hipError_t chol_diag_batch(const CholJob* jobs, int n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    chol_diag_batch_k<<<n, 256, 0, s>>>(jobs);
    return hipGetLastError();
}

hipError_t chol_diag(const double* G, long ldg, int k0, int nbk, double* L, long ldl, double* Linv, long ldi,
                     int* flag, hipStream_t s)
{
    if (nbk <= 0 || nbk > CB) return hipErrorInvalidValue;
    chol_diag_k<<<1, 256, 0, s>>>(G, ldg, k0, nbk, L, ldl, Linv, ldi, flag);
    return hipGetLastError();
}

// E = G - I on the leading nl x nl block, zero elsewhere (n x n, ld n)
__global__ void __launch_bounds__(256) eye_sub_k(const double* __restrict__ G, int n, int nl, double* __restrict__ E)
{
    const long nn = (long)n * n;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < nn; e += (long)gridDim.x * 256) {
        const int i = (int)(e / n), j = (int)(e - (long)i * n);
        E[e] = (i < nl && j < nl) ? G[e] - (i == j ? 1.0 : 0.0) : 0.0;
    }
}
hipError_t eye_sub(const double* G, int n, int nl, double* E, hipStream_t s)
{
    long blocks = ((long)n * n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    eye_sub_k<<<blocks, 256, 0, s>>>(G, n, nl, E);
    return hipGetLastError();
}

// X = I + c1 E + c2 E2 + c3 E3 and Y = I + d1 E + d2 E2 + d3 E3 (n x n)
__global__ void __launch_bounds__(256) series3_k(const double* __restrict__ E, const double* __restrict__ E2,
                                                 const double* __restrict__ E3, int n, double c1, double c2,
                                                 double c3, double d1, double d2, double d3,
                                                 double* __restrict__ X, double* __restrict__ Y)
{
    const long nn = (long)n * n;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < nn; e += (long)gridDim.x * 256) {
        const int i = (int)(e / n), j = (int)(e - (long)i * n);
        const double id = i == j ? 1.0 : 0.0, a = E[e], b = E2[e], c = E3[e];
        X[e] = id + c1 * a + c2 * b + c3 * c;
        Y[e] = id + d1 * a + d2 * b + d3 * c;
    }
}
hipError_t series3(const double* E, const double* E2, const double* E3, int n, const double c[3], const double d[3],
                   double* X, double* Y, hipStream_t s)
{
    long blocks = ((long)n * n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    series3_k<<<blocks, 256, 0, s>>>(E, E2, E3, n, c[0], c[1], c[2], d[0], d[1], d[2], X, Y);
    return hipGetLastError();
}

// G[i][i] += factor * trace(G[0:n, 0:n]) for i < n  (the shift of shifted
// CholeskyQR; trace(A^T A) = ||A||_F^2 bounds ||A||_2^2 from above)
__global__ void __launch_bounds__(256) shift_diag_k(double* __restrict__ G, long ldg, int n, double factor)
{
    __shared__ double red[4];
    __shared__ double sh;
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) acc += G[(long)i * ldg + i];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) sh = factor * (red[0] + red[1] + red[2] + red[3]);
    __syncthreads();
    const double v = sh;
    for (int i = threadIdx.x; i < n; i += 256) G[(long)i * ldg + i] += v;
}
hipError_t shift_diag(double* G, long ldg, int n, double factor, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    shift_diag_k<<<1, 256, 0, s>>>(G, ldg, n, factor);
    return hipGetLastError();
}

// G[i*ldg + i] += v for i in [i0, i1)
__global__ void add_diag_k(double* G, long ldg, int i0, int i1, double v)
{
    const int i = i0 + blockIdx.x * 256 + threadIdx.x;
    if (i < i1) G[(long)i * ldg + i] += v;
}
hipError_t add_diag(double* G, long ldg, int i0, int i1, double v, hipStream_t s)
{
    if (i1 <= i0) return hipSuccess;
    add_diag_k<<<(i1 - i0 + 255) / 256, 256, 0, s>>>(G, ldg, i0, i1, v);
    return hipGetLastError();
}

// out[0] = max_{i,j<n} |G[i][j] - delta_ij|   (deviation from the identity)
__global__ void __launch_bounds__(256) eye_dev_k(const double* __restrict__ G, long ldg, int n,
                                                 double* __restrict__ part)
{
    __shared__ double red[4];
    double m = 0.0;
    const long tot = (long)n * n;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < tot; e += (long)gridDim.x * 256) {
        const long i = e / n, j = e - i * n;
        const double v = G[i * ldg + j] - (i == j ? 1.0 : 0.0);
        m = fmax(m, isfinite(v) ? fabs(v) : 1e300);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}
hipError_t eye_deviation(const double* G, long ldg, int n, double* out, double* part, hipStream_t s)
{
    long G_ = ((long)n * n + 255) / 256;
    if (G_ > 1024) G_ = 1024;
    eye_dev_k<<<G_, 256, 0, s>>>(G, ldg, n, part);
    absmax2_k<<<1, 256, 0, s>>>(part, (int)G_, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Batched vector kernels: one job per problem (chain), problem index = last
// grid dimension.
#define BV_EPT 8
#define BV_BLOCK 256
#define BV_CHUNK (BV_BLOCK * BV_EPT)

// stage 1: part[(q * kmax + i) * G + b] = dot of chunk b of V_i and w
__global__ void __launch_bounds__(BV_BLOCK) bmdot1_k(const DotJob* __restrict__ jobs, int kmax, int G,
                                                     double* __restrict__ part)
{
    __shared__ double red[BV_BLOCK / 64];
    const DotJob& j = jobs[blockIdx.y];
    const int b = blockIdx.x;
    double* pq = part + (size_t)blockIdx.y * kmax * G;
    const long base = (long)b * BV_CHUNK + threadIdx.x;
    double wr[BV_EPT];
#pragma unroll
    for (int e = 0; e < BV_EPT; e++) {
        const long idx = base + (long)e * BV_BLOCK;
        wr[e] = idx < j.n ? j.w[idx] : 0.0;
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int i = 0; i < j.k; i++) {
        const double* vi = j.V + (long)i * j.ldv;
        double acc = 0.0;
#pragma unroll
        for (int e = 0; e < BV_EPT; e++) {
            const long idx = base + (long)e * BV_BLOCK;
            if (idx < j.n) acc += vi[idx] * wr[e];
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, 64);
        if (lane == 0) red[wid] = acc;
        __syncthreads();
        if (threadIdx.x == 0) pq[(size_t)i * G + b] = (red[0] + red[1]) + (red[2] + red[3]);
        __syncthreads();
    }
}
// stage 2: out[i] = sum_b part, one workgroup per (problem, row)
__global__ void __launch_bounds__(256) bmdot2_k(const DotJob* __restrict__ jobs, int kmax, int G,
                                                const double* __restrict__ part)
{
    __shared__ double red[4];
    const DotJob& j = jobs[blockIdx.y];
    const int i = blockIdx.x;
    if (i >= j.k) return;
    const long nb = (j.n + BV_CHUNK - 1) / BV_CHUNK;
    const double* pq = part + ((size_t)blockIdx.y * kmax + i) * G;
    double acc = 0.0;
    for (long b = threadIdx.x; b < nb; b += 256) acc += pq[b];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) j.out[i] = (red[0] + red[1]) + (red[2] + red[3]);
}
hipError_t bmdot(const DotJob* jobs, int n, int kmax, long nmax, double* part, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const int G = (int)((nmax + BV_CHUNK - 1) / BV_CHUNK);
    bmdot1_k<<<dim3(G, n), BV_BLOCK, 0, s>>>(jobs, kmax, G, part);
    bmdot2_k<<<dim3(kmax, n), 256, 0, s>>>(jobs, kmax, G, part);
    return hipGetLastError();
}
long bmdot_part_size(int n, int kmax, long nmax) { return (long)n * kmax * ((nmax + BV_CHUNK - 1) / BV_CHUNK); }

// Fused Lanczos step, batched: block (b, q) owns chunk b of job q's vectors
// (BV_CHUNK entries as BV_EPT / 2 pairs per thread), no split of the basis vectors.
#define BV_PAIRS (BV_EPT / 2)
__global__ void __launch_bounds__(BV_BLOCK) bstep_dots_k(const StepJob* __restrict__ jobs, int kmax, int G,
                                                         double* __restrict__ part)
{
    __shared__ double red[MD_MAXK][BV_BLOCK / 64];
    const StepJob& j = jobs[blockIdx.y];
    const long c0 = (long)blockIdx.x * BV_CHUNK;
    if (c0 >= j.n) return;  // the finalising sum reads only this job's chunks
    const double a = j.alpha[0];
    const double beta = j.beta_sq ? sqrt(fmax(*j.beta_sq, 0.0)) : j.beta;
    const double* vj = j.V + (long)(j.k - 1) * j.ldv;
    const double* vm = j.k >= 2 ? j.V + (long)(j.k - 2) * j.ldv : nullptr;
    double2 wr[BV_PAIRS];
#pragma unroll
    for (int e = 0; e < BV_PAIRS; e++) {
        const long idx = c0 + 2 * ((long)e * BV_BLOCK + threadIdx.x);
        if (idx < j.n) {
            double2 x = *(const double2*)(j.w + idx);
            const double2 p = *(const double2*)(vj + idx);
            x.x -= a * p.x;
            x.y -= a * p.y;
            if (vm) {
                const double2 q = *(const double2*)(vm + idx);
                x.x -= beta * q.x;
                x.y -= beta * q.y;
            }
            *(double2*)(j.w + idx) = x;
            wr[e] = x;
        } else {
            wr[e] = make_double2(0.0, 0.0);
        }
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int i = 0; i < j.k; i++) {
        const double* vi = j.V + (long)i * j.ldv;
        double acc = 0.0;
#pragma unroll
        for (int e = 0; e < BV_PAIRS; e++) {
            const long idx = c0 + 2 * ((long)e * BV_BLOCK + threadIdx.x);
            if (idx < j.n) {
                const double2 p = *(const double2*)(vi + idx);
                acc += p.x * wr[e].x + p.y * wr[e].y;
            }
        }
        acc = wave_sum(acc);
        if (lane == 0) red[i][wid] = acc;
    }
    __syncthreads();
    double* pq = part + (size_t)blockIdx.y * kmax * G;
    for (int i = threadIdx.x; i < j.k; i += BV_BLOCK) {
        double sum = 0.0;
#pragma unroll
        for (int q = 0; q < BV_BLOCK / 64; q++) sum += red[i][q];
        pq[(size_t)i * G + blockIdx.x] = sum;
    }
}
// out[i] = sum over the job's chunks, fixed order; one workgroup per (row, job)
__global__ void __launch_bounds__(256) bstep_sum_k(const StepJob* __restrict__ jobs, int kmax, int G,
                                                   const double* __restrict__ part)
{
    __shared__ double red[4];
    const StepJob& j = jobs[blockIdx.y];
    const int i = blockIdx.x;
    if (i >= j.k) return;
    const long nb = (j.n + BV_CHUNK - 1) / BV_CHUNK;
    const double* pq = part + ((size_t)blockIdx.y * kmax + i) * G;
    double acc = 0.0;
    for (long b = threadIdx.x; b < nb; b += 256) acc += pq[b];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) j.out[i] = (red[0] + red[1]) + (red[2] + red[3]);
}
hipError_t bstep_dots(const StepJob* jobs, int n, int kmax, long nmax, double* part, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    if (kmax < 1 || kmax > MD_MAXK) return hipErrorInvalidValue;
    const int G = (int)((nmax + BV_CHUNK - 1) / BV_CHUNK);
    bstep_dots_k<<<dim3(G, n), BV_BLOCK, 0, s>>>(jobs, kmax, G, part);
    bstep_sum_k<<<dim3(kmax, n), 256, 0, s>>>(jobs, kmax, G, part);
    return hipGetLastError();
}

// chunks in reverse order of bstep_dots_k (see lz_update_k)
__global__ void __launch_bounds__(BV_BLOCK) bupdate_norm_k(const UpdJob* __restrict__ jobs, int G,
                                                           double* __restrict__ part)
{
    __shared__ double c[MD_MAXK];
    __shared__ double red[BV_BLOCK / 64];
    const UpdJob& j = jobs[blockIdx.y];
    const int nb = (int)((j.n + BV_CHUNK - 1) / BV_CHUNK);
    if ((int)blockIdx.x >= nb) return;
    for (int i = threadIdx.x; i < j.k; i += BV_BLOCK) c[i] = j.coef[i];
    __syncthreads();
    const int blk = nb - 1 - blockIdx.x;
    const long c0 = (long)blk * BV_CHUNK;
    double2 acc[BV_PAIRS];
#pragma unroll
    for (int e = 0; e < BV_PAIRS; e++) {
        const long idx = c0 + 2 * ((long)e * BV_BLOCK + threadIdx.x);
        acc[e] = idx < j.n ? *(const double2*)(j.w + idx) : make_double2(0.0, 0.0);
    }
    for (int i = 0; i < j.k; i++) {
        const double* vi = j.V + (long)i * j.ldv;
        const double ci = c[i];
#pragma unroll
        for (int e = 0; e < BV_PAIRS; e++) {
            const long idx = c0 + 2 * ((long)e * BV_BLOCK + threadIdx.x);
            if (idx < j.n) {
                const double2 p = *(const double2*)(vi + idx);
                acc[e].x -= ci * p.x;
                acc[e].y -= ci * p.y;
            }
        }
    }
    double sq = 0.0;
#pragma unroll
    for (int e = 0; e < BV_PAIRS; e++) {
        const long idx = c0 + 2 * ((long)e * BV_BLOCK + threadIdx.x);
        if (idx < j.n) {
            *(double2*)(j.w + idx) = acc[e];
            sq += acc[e].x * acc[e].x + acc[e].y * acc[e].y;
        }
    }
    sq = wave_sum(sq);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
    __syncthreads();
    if (threadIdx.x == 0) part[(size_t)blockIdx.y * G + blk] = (red[0] + red[1]) + (red[2] + red[3]);
}
__global__ void __launch_bounds__(256) bupdate_sum_k(const UpdJob* __restrict__ jobs, int G,
                                                     const double* __restrict__ part)
{
    __shared__ double red[4];
    const UpdJob& j = jobs[blockIdx.x];
    const long nb = (j.n + BV_CHUNK - 1) / BV_CHUNK;
    const double* pq = part + (size_t)blockIdx.x * G;
    double acc = 0.0;
    for (long b = threadIdx.x; b < nb; b += 256) acc += pq[b];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) j.out[0] = (red[0] + red[1]) + (red[2] + red[3]);
}
hipError_t bupdate_norm(const UpdJob* jobs, int n, long nmax, double* part, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const int G = (int)((nmax + BV_CHUNK - 1) / BV_CHUNK);
    bupdate_norm_k<<<dim3(G, n), BV_BLOCK, 0, s>>>(jobs, G, part);
    bupdate_sum_k<<<n, 256, 0, s>>>(jobs, G, part);
    return hipGetLastError();
}

// deviation from the identity, many matrices: 64 workgroups per job
__global__ void __launch_bounds__(256) beye_dev_k(const EyeJob* __restrict__ jobs, double* __restrict__ part)
{
    __shared__ double red[4];
    const EyeJob& j = jobs[blockIdx.y];
    double m = 0.0;
    const long tot = (long)j.n * j.n;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < tot; e += (long)gridDim.x * 256) {
        const long i = e / j.n, c = e - i * j.n;
        const double v = j.G[i * j.ld + c] - (i == c ? 1.0 : 0.0);
        m = fmax(m, isfinite(v) ? fabs(v) : 1e300);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) part[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}
__global__ void __launch_bounds__(64) beye_max_k(const EyeJob* __restrict__ jobs, int G, const double* __restrict__ part)
{
    double m = 0.0;
    for (int b = threadIdx.x; b < G; b += 64) m = fmax(m, part[(size_t)blockIdx.x * G + b]);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if (threadIdx.x == 0) jobs[blockIdx.x].out[0] = m;
}
hipError_t beye_deviation(const EyeJob* jobs, int n, double* part, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    beye_dev_k<<<dim3(64, n), 256, 0, s>>>(jobs, part);
    beye_max_k<<<n, 64, 0, s>>>(jobs, 64, part);
    return hipGetLastError();
}

// strided 2-D copies, one job per problem: grid (column blocks, rows, problem)
__global__ void __launch_bounds__(256) bcopy2_k(const Copy2Job* __restrict__ jobs)
{
    const Copy2Job& j = jobs[blockIdx.z];
    const int col = blockIdx.x * 256 + threadIdx.x;
    const int row = blockIdx.y;
    if (col >= j.co || row >= j.ro) return;
    j.out[row * j.so0 + col * j.so1] = (row < j.r && col < j.c) ? j.in[row * j.si0 + col * j.si1] : 0.0;
}
hipError_t bcopy2(const Copy2Job* jobs, int n, int romax, int comax, hipStream_t s)
{
    if (n <= 0 || romax <= 0 || comax <= 0) return hipSuccess;
    bcopy2_k<<<dim3((comax + 255) / 256, romax, n), 256, 0, s>>>(jobs);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256) badd_diag_k(const DiagJob* __restrict__ jobs)
{
    const DiagJob& j = jobs[blockIdx.y];
    const int i = j.i0 + blockIdx.x * 256 + threadIdx.x;
    if (i < j.i1) j.G[(long)i * j.ld + i] += j.v;
}
hipError_t badd_diag(const DiagJob* jobs, int n, int lenmax, hipStream_t s)
{
    if (n <= 0 || lenmax <= 0) return hipSuccess;
    badd_diag_k<<<dim3((lenmax + 255) / 256, n), 256, 0, s>>>(jobs);
    return hipGetLastError();
}

// w = beta w + cscale sum_i coef[i] V_i
__global__ void __launch_bounds__(256) bgemv_k(const GemvJob* __restrict__ jobs)
{
    __shared__ double cf[MD_MAXK];
    const GemvJob& j = jobs[blockIdx.y];
    for (int i = threadIdx.x; i < j.k; i += 256) cf[i] = j.coef[i] * j.cscale;
    __syncthreads();
    for (long idx = blockIdx.x * 256L + threadIdx.x; idx < j.n; idx += (long)gridDim.x * 256) {
        double acc = (j.beta == 0.0) ? 0.0 : j.beta * j.w[idx];
        for (int i = 0; i < j.k; i++) acc += cf[i] * j.V[(long)i * j.ldv + idx];
        j.w[idx] = acc;
    }
}
hipError_t bgemv(const GemvJob* jobs, int n, long nmax, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    long blocks = (nmax + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    bgemv_k<<<dim3(blocks, n), 256, 0, s>>>(jobs);
    return hipGetLastError();
}

// w -= alpha[0] v + beta u
__global__ void __launch_bounds__(256) bthree_k(const ThreeJob* __restrict__ jobs)
{
    const ThreeJob& j = jobs[blockIdx.y];
    const double a = j.alpha[0];
    for (long i = blockIdx.x * 256L + threadIdx.x; i < j.n; i += (long)gridDim.x * 256) {
        double r = j.w[i] - a * j.v[i];
        if (j.u) r -= j.beta * j.u[i];
        j.w[i] = r;
    }
}
hipError_t bthree(const ThreeJob* jobs, int n, long nmax, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    long blocks = (nmax + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    bthree_k<<<dim3(blocks, n), 256, 0, s>>>(jobs);
    return hipGetLastError();
}

// y = a x
__global__ void __launch_bounds__(256) bscale_k(const ScaleJob* __restrict__ jobs)
{
    const ScaleJob& j = jobs[blockIdx.y];
    const double a = j.a_sq ? 1.0 / sqrt(*j.a_sq) : j.a;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < j.n; i += (long)gridDim.x * 256) j.y[i] = a * j.x[i];
}
hipError_t bscale(const ScaleJob* jobs, int n, long nmax, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    long blocks = (nmax + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    bscale_k<<<dim3(blocks, n), 256, 0, s>>>(jobs);
    return hipGetLastError();
}

// the scaling of the next Krylov vector and its FP32 copy in one pass
__global__ void __launch_bounds__(256) bscale_conv_k(const ScaleConvJob* __restrict__ jobs)
{
    const ScaleConvJob& j = jobs[blockIdx.y];
    const double a = j.a_sq ? 1.0 / sqrt(*j.a_sq) : j.a;
    const double* x = j.x;  // y may be x (in place)
    double* y = j.y;
    float* __restrict__ y32 = j.y32;
    const long n = j.n;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        const double v = a * x[i];
        y[i] = v;
        y32[i] = (float)v;
    }
}
hipError_t bscale_conv(const ScaleConvJob* jobs, int n, long nmax, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    long blocks = (nmax + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    bscale_conv_k<<<dim3(blocks, n), 256, 0, s>>>(jobs);
    return hipGetLastError();
}

// FP64 -> FP32 copy
__global__ void __launch_bounds__(256) bconvert_k(const ConvJob* __restrict__ jobs)
{
    const ConvJob& j = jobs[blockIdx.y];
    for (long i = blockIdx.x * 256L + threadIdx.x; i < j.n; i += (long)gridDim.x * 256) j.y[i] = (float)j.x[i];
}
hipError_t bconvert(const ConvJob* jobs, int n, long nmax, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    long blocks = (nmax + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    bconvert_k<<<dim3(blocks, n), 256, 0, s>>>(jobs);
    return hipGetLastError();
}

// MPO mixing (FP32 in, TO out) for many problems, the problem in grid z.  A
// workgroup takes bw values of b times 256 / bw of x, bw the largest of 256, 128
// and 64 that leaves no more threads idle than 64 does (128 chains of 32 to 256: 48
// us with 64 throughout, 43 so).
__host__ __device__ static inline int bwmix_width(int Bn)
{
    const int pad = (Bn + 63) & ~63;
    return ((Bn + 255) & ~255) == pad ? 256 : (((Bn + 127) & ~127) == pad ? 128 : 64);
}
template <typename TO, bool STG>
__global__ void __launch_bounds__(256) bwmix_k(const MixJob* __restrict__ jobs, int groups)
{
    __shared__ typename std::conditional<STG, MixLds<float>, int>::type lds;
    const MixJob& j = jobs[blockIdx.z / groups];
    const int bw = bwmix_width(j.Bn), rows = 256 / bw, nb = (j.Bn + bw - 1) / bw;
    const int by = blockIdx.x / nb, bx = blockIdx.x - by * nb;
    if (by * rows >= j.X) return;  // the whole workgroup
    const MixTable t = j.t;
    const bool idt = t.esel != nullptr;
    const MixView<float, STG, false> m = mix_view<float, STG>(t, (MixLds<float>*)&lds);
    const int b = bx * bw + (threadIdx.x & (bw - 1));
    const long x = by * rows + (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * 64) / bw;
    if (b >= j.Bn || x >= j.X) return;
    const float* ip = (const float*)j.in + x * j.isx + b;
    TO* op = (TO*)j.out + x * j.osx + b;
    const float* ip2 = idt ? j.in2 + x * j.isx2 + b : nullptr;
    for (int o = blockIdx.z % groups; o < t.nout; o += groups) {
        const int e0 = m.optr(o), e1 = m.optr(o + 1);
        float acc = 0.0f;
#pragma unroll 4
        for (int e = e0; e < e1; e++)
            acc += m.eval(e) * (idt && m.esel(e) ? ip2[m.eoff(e)] : ip[m.eoff(e)]);
        if (idt && m.osel(o)) j.out2[x * j.osx2 + m.ooff(o) + b] = (double)acc;
        else op[m.ooff(o)] = cvt_from_f<TO>(acc);
    }
}
hipError_t bwmix(int tout, const MixJob* jobs, int n, int Xmax, int Bnmax, int nout_max, int nnz_max, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    // workgroups of the widest problem: no width takes more than 64 does
    dim3 grid(((Bnmax + 63) / 64) * ((Xmax + 3) / 4));
    const int groups = mix_groups((long)grid.x * n, nout_max);
    grid.z = n * groups;
    const bool stg = nout_max <= MIX_MAXO && nnz_max <= MIX_MAXE;
    if (tout == T_F32 && stg) bwmix_k<float, true><<<grid, 256, 0, s>>>(jobs, groups);
    else if (tout == T_F32) bwmix_k<float, false><<<grid, 256, 0, s>>>(jobs, groups);
    else if (tout == T_F64 && stg) bwmix_k<double, true><<<grid, 256, 0, s>>>(jobs, groups);
    else if (tout == T_F64) bwmix_k<double, false><<<grid, 256, 0, s>>>(jobs, groups);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace tn
