// tn_gemm.hip -- the matrix-core GEMMs (gfx950).
//
// * gemm_pipe_k : FP64 and FP32 GEMM (v_mfma 16x16x4), operands copied straight
//                into LDS, several stages deep, XCD-aware tile order.  The three
//                stages of Heff*psi and of the environment updates
//                (MPSSite_Contractions.C:155-400) are GEMMs once the MPO index is
//                mixed (wmix, tn_kernels.hip).
// * gemm_grouped_k : one launch over the tiles of many problems.
// * gemm_k     : bf16 GEMM, register-prefetch pipelined.
// * gemm_x3_k  : the split-bfloat16 product.
// * x3_stage1_mix_k : its Heff stage 1 with the MPO stage in the epilogue.
#include "tn_device.h"

namespace tn {

struct GemmParams {
    const void* A;
    const void* B;
    void* C;
    int M, N, K;
    long lda, ldb, ldc, sA, sB, sC;
    float alpha;
    int accumulate;
};

// element j of a 16-byte vector of bfloat16 values
__device__ __forceinline__ bf16 vec_elem(const u32x4& v, int j)
{
    const uint32_t w = (j >> 1) == 0 ? v.x : ((j >> 1) == 1 ? v.y : ((j >> 1) == 2 ? v.z : v.w));
    return (bf16)((j & 1) ? (w >> 16) : (w & 0xffffu));
}

// global -> registers for one bfloat16 operand tile (ROWS x BK, K-major in LDS)
//   KM  : operand(row, k) = G[row*ld + k]   (vector loads along k)
//   !KM : operand(row, k) = G[k*ld + row]   (vector loads along row)
template <int ROWS, int BK, bool KM, int R>
__device__ __forceinline__ void tile_gload(u32x4 (&rg)[R], const bf16* __restrict__ G, long ld,
                                           int r0, int k0, int tid)
{
    constexpr int VEC = MT<bf16>::VEC;
    constexpr int TOT = ROWS * BK / VEC;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int v = tid + r * 256;
        if (TOT % 256 == 0 || v < TOT) {
            if constexpr (KM) {
                const int row = v / (BK / VEC), kv = v % (BK / VEC);
                rg[r] = *(const u32x4*)(G + (long)(r0 + row) * ld + k0 + kv * VEC);
            } else {
                const int kk = v / (ROWS / VEC), rv = v % (ROWS / VEC);
                rg[r] = *(const u32x4*)(G + (long)(k0 + kk) * ld + r0 + rv * VEC);
            }
        }
    }
}
template <int ROWS, int BK, bool KM, int R>
__device__ __forceinline__ void tile_sstore(const u32x4 (&rg)[R], bf16* __restrict__ S, int tid)
{
    constexpr int VEC = MT<bf16>::VEC;
    constexpr int TOT = ROWS * BK / VEC;
    constexpr int LDK = BK + MT<bf16>::PAD;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int v = tid + r * 256;
        if (TOT % 256 == 0 || v < TOT) {
            if constexpr (KM) {
                const int row = v / (BK / VEC), kv = v % (BK / VEC);
                *(u32x4*)(S + row * LDK + kv * VEC) = rg[r];
            } else {
                const int kk = v / (ROWS / VEC), rv = v % (ROWS / VEC);
#pragma unroll
                for (int j = 0; j < VEC; j++) S[(rv * VEC + j) * LDK + kk] = vec_elem(rg[r], j);
            }
        }
    }
}

// One BM x BN output tile of a bfloat16 product: 256 threads = 4 waves in a 2x2
// arrangement, wave tile (BM/2) x (BN/2); operand tiles staged through LDS (As,
// Bs) with the next K-slice prefetched into registers.
template <typename TO, int BM, int BN, int BK, bool AKM, bool BKM>
__device__ __forceinline__ void gemm_tile(const bf16* __restrict__ A, const bf16* __restrict__ B, TO* __restrict__ C,
                                          long lda, long ldb, long ldc, int K, float alpha, int accumulate,
                                          int m0, int n0, bf16* __restrict__ As, bf16* __restrict__ Bs)
{
    typedef MT<bf16> T;
    typedef typename T::frag_t frag_t;
    typedef typename T::acc_t acc_t;
    constexpr int LDK = BK + T::PAD;
    constexpr int WM = BM / 2, WN = BN / 2, FM = WM / 16, FN = WN / 16;
    constexpr int VEC = T::VEC;
    constexpr int TA = BM * BK / VEC, TB = BN * BK / VEC;
    constexpr int RA = (TA + 255) / 256, RB = (TB + 255) / 256;
    static_assert(FM >= 1 && FN >= 1, "tile");
    static_assert(BK % T::MK == 0, "BK");

    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int wm0 = (wid >> 1) * WM, wn0 = (wid & 1) * WN;

    u32x4 ra[RA], rb[RB];
    acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = 0;

    const int nk = K / BK;
    tile_gload<BM, BK, AKM>(ra, A, lda, m0, 0, tid);
    tile_gload<BN, BK, BKM>(rb, B, ldb, n0, 0, tid);
    tile_sstore<BM, BK, AKM>(ra, As, tid);
    tile_sstore<BN, BK, BKM>(rb, Bs, tid);
    __syncthreads();
    for (int t = 0; t < nk; t++) {
        if (t + 1 < nk) {
            tile_gload<BM, BK, AKM>(ra, A, lda, m0, (t + 1) * BK, tid);
            tile_gload<BN, BK, BKM>(rb, B, ldb, n0, (t + 1) * BK, tid);
        }
        // the MFMA section of a slice at raised wave priority: a wave that has
        // its operands in LDS issues ahead of waves still loading or storing
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < BK; kk += T::MK) {
            frag_t a[FM], b[FN];
#pragma unroll
            for (int i = 0; i < FM; i++)
                a[i] = *(const frag_t*)(As + (wm0 + i * 16 + (lane & 15)) * LDK + kk + (lane >> 4) * T::KPL);
#pragma unroll
            for (int j = 0; j < FN; j++)
                b[j] = *(const frag_t*)(Bs + (wn0 + j * 16 + (lane & 15)) * LDK + kk + (lane >> 4) * T::KPL);
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) acc[i][j] = mma(a[i], b[j], acc[i][j]);
        }
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();
        if (t + 1 < nk) {
            tile_sstore<BM, BK, AKM>(ra, As, tid);
            tile_sstore<BN, BK, BKM>(rb, Bs, tid);
            __syncthreads();
        }
    }
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const long row = m0 + wm0 + i * 16 + T::crow(lane, r);
                const long col = n0 + wn0 + j * 16 + (lane & 15);
                TO* cp = C + row * ldc + col;
                if constexpr (std::is_same<TO, double>::value) {
                    double v = (double)acc[i][j][r] * (double)alpha;
                    if (accumulate) v += to_d(*cp);
                    *cp = cvt_from_d<TO>(v);
                } else {
                    float v = (float)acc[i][j][r] * alpha;
                    if (accumulate) v += to_f(*cp);
                    *cp = cvt_from_f<TO>(v);
                }
            }
}

template <typename TO, int BM, int BN, int BK, bool AKM, bool BKM>
__global__ void __launch_bounds__(256) gemm_k(GemmParams p)
{
    constexpr int LDK = BK + MT<bf16>::PAD;
    __shared__ __attribute__((aligned(16))) bf16 As[BM * LDK];
    __shared__ __attribute__((aligned(16))) bf16 Bs[BN * LDK];
    const int ntn = p.N / BN, ntm = p.M / BM;
    const int nblk = ntn * ntm;
    int bid = blockIdx.x;
    // consecutive block ids land on different XCDs; give each XCD a contiguous
    // range of output tiles so tiles sharing operands share an L2
    if ((nblk & 7) == 0) bid = (bid & 7) * (nblk >> 3) + (bid >> 3);
    // inside the range, GM tile rows at a time and column by column within
    // them: the tiles resident together on an XCD share GM row blocks of A and
    // a few column blocks of B, instead of one row block of A and all of B
    constexpr int GM = 8;
    const int gsz = GM * ntn, g = bid / gsz, first = g * GM;
    const int rows = ntm - first < GM ? ntm - first : GM;
    const int local = bid - g * gsz;
    const int tm = first + local % rows, tn = local / rows;
    const long bz = blockIdx.y;
    gemm_tile<TO, BM, BN, BK, AKM, BKM>((const bf16*)p.A + bz * p.sA, (const bf16*)p.B + bz * p.sB,
                                            (TO*)p.C + bz * p.sC, p.lda, p.ldb, p.ldc, p.K, p.alpha,
                                            p.accumulate, tm * BM, tn * BN, As, Bs);
}

// ---------------------------------------------------------------------------
// FP64 and FP32 tiles, staged by the copy engine of the vector memory path:
// global memory straight into LDS (no registers, no LDS store instructions),
// S stages deep, one barrier per K step.  Bound by the matrix pipes once two
// waves per SIMD are resident; what the register-staged loop (gemm_tile) lost
// was the wait for its stores and its second barrier per step.  FP64,
// 3072 x 4096 x 1024: 419 us (register-staged, its best tile) -> 364 us, 70.7
// of the 72.6 TFLOP/s a large library product reaches.
//
// An operand stage holds 128 bytes of K per row as 16-byte units (K-major
// operands: [row][unit], row-major ones: [k][row]).  A copy writes 64
// consecutive units in lane order, so the bank swizzle is applied to the
// global address: slot u of row r holds unit u ^ (r & 7) (K-major), slot u of
// k-row k holds unit u ^ sw(k) (row-major).  Fragment reads then touch every
// bank once per 128 bytes.
__device__ __forceinline__ uint32_t lds_offset(const void* p)
{
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}
// 64 lanes copy 16 bytes each from base + off (off per lane, 32 bits unsigned) to
// LDS address dst + 16 * lane (dst uniform).  The instruction takes dst from M0.  M0
// is reserved: the compiler writes it right before an instruction of its own that
// reads it and keeps nothing there otherwise, so it need not be preserved (putting
// the old value back cost 2-3 % of an apply at a left bond of 64); the clobber, of
// which clang warns for reserved registers, keeps such a write from moving or
// being shared across a copy.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void copy_to_lds(const void* base, uint32_t off, uint32_t dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(dst), "v"(off), "s"(base)
                 : "memory", "m0");
}
__device__ __forceinline__ void copy_to_lds(const void* base, uint64_t off, uint32_t dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(dst), "v"((const char*)base + off)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
// all but the last N copies have arrived and every LDS read has returned
template <int N> __device__ __forceinline__ void wait_copies()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory");
}

// one operand's stage: ROWS x BK values, loads and fragment reads
template <typename TI, int ROWS, int BK, bool KM> struct Stage {
    static constexpr int E = 16 / sizeof(TI);          // values per unit
    static constexpr int UNITS = ROWS * BK / E;        // units per stage
    static constexpr int UPK = BK / E;                 // units per row (K-major)
    static constexpr int UPR = ROWS / E;               // units per k-row (row-major)
    static constexpr bool F64 = sizeof(TI) == 8;
    static __device__ __forceinline__ int rsw(int row)
    {
        return UPK == 8 && !F64 ? (row & 7) : ((row >> 1) & (UPK - 1));
    }
    static __device__ __forceinline__ int ksw(int k)
    {
        return (F64 ? (((k >> 1) & 1) << 3) : ((k & 3) << 2)) & (UPR - 1);
    }
    // byte offset, from the operand's first row and K index of the step, of the
    // unit that slot `slot` holds
    template <typename OFF> static __device__ __forceinline__ OFF goff(int slot, long ld)
    {
        if constexpr (KM) {
            const int row = slot / UPK, u = (slot % UPK) ^ rsw(row);
            return (OFF)((row * ld + u * E) * (long)sizeof(TI));
        } else {
            const int k = slot / UPR, u = (slot % UPR) ^ ksw(k);
            return (OFF)((k * ld + u * E) * (long)sizeof(TI));
        }
    }
    // values between the starts of consecutive K steps
    static __device__ __forceinline__ long kstep(long ld) { return KM ? (long)BK : (long)BK * ld; }
    // operand(row, k)
    static __device__ __forceinline__ TI at(const TI* S, int row, int k)
    {
        if constexpr (KM) return S[row * BK + (((k / E) ^ rsw(row)) * E) + k % E];
        else return S[k * ROWS + ((row / E) ^ ksw(k)) * E + row % E];
    }
};

template <int BM, int BN, int BK, int S, typename TI> constexpr int stage_bytes()
{
    return S * (BM + BN) * BK * (int)sizeof(TI);
}

// One BM x BN output tile: WGM x WGN waves of (BM / WGM) x (BN / WGN).  The
// caller's LDS holds S stages (stage_bytes) and is free when the tile starts;
// every copy has arrived and every LDS read has returned when it ends, but
// other waves may still be reading (barrier before reusing the LDS).
//
// Sums over k in increasing order for every tile shape and operand layout (a
// 16-byte FP64 fragment read, two k per lane, would give another order and only
// 2-4 % more speed at 3072 x 4096 x 1024).
//
// A lane keeps its copies' offsets as 32-bit registers beside a uniform base;
// WIDE holds them in 64 bits, for operands whose rows lie too far apart (see
// gemm_wide).
template <typename TI, typename TO, int BM, int BN, int BK, int WGM, int WGN, int S, bool AKM, bool BKM, bool WIDE>
__device__ __forceinline__ void pipe_tile(const TI* __restrict__ A, const TI* __restrict__ B, TO* __restrict__ C,
                                          long lda, long ldb, long ldc, int K, float alpha, int accumulate, int m0,
                                          int n0, TI* __restrict__ sm)
{
    typedef MT<TI> T;
    typedef typename T::acc_t acc_t;
    typedef Stage<TI, BM, BK, AKM> SA;
    typedef Stage<TI, BN, BK, BKM> SB;
    constexpr int NW = WGM * WGN, WM = BM / WGM, WN = BN / WGN, FM = WM / 16, FN = WN / 16;
    constexpr int CA = SA::UNITS / 64, CB = SB::UNITS / 64, CH = CA + CB;
    static_assert(FM * 16 * WGM == BM && FN * 16 * WGN == BN, "wave tile");
    static_assert(CA * 64 == SA::UNITS && CB * 64 == SB::UNITS && CH % NW == 0, "copies per wave");
    constexpr int L = CH / NW;              // copies per wave and step
    constexpr int STG = (BM + BN) * BK;     // values per stage
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm0 = (wid / WGN) * WM, wn0 = (wid % WGN) * WN;
    const int r = lane & 15, kq = lane >> 4;

    const TI* Ab = AKM ? A + (long)m0 * lda : A + m0;
    const TI* Bb = BKM ? B + (long)n0 * ldb : B + n0;
    typedef typename std::conditional<WIDE, uint64_t, uint32_t>::type OFF;
    OFF off[L];
#pragma unroll
    for (int i = 0; i < L; i++) {
        const int c = wid * L + i;
        off[i] = c < CA ? SA::template goff<OFF>(c * 64 + lane, lda) : SB::template goff<OFF>((c - CA) * 64 + lane, ldb);
    }
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_offset(sm));
    const long ka = SA::kstep(lda), kb = SB::kstep(ldb);
    auto issue = [&](int st) {  // the next K step into stage st
#pragma unroll
        for (int i = 0; i < L; i++) {
            const int c = wid * L + i;
            copy_to_lds(c < CA ? (const void*)Ab : (const void*)Bb, off[i],
                        base + (uint32_t)(st * STG * (int)sizeof(TI) + c * 1024));
        }
        Ab += ka;
        Bb += kb;
    };
    acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) acc[i][j][q] = 0;

    const int nk = K / BK;
#pragma unroll
    for (int t = 0; t < S - 1; t++)
        if (t < nk) issue(t);
    int st = 0;
    for (int t = 0; t < nk; t++) {
        // stage st has arrived (this wave's copies, then, past the barrier,
        // everyone's), and everyone is done reading the stage before it
        if (t + S - 2 < nk) wait_copies<(S - 2) * L>();
        else wait_copies<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" : : : "memory");  // no LDS read of this step moves above the barrier
        if (t + S - 1 < nk) issue(st == 0 ? S - 1 : st - 1);
        const TI* As = sm + st * STG;
        const TI* Bs = As + BM * BK;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            TI a[FM], b[FN];
#pragma unroll
            for (int i = 0; i < FM; i++) a[i] = SA::at(As, wm0 + i * 16 + r, kk + kq);
#pragma unroll
            for (int j = 0; j < FN; j++) b[j] = SB::at(Bs, wn0 + j * 16 + r, kk + kq);
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) acc[i][j] = mma(a[i], b[j], acc[i][j]);
        }
        __builtin_amdgcn_s_setprio(0);
        asm volatile("" : : : "memory");  // nor below the next one's wait
        st = st + 1 == S ? 0 : st + 1;
    }
    wait_copies<0>();
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const long row = m0 + wm0 + i * 16 + T::crow(lane, q);
                const long col = n0 + wn0 + j * 16 + r;
                TO* cp = C + row * ldc + col;
                if constexpr (std::is_same<TO, double>::value) {
                    double v = (double)acc[i][j][q] * (double)alpha;
                    if (accumulate) v += to_d(*cp);
                    *cp = v;
                } else {
                    float v = (float)acc[i][j][q] * alpha;
                    if (accumulate) v += to_f(*cp);
                    *cp = cvt_from_f<TO>(v);
                }
            }
}

// XCD-aware tile order: consecutive block ids land on different XCDs, so each
// XCD gets a contiguous range of tiles (also when their number is no multiple of
// 8: FP32 992 x 2976 x 3968 in 32x32, 2883 tiles, 280 us in launch order, 264 so;
// 1504 x 4512 x 6016 870 and 821), and inside it 8 tile rows at a time go
// column by column (tiles resident together share 8 row blocks of A and a few
// column blocks of B)
__device__ __forceinline__ void tile_of_block(int bid, int ntm, int ntn, int& tm, int& tn)
{
    // (two branches: with one formula the compiler read the kernel's arguments later,
    // and the smallest products took 5 % longer)
    const int nblk = ntm * ntn, xcd = bid & 7, rest = nblk & 7;
    if (rest == 0) bid = xcd * (nblk >> 3) + (bid >> 3);
    else bid = xcd * (nblk >> 3) + (xcd < rest ? xcd : rest) + (bid >> 3);
    constexpr int GM = 8;
    const int gsz = GM * ntn, g = bid / gsz, first = g * GM;
    const int rows = ntm - first < GM ? ntm - first : GM;
    const int local = bid - g * gsz;
    tm = first + local % rows;
    tn = local / rows;
}

template <typename TI, typename TO, int BM, int BN, int BK, int WGM, int WGN, int S, int OCC, bool AKM, bool BKM,
          bool WIDE = false>
__global__ void __launch_bounds__(64 * WGM * WGN, OCC) gemm_pipe_k(GemmParams p)
{
    __shared__ __attribute__((aligned(1024))) TI sm[stage_bytes<BM, BN, BK, S, TI>() / sizeof(TI)];
    int tm, tn;
    tile_of_block(blockIdx.x, p.M / BM, p.N / BN, tm, tn);
    const long bz = blockIdx.y;
    pipe_tile<TI, TO, BM, BN, BK, WGM, WGN, S, AKM, BKM, WIDE>(
        (const TI*)p.A + bz * p.sA, (const TI*)p.B + bz * p.sB, (TO*)p.C + bz * p.sC, p.lda, p.ldb, p.ldc, p.K,
        p.alpha, p.accumulate, tm * BM, tn * BN, sm);
}

// Split-product LDS layout for BK = 32: rows of 64 bytes without padding,
// the four 16-byte k-units of row r stored in the order u ^ g(r), g(r) =
// ((r >> 1) ^ (r >> 2)) & 3.  A tile store (lanes 4i .. 4i+3 write the four
// units of one row) and a fragment read (lanes 0..15 read one unit of rows
// 0..15) then fall on distinct banks in every group of 8 or 16 lanes, with
// 32 or with 64 banks of 4 bytes; the padded layout (80-byte rows) leaves the
// stores 2-way conflicted.
__device__ __forceinline__ int x3_swz(int row, int unit) { return row * 32 + ((unit ^ ((row >> 1) ^ (row >> 2))) & 3) * 8; }

template <int ROWS, int BK, int R>
__device__ __forceinline__ void x3_sstore(const u32x4 (&rg)[R], bf16* __restrict__ S, int tid)
{
    constexpr int UPR = BK / 8;  // 16-byte units per row
    constexpr int TOT = ROWS * UPR;
    constexpr int LDK = BK == 32 ? BK : BK + MT<bf16>::PAD;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int v = tid + r * 256;
        if (TOT % 256 == 0 || v < TOT) {
            const int row = v / UPR, kv = v % UPR;
            if constexpr (BK == 32) *(u32x4*)(S + x3_swz(row, kv)) = rg[r];
            else *(u32x4*)(S + row * LDK + kv * 8) = rg[r];
        }
    }
}

// One BM x BN output tile of the split-bfloat16 product: A and B each held as
// three bfloat16 planes (A = A0 + A1 + A2), K-major, every plane staged
// through LDS; each K step issues the six leading cross products A_i B_j
// (i + j <= 2) of v_mfma_f32_16x16x32_bf16 into one FP32 accumulator.  Same
// wave layout, register prefetch and wave-priority scheme as gemm_tile.
template <typename TO, int BM, int BN, int BK>
__device__ __forceinline__ void gemm_tile_x3(const bf16* __restrict__ A, long psA, const bf16* __restrict__ B,
                                             long psB, TO* __restrict__ C, long lda, long ldb, long ldc, int K,
                                             float alpha, int accumulate, int m0, int n0, bf16* __restrict__ As,
                                             bf16* __restrict__ Bs)
{
    typedef MT<bf16> T;
    typedef T::frag_t frag_t;
    typedef T::acc_t acc_t;
    constexpr bool SWZ = BK == 32;
    constexpr int LDK = SWZ ? BK : BK + T::PAD;
    constexpr int WM = BM / 2, WN = BN / 2, FM = WM / 16, FN = WN / 16;
    constexpr int TA = BM * BK / T::VEC, TB = BN * BK / T::VEC;
    constexpr int RA = (TA + 255) / 256, RB = (TB + 255) / 256;
    constexpr int SA = BM * LDK, SB = BN * LDK;
    static_assert(FM >= 1 && FN >= 1 && BK % T::MK == 0, "tile");

    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int wm0 = (wid >> 1) * WM, wn0 = (wid & 1) * WN;
    // LDS element offset of the fragment of row `row` at k-step kk
    auto foff = [&](int row, int kk) {
        if constexpr (SWZ) return x3_swz(row, (lane >> 4) + kk / 8);
        else return row * LDK + kk + (lane >> 4) * T::KPL;
    };

    u32x4 ra[3][RA], rb[3][RB];
    acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = 0;

    const int nk = K / BK;
#pragma unroll
    for (int p = 0; p < 3; p++) {
        tile_gload<BM, BK, true>(ra[p], A + p * psA, lda, m0, 0, tid);
        tile_gload<BN, BK, true>(rb[p], B + p * psB, ldb, n0, 0, tid);
    }
#pragma unroll
    for (int p = 0; p < 3; p++) {
        x3_sstore<BM, BK>(ra[p], As + p * SA, tid);
        x3_sstore<BN, BK>(rb[p], Bs + p * SB, tid);
    }
    __syncthreads();
    for (int t = 0; t < nk; t++) {
        if (t + 1 < nk) {
#pragma unroll
            for (int p = 0; p < 3; p++) {
                tile_gload<BM, BK, true>(ra[p], A + p * psA, lda, m0, (t + 1) * BK, tid);
                tile_gload<BN, BK, true>(rb[p], B + p * psB, ldb, n0, (t + 1) * BK, tid);
            }
        }
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < BK; kk += T::MK) {
            frag_t a[3][FM], b[3][FN];
#pragma unroll
            for (int p = 0; p < 3; p++) {
#pragma unroll
                for (int i = 0; i < FM; i++)
                    a[p][i] = *(const frag_t*)(As + p * SA + foff(wm0 + i * 16 + (lane & 15), kk));
#pragma unroll
                for (int j = 0; j < FN; j++)
                    b[p][j] = *(const frag_t*)(Bs + p * SB + foff(wn0 + j * 16 + (lane & 15), kk));
            }
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) {
                    // smallest terms first
                    acc[i][j] = mma(a[2][i], b[0][j], acc[i][j]);
                    acc[i][j] = mma(a[0][i], b[2][j], acc[i][j]);
                    acc[i][j] = mma(a[1][i], b[1][j], acc[i][j]);
                    acc[i][j] = mma(a[1][i], b[0][j], acc[i][j]);
                    acc[i][j] = mma(a[0][i], b[1][j], acc[i][j]);
                    acc[i][j] = mma(a[0][i], b[0][j], acc[i][j]);
                }
        }
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();
        if (t + 1 < nk) {
#pragma unroll
            for (int p = 0; p < 3; p++) {
                x3_sstore<BM, BK>(ra[p], As + p * SA, tid);
                x3_sstore<BN, BK>(rb[p], Bs + p * SB, tid);
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const long row = m0 + wm0 + i * 16 + T::crow(lane, r);
                const long col = n0 + wn0 + j * 16 + (lane & 15);
                TO* cp = C + row * ldc + col;
                if constexpr (std::is_same<TO, double>::value) {
                    double v = (double)acc[i][j][r] * (double)alpha;
                    if (accumulate) v += *cp;
                    *cp = v;
                } else {
                    float v = acc[i][j][r] * alpha;
                    if (accumulate) v += to_f(*cp);
                    *cp = cvt_from_f<TO>(v);
                }
            }
}

struct GemmX3Params {
    const bf16* A;
    const bf16* B;
    void* C;
    int M, N, K;
    long lda, ldb, ldc, sA, sB, sC, psA, psB;
    float alpha;
    int accumulate;
};

template <typename TO, int BM, int BN, int BK>
__global__ void __launch_bounds__(256) gemm_x3_k(GemmX3Params p)
{
    constexpr int LDK = BK == 32 ? BK : BK + MT<bf16>::PAD;
    __shared__ __attribute__((aligned(16))) bf16 As[3 * BM * LDK];
    __shared__ __attribute__((aligned(16))) bf16 Bs[3 * BN * LDK];
    const int ntn = p.N / BN, ntm = p.M / BM;
    const int nblk = ntn * ntm;
    int bid = blockIdx.x;
    // XCD-aware tile order as in gemm_k
    if ((nblk & 7) == 0) bid = (bid & 7) * (nblk >> 3) + (bid >> 3);
    constexpr int GM = 8;
    const int gsz = GM * ntn, g = bid / gsz, first = g * GM;
    const int rows = ntm - first < GM ? ntm - first : GM;
    const int local = bid - g * gsz;
    const int tm = first + local % rows, tn = local / rows;
    const long bz = blockIdx.y;
    gemm_tile_x3<TO, BM, BN, BK>(p.A + bz * p.sA, p.psA, p.B + bz * p.sB, p.psB, (TO*)p.C + bz * p.sC, p.lda, p.ldb,
                                 p.ldc, p.K, p.alpha, p.accumulate, tm * BM, tn * BN, As, Bs);
}

// The split product with eight waves per workgroup and one workgroup per CU
// (the whole chip in one round at the bulk shapes: 3072 x 4096 in 192 x 256
// tiles, 1024 x 3072 in 256 x 192 tiles with a 4-way K split).  Wave grid
// WGM x WGN, wave tile (BM / WGM) x (BN / WGN) = 96 x 64 or 64 x 96: 0.28 KB
// of LDS traffic per MFMA against 0.44 KB for the 96 x 128 four-wave tile.
// Same swizzled LDS layout, register prefetch and priority scheme; the
// fragments of B are loaded column block by column block to bound registers.
template <int ROWS, int R>
__device__ __forceinline__ void x3w_gload(u32x4 (&rg)[R], const bf16* __restrict__ G, long ld, int r0, int k0, int tid)
{
    constexpr int TOT = ROWS * 4;  // 16-byte units of a 32-wide K slice
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int v = tid + r * 512;
        if (TOT % 512 == 0 || v < TOT) rg[r] = *(const u32x4*)(G + (long)(r0 + v / 4) * ld + k0 + (v % 4) * 8);
    }
}
template <int ROWS, int R>
__device__ __forceinline__ void x3w_sstore(const u32x4 (&rg)[R], bf16* __restrict__ S, int tid)
{
    constexpr int TOT = ROWS * 4;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int v = tid + r * 512;
        if (TOT % 512 == 0 || v < TOT) *(u32x4*)(S + x3_swz(v / 4, v % 4)) = rg[r];
    }
}

template <typename TO, int BM, int BN, int WGM, int WGN, bool DB>
__global__ void __launch_bounds__(512) gemm_x3w_k(GemmX3Params p)
{
    typedef MT<bf16> T;
    typedef T::frag_t frag_t;
    typedef T::acc_t acc_t;
    static_assert(WGM * WGN == 8, "eight waves");
    constexpr int BK = 32;
    constexpr int WM = BM / WGM, WN = BN / WGN, FM = WM / 16, FN = WN / 16;
    static_assert(FM * 16 == WM && FN * 16 == WN, "wave tile");
    constexpr int RA = (BM * 4 + 511) / 512, RB = (BN * 4 + 511) / 512;
    constexpr int SA = BM * BK, SB = BN * BK;
    // DB: two LDS stages, the next K slice stored into the other stage while
    // the current one is in use, one barrier per step
    constexpr int NS = DB ? 2 : 1;
    __shared__ __attribute__((aligned(16))) bf16 As[NS * 3 * SA];
    __shared__ __attribute__((aligned(16))) bf16 Bs[NS * 3 * SB];

    const int ntn = p.N / BN, ntm = p.M / BM;
    const int nblk = ntn * ntm;
    int bid = blockIdx.x;
    if ((nblk & 7) == 0) bid = (bid & 7) * (nblk >> 3) + (bid >> 3);
    constexpr int GM = 8;
    const int gsz = GM * ntn, g = bid / gsz, first = g * GM;
    const int rows = ntm - first < GM ? ntm - first : GM;
    const int local = bid - g * gsz;
    const int m0 = (first + local % rows) * BM, n0 = (local / rows) * BN;
    const long bz = blockIdx.y;
    const bf16* __restrict__ A = p.A + bz * p.sA;
    const bf16* __restrict__ B = p.B + bz * p.sB;
    TO* __restrict__ C = (TO*)p.C + bz * p.sC;
    const long lda = p.lda, ldb = p.ldb, psA = p.psA, psB = p.psB;

    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int wm0 = (wid / WGN) * WM, wn0 = (wid % WGN) * WN;

    u32x4 ra[3][RA], rb[3][RB];
    acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = 0;

    const int nk = p.K / BK;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        x3w_gload<BM>(ra[q], A + q * psA, lda, m0, 0, tid);
        x3w_gload<BN>(rb[q], B + q * psB, ldb, n0, 0, tid);
    }
#pragma unroll
    for (int q = 0; q < 3; q++) {
        x3w_sstore<BM>(ra[q], As + q * SA, tid);
        x3w_sstore<BN>(rb[q], Bs + q * SB, tid);
    }
    __syncthreads();
    for (int t = 0; t < nk; t++) {
        const int st = DB ? (t & 1) : 0;
        const bf16* Ac = As + st * 3 * SA;
        const bf16* Bc = Bs + st * 3 * SB;
        if (t + 1 < nk) {
#pragma unroll
            for (int q = 0; q < 3; q++) {
                x3w_gload<BM>(ra[q], A + q * psA, lda, m0, (t + 1) * BK, tid);
                x3w_gload<BN>(rb[q], B + q * psB, ldb, n0, (t + 1) * BK, tid);
            }
        }
        __builtin_amdgcn_s_setprio(1);
        frag_t a[3][FM];
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int i = 0; i < FM; i++)
                a[q][i] = *(const frag_t*)(Ac + q * SA + x3_swz(wm0 + i * 16 + (lane & 15), lane >> 4));
#pragma unroll
        for (int j = 0; j < FN; j++) {
            frag_t b[3];
#pragma unroll
            for (int q = 0; q < 3; q++)
                b[q] = *(const frag_t*)(Bc + q * SB + x3_swz(wn0 + j * 16 + (lane & 15), lane >> 4));
#pragma unroll
            for (int i = 0; i < FM; i++) {
                // smallest terms first
                acc[i][j] = mma(a[2][i], b[0], acc[i][j]);
                acc[i][j] = mma(a[0][i], b[2], acc[i][j]);
                acc[i][j] = mma(a[1][i], b[1], acc[i][j]);
                acc[i][j] = mma(a[1][i], b[0], acc[i][j]);
                acc[i][j] = mma(a[0][i], b[1], acc[i][j]);
                acc[i][j] = mma(a[0][i], b[0], acc[i][j]);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        if constexpr (DB) {
            // the other stage was last read in step t - 1, before the barrier
            // that ended it
            if (t + 1 < nk) {
                bf16* An = As + (st ^ 1) * 3 * SA;
                bf16* Bn = Bs + (st ^ 1) * 3 * SB;
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    x3w_sstore<BM>(ra[q], An + q * SA, tid);
                    x3w_sstore<BN>(rb[q], Bn + q * SB, tid);
                }
            }
            __syncthreads();
        } else {
            __syncthreads();
            if (t + 1 < nk) {
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    x3w_sstore<BM>(ra[q], As + q * SA, tid);
                    x3w_sstore<BN>(rb[q], Bs + q * SB, tid);
                }
                __syncthreads();
            }
        }
    }
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const long row = m0 + wm0 + i * 16 + T::crow(lane, r);
                const long col = n0 + wn0 + j * 16 + (lane & 15);
                TO* cp = C + row * p.ldc + col;
                if constexpr (std::is_same<TO, double>::value) {
                    double v = (double)acc[i][j][r] * (double)p.alpha;
                    if (p.accumulate) v += *cp;
                    *cp = v;
                } else {
                    float v = acc[i][j][r] * p.alpha;
                    if (p.accumulate) v += to_f(*cp);
                    *cp = cvt_from_f<TO>(v);
                }
            }
}

// Grouped GEMM: one persistent launch over the output tiles of many problems
// (problem q owns tiles [off[q], off[q+1]), row-major over its N/BN columns).
// Workgroups stride over the tile list; the owning problem is found by a
// binary search of off.
template <typename TI, typename TO, int BM, int BN, int BK, int WGM, int WGN, int S, int OCC, bool AKM, bool BKM>
__global__ void __launch_bounds__(256, OCC) gemm_grouped_k(const GemmProb* __restrict__ probs,
                                                           const int* __restrict__ off, int nprob)
{
    __shared__ __attribute__((aligned(1024))) TI sm[stage_bytes<BM, BN, BK, S, TI>() / sizeof(TI)];
    const int total = off[nprob];
    for (int t = blockIdx.x; t < total; t += gridDim.x) {
        int lo = 0, hi = nprob - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (off[mid] <= t) lo = mid;
            else hi = mid - 1;
        }
        const GemmProb& q = probs[lo];
        const int local = t - off[lo], ntn = q.N / BN;
        const int tm = local / ntn, tn = local - tm * ntn;
        __syncthreads();  // LDS of the previous tile is free
        pipe_tile<TI, TO, BM, BN, BK, WGM, WGN, S, AKM, BKM, false>((const TI*)q.A, (const TI*)q.B, (TO*)q.C, q.lda,
                                                                    q.ldb, q.ldc, q.K, q.alpha, q.accumulate, tm * BM,
                                                                    tn * BN, sm);
    }
}

// tile menu (code -> BM x BN).  "deep" tiles: bf16 and split bf16 stage twice the
// K slice per LDS round, halving the barriers per flop at twice the LDS footprint;
// FP64 and FP32 keep one LDS stage more.  For every type they take K in multiples
// of twice the plain step, the shapes for which saved tuning tables name them.
// The 96-wide tiles exist for the split-bfloat16 product only: at two workgroups
// per CU, 3072 x 4096 in 96 x 128 tiles (and 1024 x 3072 in 128 x 96 tiles,
// split-K 2) fills the 256 CUs in whole rounds, where 128 x 128 tiles leave the
// last round half empty.
struct TileCfg { int bm, bn; bool deep; const char* name; bool x3only; };
static const TileCfg kTiles[] = {
    {128, 128, false, "128x128", false}, {128, 64, false, "128x64", false}, {64, 128, false, "64x128", false},
    {64, 64, false, "64x64", false},     {32, 64, false, "32x64", false},   {64, 32, false, "64x32", false},
    {32, 32, false, "32x32", false},     {128, 128, true, "128x128d", false}, {128, 64, true, "128x64d", false},
    {64, 128, true, "64x128d", false},   {96, 128, false, "96x128", true},  {128, 96, false, "128x96", true},
    {192, 256, false, "192x256w8", true}, {256, 192, false, "256x192w8", true},
    {192, 128, false, "192x128w8db", true}, {128, 192, false, "128x192w8db", true},
};
static const int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);
int gemm_num_tiles() { return kNumTiles; }
const char* gemm_tile_name(int code) { return (code >= 1 && code <= kNumTiles) ? kTiles[code - 1].name : "auto"; }

template <typename TO, int BK, bool AKM, bool BKM>
static hipError_t launch_bf16(int code, const GemmParams& p, int batch, hipStream_t s)
{
    const TileCfg& t = kTiles[code];
    dim3 grid((p.M / t.bm) * (p.N / t.bn), batch);
    switch (code) {
    case 0: gemm_k<TO, 128, 128, BK, AKM, BKM><<<grid, 256, 0, s>>>(p); break;
    case 1: gemm_k<TO, 128, 64, BK, AKM, BKM><<<grid, 256, 0, s>>>(p); break;
    case 2: gemm_k<TO, 64, 128, BK, AKM, BKM><<<grid, 256, 0, s>>>(p); break;
    case 3: gemm_k<TO, 64, 64, BK, AKM, BKM><<<grid, 256, 0, s>>>(p); break;
    case 4: gemm_k<TO, 32, 64, BK, AKM, BKM><<<grid, 256, 0, s>>>(p); break;
    case 5: gemm_k<TO, 64, 32, BK, AKM, BKM><<<grid, 256, 0, s>>>(p); break;
    case 6: gemm_k<TO, 32, 32, BK, AKM, BKM><<<grid, 256, 0, s>>>(p); break;
    case 7: gemm_k<TO, 128, 128, 2 * BK, AKM, BKM><<<grid, 256, 0, s>>>(p); break;
    case 8: gemm_k<TO, 128, 64, 2 * BK, AKM, BKM><<<grid, 256, 0, s>>>(p); break;
    default: gemm_k<TO, 64, 128, 2 * BK, AKM, BKM><<<grid, 256, 0, s>>>(p); break;
    }
    return hipGetLastError();
}

// Whether the rows of one tile (K-major: its BM or BN rows, else the rows of a K
// step) span more than 32-bit byte offsets reach: with 128 rows of FP64 from a
// leading dimension of 4.2 million on.  Such a problem takes the 32x32 tile with
// 64-bit offsets (the same sums: every tile adds over k in order).
bool gemm_wide(int code, int tin, bool akm, bool bkm, long lda, long ldb)
{
    if ((tin != T_F64 && tin != T_F32) || code < 1 || code > kNumTiles) return false;
    const long es = tin == T_F64 ? 8 : 4, bk = 128 / es;
    auto far = [&](bool km, int rows, long ld) { return (km ? rows : bk) * es * ld > 1L << 32; };
    return far(akm, kTiles[code - 1].bm, lda) || far(bkm, kTiles[code - 1].bn, ldb);
}

// FP64 / FP32: K values of a step, waves, LDS stages and workgroups per CU of
// every tile.  The small FP64 tiles have little work between barriers and take
// four stages; the "deep" codes take one stage more than their plain form.
// FP32 tiles want workgroups on the CU more than stages.  Operands from memory
// (a dozen buffers in turn), 4512 x 6016 x 1504, in 32x64: 805 us with three
// workgroups of four stages, 760 with six of two (register-staged loop 783); 1504 x
// 4512 x 6016 in 32x32: 888 with four of four stages, 810 with eight of two
// (846).  3072 x 4096 x 1024 in 128x128: 199 us with two workgroups on 128-byte
// rows, 190 with three on 64-byte rows (195).
#define PIPE_F64(X)                                                                                       \
    X(0, 128, 128, 16, 2, 2, 2, 2) X(1, 128, 64, 16, 2, 2, 2, 3) X(2, 64, 128, 16, 2, 2, 2, 3)            \
    X(3, 64, 64, 16, 2, 2, 2, 4) X(4, 32, 64, 16, 1, 4, 4, 3) X(5, 64, 32, 16, 2, 2, 4, 3)                \
    X(6, 32, 32, 16, 2, 2, 4, 4) X(7, 128, 128, 16, 2, 2, 3, 1) X(8, 128, 64, 16, 2, 2, 3, 2)             \
    X(9, 64, 128, 16, 2, 2, 3, 2)
#define PIPE_F32(X)                                                                                       \
    X(0, 128, 128, 16, 2, 2, 2, 3) X(1, 128, 64, 32, 2, 2, 2, 3) X(2, 64, 128, 32, 2, 2, 2, 3)            \
    X(3, 64, 64, 32, 2, 2, 2, 4) X(4, 32, 64, 32, 1, 4, 2, 6) X(5, 64, 32, 32, 2, 2, 2, 6)                \
    X(6, 32, 32, 32, 2, 2, 2, 8) X(7, 128, 128, 32, 2, 2, 3, 1) X(8, 128, 64, 32, 2, 2, 3, 2)             \
    X(9, 64, 128, 32, 2, 2, 3, 2)

template <typename TI, typename TO, bool AKM, bool BKM>
static hipError_t launch_pipe(int code, const GemmParams& p, int batch, hipStream_t s)
{
    constexpr int BK = 128 / sizeof(TI);
    const dim3 grid32((p.M / 32) * (p.N / 32), batch);
    if (p.K % BK) {
        // FP32 with K an odd multiple of 16: the smallest tile on 64-byte rows
        if constexpr (std::is_same<TI, float>::value) {
            gemm_pipe_k<TI, TO, 32, 32, 16, 2, 2, 4, 4, AKM, BKM, true><<<grid32, 256, 0, s>>>(p);
            return hipGetLastError();
        }
        return hipErrorInvalidValue;
    }
    if (gemm_wide(code + 1, sizeof(TI) == 8 ? T_F64 : T_F32, AKM, BKM, p.lda, p.ldb)) {
        gemm_pipe_k<TI, TO, 32, 32, BK, 2, 2, 4, 4, AKM, BKM, true><<<grid32, 256, 0, s>>>(p);
        return hipGetLastError();
    }
    const TileCfg& t = kTiles[code];
    const dim3 grid((p.M / t.bm) * (p.N / t.bn), batch);
    if constexpr (std::is_same<TI, float>::value) {
        // FP32 128x64 and 64x128: three workgroups per CU on 128-byte rows while that
        // takes all of them at once (1024 x 3072 x 4096 in two K halves, 64x128: 197
        // us, four on 64-byte rows 201), else four on 64-byte rows (1984 x 3968 x 992,
        // 961 workgroups: 138 -> 132 us; 3072 x 4096 x 1024, 128x64: 199 -> 193)
        if ((long)grid.x * batch > 768 && (code == 1 || code == 2)) {
            if (code == 1) gemm_pipe_k<TI, TO, 128, 64, 16, 2, 2, 2, 4, AKM, BKM><<<grid, 256, 0, s>>>(p);
            else gemm_pipe_k<TI, TO, 64, 128, 16, 2, 2, 2, 4, AKM, BKM><<<grid, 256, 0, s>>>(p);
            return hipGetLastError();
        }
    }
#define PIPE_CASE(c, bm, bn, bk, wm, wn, st, occ)                                                  \
    case c: gemm_pipe_k<TI, TO, bm, bn, bk, wm, wn, st, occ, AKM, BKM><<<grid, 256, 0, s>>>(p); break;
    if constexpr (std::is_same<TI, double>::value) {
        switch (code) {
            PIPE_F64(PIPE_CASE)
        default: return hipErrorInvalidValue;
        }
    } else {
        switch (code) {
            PIPE_F32(PIPE_CASE)
        default: return hipErrorInvalidValue;
        }
    }
#undef PIPE_CASE
    return hipGetLastError();
}

template <typename TI, typename TO, bool AKM, bool BKM>
static hipError_t launch_grouped(int code, const GemmProb* probs, const int* off, int nprob, int grid, hipStream_t s)
{
#define PIPE_CASE(c, bm, bn, bk, wm, wn, st, occ)                                                                  \
    case c:                                                                                                         \
        gemm_grouped_k<TI, TO, bm, bn, bk, wm, wn, st, occ, AKM, BKM><<<grid, 256, 0, s>>>(probs, off, nprob); \
        break;
    if constexpr (std::is_same<TI, double>::value) {
        switch (code) {
            PIPE_F64(PIPE_CASE)
        default: return hipErrorInvalidValue;
        }
    } else {
        switch (code) {
            PIPE_F32(PIPE_CASE)
        default: return hipErrorInvalidValue;
        }
    }
#undef PIPE_CASE
    return hipGetLastError();
}

template <bool AKM, bool BKM>
static hipError_t grouped_layout(int tin, int tout, int code, const GemmProb* probs, const int* off, int nprob,
                                 int grid, hipStream_t s)
{
    if (tin == T_F64 && tout == T_F64) return launch_grouped<double, double, AKM, BKM>(code, probs, off, nprob, grid, s);
    if (tin == T_F32 && tout == T_F32) return launch_grouped<float, float, AKM, BKM>(code, probs, off, nprob, grid, s);
    if (tin == T_F32 && tout == T_F64) return launch_grouped<float, double, AKM, BKM>(code, probs, off, nprob, grid, s);
    return hipErrorInvalidValue;
}

template <typename TO>
static hipError_t launch_x3(int code, const GemmX3Params& p, int batch, hipStream_t s)
{
    const TileCfg& t = kTiles[code];
    dim3 grid((p.M / t.bm) * (p.N / t.bn), batch);
    switch (code) {
    case 0: gemm_x3_k<TO, 128, 128, 32><<<grid, 256, 0, s>>>(p); break;
    case 1: gemm_x3_k<TO, 128, 64, 32><<<grid, 256, 0, s>>>(p); break;
    case 2: gemm_x3_k<TO, 64, 128, 32><<<grid, 256, 0, s>>>(p); break;
    case 3: gemm_x3_k<TO, 64, 64, 32><<<grid, 256, 0, s>>>(p); break;
    case 4: gemm_x3_k<TO, 32, 64, 32><<<grid, 256, 0, s>>>(p); break;
    case 5: gemm_x3_k<TO, 64, 32, 32><<<grid, 256, 0, s>>>(p); break;
    case 6: gemm_x3_k<TO, 32, 32, 32><<<grid, 256, 0, s>>>(p); break;
    // deep tiles: a K step of 64 per LDS round (half the barriers per MFMA)
    case 7: gemm_x3_k<TO, 128, 128, 64><<<grid, 256, 0, s>>>(p); break;
    case 8: gemm_x3_k<TO, 128, 64, 64><<<grid, 256, 0, s>>>(p); break;
    case 9: gemm_x3_k<TO, 64, 128, 64><<<grid, 256, 0, s>>>(p); break;
    case 10: gemm_x3_k<TO, 96, 128, 32><<<grid, 256, 0, s>>>(p); break;
    case 11: gemm_x3_k<TO, 128, 96, 32><<<grid, 256, 0, s>>>(p); break;
    // eight waves, one workgroup per CU
    case 12: gemm_x3w_k<TO, 192, 256, 2, 4, false><<<grid, 512, 0, s>>>(p); break;
    case 13: gemm_x3w_k<TO, 256, 192, 4, 2, false><<<grid, 512, 0, s>>>(p); break;
    // eight waves, two LDS stages
    case 14: gemm_x3w_k<TO, 192, 128, 4, 2, true><<<grid, 512, 0, s>>>(p); break;
    default: gemm_x3w_k<TO, 128, 192, 2, 4, true><<<grid, 512, 0, s>>>(p); break;
    }
    return hipGetLastError();
}

// the split-bfloat16 product: K-major planes only, K a multiple of 32
static hipError_t gemm_x3(const GemmDesc& g, hipStream_t s)
{
    if (!g.a_kmajor || !g.b_kmajor || g.K % 32 || g.psA <= 0 || g.psB <= 0) return hipErrorInvalidValue;
    GemmX3Params p;
    p.A = (const bf16*)g.A; p.B = (const bf16*)g.B; p.C = g.C;
    p.M = g.M; p.N = g.N; p.K = g.K;
    p.lda = g.lda; p.ldb = g.ldb; p.ldc = g.ldc;
    p.sA = g.sA; p.sB = g.sB; p.sC = g.sC;
    p.psA = g.psA; p.psB = g.psB;
    p.alpha = g.alpha; p.accumulate = g.accumulate;
    int code = g.tile - 1;
    if (g.tile <= 0) {
        int ks;
        gemm_default(g.tin, g.M, g.N, g.K, g.batch, false, &code, &ks);
        code--;
    }
    if (code < 0 || code >= kNumTiles || g.M % kTiles[code].bm || g.N % kTiles[code].bn) return hipErrorInvalidValue;
    if (kTiles[code].deep && g.K % 64) return hipErrorInvalidValue;
    if (g.tout == T_F32) return launch_x3<float>(code, p, g.batch, s);
    if (g.tout == T_F64) return launch_x3<double>(code, p, g.batch, s);
    return hipErrorInvalidValue;
}

// K values of a step
static int gemm_k_step(int tin, int K)
{
    if (tin == T_F64) return 16;
    if (tin == T_F32) return K % 32 == 0 ? 32 : 16;
    return K % 64 == 0 ? 64 : 32;
}

bool gemm_tile_ok(int code, int tin, int M, int N, int K)
{
    if (code < 1 || code > kNumTiles) return false;
    const TileCfg& t = kTiles[code - 1];
    if (M % t.bm || N % t.bn || (t.x3only && tin != T_BF16X3)) return false;
    if (tin == T_BF16X3) return K % (t.deep ? 64 : 32) == 0;
    const int bk = gemm_k_step(tin, K);
    return K % (t.deep ? 2 * bk : bk) == 0;
}
int gemm_tile_bm(int code) { return (code >= 1 && code <= kNumTiles) ? kTiles[code - 1].bm : 0; }
int gemm_tile_bn(int code) { return (code >= 1 && code <= kNumTiles) ? kTiles[code - 1].bn : 0; }
static int choose_tile(int M, int N, int batch);
int gemm_grouped_tile(int M, int N) { return choose_tile(M, N, 1) + 1; }

hipError_t gemm_grouped(int tin, int tout, bool akm, bool bkm, int tile, const GemmProb* probs, const int* off,
                         int nprob, int total_tiles, hipStream_t s)
{
    if (nprob <= 0 || total_tiles <= 0) return hipSuccess;
    if (tile < 1 || tile > kNumTiles || kTiles[tile - 1].x3only) return hipErrorInvalidValue;
    const int grid = total_tiles < 2048 ? total_tiles : 2048;
    if (akm && bkm) return grouped_layout<true, true>(tin, tout, tile - 1, probs, off, nprob, grid, s);
    if (akm && !bkm) return grouped_layout<true, false>(tin, tout, tile - 1, probs, off, nprob, grid, s);
    if (!akm && !bkm) return grouped_layout<false, false>(tin, tout, tile - 1, probs, off, nprob, grid, s);
    return grouped_layout<false, true>(tin, tout, tile - 1, probs, off, nprob, grid, s);
}

// bf16 and grouped launches: pick the largest tile that divides the problem and still
// gives >= ~1.5 workgroups per CU (256 CUs); fall back to the tile with the
// most blocks.
static int choose_tile(int M, int N, int batch)
{
    int best = -1;
    long best_blocks = -1;
    for (int c = 0; c < kNumTiles; c++) {
        if (kTiles[c].deep || kTiles[c].x3only || M % kTiles[c].bm || N % kTiles[c].bn) continue;
        long blocks = (long)(M / kTiles[c].bm) * (N / kTiles[c].bn) * batch;
        if (blocks >= 384) return c;
        if (blocks > best_blocks) { best_blocks = blocks; best = c; }
    }
    return best;
}

// FP64, FP32 and split-bf16 tile and k-split from a model of the time, in us, fitted to the
// tiles timed one by one (M x N x K from 32 x 96 x 128 to 3072 x 4096 x 1024, all
// layouts; within 8 % of the measured time from 5 us up):
//   3.7 + steps * max(n * busy, alone)   + for a split  3 + bytes / 10 TB/s
// steps: K steps (16 FP64, 32 FP32 values) of one workgroup; n: workgroups on the
// fullest CU; busy: matrix-pipe time of a workgroup's step; alone: the step of a
// workgroup that has a CU to itself (copy, barrier and instruction latency).
struct StepCost { int code; float busy, alone; };
static const StepCost kCostF64[] = {  // 128x64, 64x128, 64x64, 32x64, 64x32, 32x32
    {1, 0.933f, 1.05f}, {2, 0.933f, 1.05f}, {3, 0.485f, 0.53f}, {4, 0.259f, 0.30f}, {5, 0.259f, 0.30f},
    {6, 0.138f, 0.235f}};
static const StepCost kCostF32[] = {  // and 128x128
    {0, 1.95f, 2.40f}, {1, 1.016f, 1.15f}, {2, 1.016f, 1.15f}, {3, 0.608f, 0.70f}, {4, 0.353f, 0.45f}, {5, 0.353f, 0.45f},
    {6, 0.205f, 0.355f}};
// split bf16 (steps of 32): 128x128 .. 32x32, 96x128, 128x96, 192x256, 256x192,
// 192x128, 128x192.  1024 x 3072 x 4096: 208 us in the 128x64 tiles of the
// block-count rule, 134 us in 128x192 with a 2-way split (1.15 PFLOP/s of bf16);
// 512 x 1536 x 2048: 36 -> 32 us; 320 x 448 x 1280: 19 -> 12 us.  Small tiles of
// long products are bound by what they read from the caches, at most about 13 TB/s
// (672 x 2688 x 2688: 162 us in 32x64, 97 us in 96x128, both in two K halves).
static const StepCost kCostX3[] = {
    {0, 1.42f, 1.60f}, {1, 0.715f, 1.00f}, {2, 0.708f, 1.00f}, {3, 0.418f, 0.60f},  {4, 0.285f, 0.41f},
    {5, 0.274f, 0.36f}, {6, 0.167f, 0.266f}, {10, 1.02f, 1.48f}, {11, 1.00f, 1.48f}, {12, 4.0f, 4.0f},
    {13, 4.0f, 4.0f}, {14, 2.0f, 2.0f}, {15, 1.95f, 1.95f}};
void gemm_default(int tin, int M, int N, int K, int batch, bool split, int* tile, int* ksplit)
{
    *ksplit = 1;
    const StepCost* cost = tin == T_F64 ? kCostF64 : (tin == T_F32 ? kCostF32 : kCostX3);
    const int ncost = tin == T_BF16X3 ? (int)(sizeof(kCostX3) / sizeof(kCostX3[0])) : (tin == T_F32 ? 7 : 6);
    if (tin == T_BF16) {
        *tile = choose_tile(M, N, batch) + 1;
        return;
    }
    const int bk = tin == T_F64 ? 16 : 32, es = tin == T_F64 ? 8 : 4;
    float best = 1e30f;
    *tile = 7;
    for (int q = 0; q < ncost; q++) {
        const StepCost& c = cost[q];
        const TileCfg& t = kTiles[c.code];
        if (M % t.bm || N % t.bn) continue;
        for (int ks = 1; ks <= 4; ks *= 2) {
            if (ks > 1 && (!split || batch != 1 || K % (64 * ks))) break;
            const long blocks = (long)(M / t.bm) * (N / t.bn) * batch * ks;
            const float busy = (float)((blocks + 255) / 256) * c.busy;
            float us = (float)(K / ks) / bk * (busy > c.alone ? busy : c.alone);
            if (tin == T_BF16X3) us = std::max(us, (float)blocks * (K / ks) * (t.bm + t.bn) * 6 / 13e6f);
            us += 3.7f;
            if (ks > 1) us += 3.0f + (float)M * N * (2 * ks * es + 8) * 1e-7f;
            if (us < best) {
                best = us;
                *tile = c.code + 1;
                *ksplit = ks;
            }
        }
    }
}

template <typename TI, typename TO, bool AKM, bool BKM>
static hipError_t gemm_typed(const GemmDesc& g, hipStream_t s)
{
    GemmParams p;
    p.A = g.A; p.B = g.B; p.C = g.C;
    p.M = g.M; p.N = g.N; p.K = g.K;
    p.lda = g.lda; p.ldb = g.ldb; p.ldc = g.ldc;
    p.sA = g.sA; p.sB = g.sB; p.sC = g.sC;
    p.alpha = g.alpha; p.accumulate = g.accumulate;
    int code = g.tile - 1;
    if (g.tile <= 0) {
        int ks;
        gemm_default(g.tin, g.M, g.N, g.K, g.batch, false, &code, &ks);
        code--;
    }
    if (code < 0 || code >= kNumTiles || kTiles[code].x3only || g.M % kTiles[code].bm || g.N % kTiles[code].bn)
        return hipErrorInvalidValue;
    if (kTiles[code].deep && g.K % (2 * gemm_k_step(g.tin, g.K))) return hipErrorInvalidValue;
    if constexpr (std::is_same<TI, bf16>::value) {
        if (g.K % 64 == 0) return launch_bf16<TO, 64, AKM, BKM>(code, p, g.batch, s);
        if (g.K % 32) return hipErrorInvalidValue;
        return launch_bf16<TO, 32, AKM, BKM>(code, p, g.batch, s);
    } else {
        if (g.K % 16) return hipErrorInvalidValue;
        return launch_pipe<TI, TO, AKM, BKM>(code, p, g.batch, s);
    }
}

template <bool AKM, bool BKM>
static hipError_t gemm_layout(const GemmDesc& g, hipStream_t s)
{
    if (g.tin == T_F64) {
        if (g.tout == T_F64) return gemm_typed<double, double, AKM, BKM>(g, s);
        return hipErrorInvalidValue;
    }
    if (g.tin == T_F32) {
        if (g.tout == T_F32) return gemm_typed<float, float, AKM, BKM>(g, s);
        if (g.tout == T_F64) return gemm_typed<float, double, AKM, BKM>(g, s);
        return hipErrorInvalidValue;
    }
    if (g.tin == T_BF16) {
        if (g.tout == T_F32) return gemm_typed<bf16, float, AKM, BKM>(g, s);
        if (g.tout == T_F64) return gemm_typed<bf16, double, AKM, BKM>(g, s);
        if (g.tout == T_BF16) return gemm_typed<bf16, bf16, AKM, BKM>(g, s);
    }
    return hipErrorInvalidValue;
}

hipError_t gemm(const GemmDesc& g, hipStream_t s)
{
    if (g.M <= 0 || g.N <= 0 || g.K <= 0 || g.batch <= 0) return hipErrorInvalidValue;
    if (g.M % 32 || g.N % 32 || g.K % 16) return hipErrorInvalidValue;
    if (g.tin == T_BF16X3) return gemm_x3(g, s);
    if (g.a_kmajor && g.b_kmajor) return gemm_layout<true, true>(g, s);
    if (g.a_kmajor && !g.b_kmajor) return gemm_layout<true, false>(g, s);
    if (!g.a_kmajor && !g.b_kmajor) return gemm_layout<false, false>(g, s);
    return gemm_layout<false, true>(g, s);
}

// split-K reduction: C[i*ldc + j] (+)= sum_z W[z*M*N + i*N + j]
template <typename TA, typename TO>
__global__ void __launch_bounds__(256) splitk_reduce_k(const TA* __restrict__ W, int ks, int M, int N,
                                                       TO* __restrict__ C, long ldc, int accumulate)
{
    const long MN = (long)M * N;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < MN; e += (long)gridDim.x * 256) {
        const long i = e / N, j = e - i * N;
        if constexpr (std::is_same<TA, double>::value) {
            double v = 0.0;
            for (int z = 0; z < ks; z++) v += W[z * MN + e];
            TO* cp = C + i * ldc + j;
            if (accumulate) v += to_d(*cp);
            *cp = cvt_from_d<TO>(v);
        } else {
            float v = 0.0f;
            for (int z = 0; z < ks; z++) v += W[z * MN + e];
            TO* cp = C + i * ldc + j;
            if constexpr (std::is_same<TO, double>::value) {
                double dv = (double)v;
                if (accumulate) dv += *cp;
                *cp = dv;
            } else {
                if (accumulate) v += to_f(*cp);
                *cp = cvt_from_f<TO>(v);
            }
        }
    }
}

hipError_t splitk_reduce(int tacc, const void* W, int ks, int M, int N, int tout, void* C, long ldc, int accumulate,
                         hipStream_t s)
{
    long blocks = ((long)M * N + 255) / 256;
    if (blocks > 4096) blocks = 4096;
#define SK_CASE(TAc, TOc, TAt, TOt)                                                                  \
    if (tacc == TAc && tout == TOc) {                                                                \
        splitk_reduce_k<TAt, TOt><<<blocks, 256, 0, s>>>((const TAt*)W, ks, M, N, (TOt*)C, ldc, accumulate); \
        return hipGetLastError();                                                                    \
    }
    SK_CASE(T_F64, T_F64, double, double)
    SK_CASE(T_F32, T_F32, float, float)
    SK_CASE(T_F32, T_F64, float, double)
    SK_CASE(T_F32, T_BF16, float, bf16)
#undef SK_CASE
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------
// Stage 1 of the split-bfloat16 Heff apply with the MPO stage fused into its
// epilogue.  A workgroup owns 32 a' x 32 b: its stage-1 tile is rows
// (a', n) for the 32 a' (32 P rows of x) and columns (w', b) for every kept
// right channel w' and the 32 b (the R rows w' D2p + b0 + 0..31), so every
// (n, w') term of the MPO stage for its outputs is in the tile.  The K loop
// is the four-wave loop of gemm_tile_x3 (swizzled LDS, register prefetch);
// then the FP32 tile and the FP64 x slice of the right identity channel go
// to LDS and the mixing sums are formed there: outputs of the kept left
// channels with lanes along a' (32 consecutive a' of one (m, b, w) are one
// 64-byte run of each plane), the left identity channel's outputs with
// lanes along b (coalesced FP64 rows of y).
struct X3MixParams {
    const bf16* X;
    long psX;
    const bf16* R;
    long psR;
    const double* x;
    bf16* T2;
    long ps2, ldo;
    double* y;
    int D1p, D2p;
    const int* optr;
    const int* ocode;
    const int* ecode;
    const float* val;
    int nout, nnz;
};

template <int P, int NR>
__global__ void __launch_bounds__(256) x3_stage1_mix_k(X3MixParams q)
{
    typedef MT<bf16> T;
    typedef T::frag_t frag_t;
    typedef T::acc_t acc_t;
    constexpr int BM = 32 * P, BN = 32 * NR, BK = 32;
    constexpr int WM = BM / 2, WN = BN / 2, FM = WM / 16, FN = WN / 16;
    constexpr int SA = BM * BK, SB = BN * BK;
    constexpr int RA = (BM * 4 + 255) / 256, RB = (BN * 4 + 255) / 256;
    constexpr int TS = BN + 1;  // row stride of the FP32 tile (floats)
    constexpr int XS = 33;      // row stride of the x slice
    constexpr int OPB = 3 * (SA + SB) * 2;
    constexpr int EPB = (BM * TS + BM * XS) * 4;
    constexpr int LB = OPB > EPB ? OPB : EPB;
    __shared__ __attribute__((aligned(16))) unsigned char smem[LB];
    __shared__ int s_optr[33], s_ocode[32], s_ecode[256];
    __shared__ float s_val[256];
    bf16* As = (bf16*)smem;
    bf16* Bs = As + 3 * SA;
    float* Ts = (float*)smem;
    float* Xs = Ts + BM * TS;

    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int ntm = q.D1p / 32, ntn = q.D2p / 32, nblk = ntm * ntn;
    int bid = blockIdx.x;
    if ((nblk & 7) == 0) bid = (bid & 7) * (nblk >> 3) + (bid >> 3);
    constexpr int GM = 8;
    const int gsz = GM * ntn, g = bid / gsz, first = g * GM;
    const int rows = ntm - first < GM ? ntm - first : GM;
    const int local = bid - g * gsz;
    const int a0 = (first + local % rows) * 32, b0 = (local / rows) * 32;
    const int m0 = a0 * P;
    const long D2p = q.D2p;

    for (int i = tid; i <= q.nout; i += 256) s_optr[i] = q.optr[i];
    for (int i = tid; i < q.nout; i += 256) s_ocode[i] = q.ocode[i];
    for (int i = tid; i < q.nnz; i += 256) {
        s_ecode[i] = q.ecode[i];
        s_val[i] = q.val[i];
    }
    // the x slice of the right identity channel (rows (a', n), 32 b), read
    // now so that its latency hides behind the K loop
    constexpr int XR = BM * 32 / 256;
    float xr[XR];
#pragma unroll
    for (int k = 0; k < XR; k++) {
        const int v = tid + k * 256;
        xr[k] = (float)q.x[(long)(m0 + (v >> 5)) * D2p + b0 + (v & 31)];
    }

    const int wm0 = (wid >> 1) * WM, wn0 = (wid & 1) * WN;
    u32x4 ra[3][RA], rb[3][RB];
    acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = 0;
    // operand slices: A rows m0 + t, B rows (t / 32) D2p + b0 + t % 32
    auto gload = [&](int k0) {
#pragma unroll
        for (int pl = 0; pl < 3; pl++) {
#pragma unroll
            for (int r = 0; r < RA; r++) {
                const int v = tid + r * 256;
                if ((BM * 4) % 256 == 0 || v < BM * 4)
                    ra[pl][r] = *(const u32x4*)(q.X + pl * q.psX + (long)(m0 + v / 4) * D2p + k0 + (v % 4) * 8);
            }
#pragma unroll
            for (int r = 0; r < RB; r++) {
                const int v = tid + r * 256;
                if ((BN * 4) % 256 == 0 || v < BN * 4) {
                    const int t = v / 4;
                    const long row = (long)(t >> 5) * D2p + b0 + (t & 31);
                    rb[pl][r] = *(const u32x4*)(q.R + pl * q.psR + row * D2p + k0 + (v % 4) * 8);
                }
            }
        }
    };
    auto sstore = [&]() {
#pragma unroll
        for (int pl = 0; pl < 3; pl++) {
            x3_sstore<BM, BK>(ra[pl], As + pl * SA, tid);
            x3_sstore<BN, BK>(rb[pl], Bs + pl * SB, tid);
        }
    };
    const int nk = (int)(D2p / BK);
    gload(0);
    sstore();
    __syncthreads();
    for (int t = 0; t < nk; t++) {
        if (t + 1 < nk) gload((t + 1) * BK);
        __builtin_amdgcn_s_setprio(1);
        frag_t a[3][FM], b[3][FN];
#pragma unroll
        for (int pl = 0; pl < 3; pl++) {
#pragma unroll
            for (int i = 0; i < FM; i++)
                a[pl][i] = *(const frag_t*)(As + pl * SA + x3_swz(wm0 + i * 16 + (lane & 15), lane >> 4));
#pragma unroll
            for (int j = 0; j < FN; j++)
                b[pl][j] = *(const frag_t*)(Bs + pl * SB + x3_swz(wn0 + j * 16 + (lane & 15), lane >> 4));
        }
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) {
                acc[i][j] = mma(a[2][i], b[0][j], acc[i][j]);
                acc[i][j] = mma(a[0][i], b[2][j], acc[i][j]);
                acc[i][j] = mma(a[1][i], b[1][j], acc[i][j]);
                acc[i][j] = mma(a[1][i], b[0][j], acc[i][j]);
                acc[i][j] = mma(a[0][i], b[1][j], acc[i][j]);
                acc[i][j] = mma(a[0][i], b[0][j], acc[i][j]);
            }
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();
        if (t + 1 < nk) {
            sstore();
            __syncthreads();
        }
    }
    // the operand tiles are consumed (barrier above): the LDS takes the FP32
    // stage-1 tile and the x slice (rows (a', n), 32 b)
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                Ts[(wm0 + i * 16 + T::crow(lane, r)) * TS + wn0 + j * 16 + (lane & 15)] = acc[i][j][r];
#pragma unroll
    for (int k = 0; k < XR; k++) {
        const int v = tid + k * 256;
        Xs[(v >> 5) * XS + (v & 31)] = xr[k];
    }
    __syncthreads();
    // sums of the table entries of output o for NV values at rows a_i = al0 +
    // i * astep (a' within the tile) and column bl: an entry's code and value
    // are read once, then its NV source reads are independent
    auto mixsums = [&](int o, int al0, int astep, int bl, float* sum, auto nv) {
        constexpr int NV = decltype(nv)::value;
#pragma unroll
        for (int i = 0; i < NV; i++) sum[i] = 0.f;
        const int e1 = s_optr[o + 1];
        for (int e = s_optr[o]; e < e1; e++) {
            const int ec = s_ecode[e], n = ec & 255;
            const float v = s_val[e];
            const bool fromx = ec >> 16;
            const float* src = fromx ? Xs + n * XS + bl : Ts + n * TS + ((ec >> 8) & 255) * 32 + bl;
            const int rs = (fromx ? XS : TS) * P;  // row step per a'
#pragma unroll
            for (int i = 0; i < NV; i++) sum[i] += v * src[(al0 + i * astep) * rs];
        }
    };
    // kept left channels: T2t[(m, b)][(w, a')] as three planes; a lane forms
    // 8 consecutive a' of one (m, b, w) and stores them as one 16-byte write
    // per plane (4 lanes cover the tile's 32 a'), the two halves of the
    // workgroup take alternate outputs
    {
        const int a8 = (tid & 3) * 8, bl = (tid >> 2) & 31, oh = tid >> 7;
        for (int o = oh; o < q.nout; o += 2) {
            const int oc = s_ocode[o];
            if (oc >> 16) continue;
            float v8[8];
            mixsums(o, a8, 1, bl, v8, std::integral_constant<int, 8>());
            uint32_t h[3][4];
#pragma unroll
            for (int i = 0; i < 8; i += 2) {
                bf16 p0, p1, p2, r0, r1, r2;
                split3_val(v8[i], p0, p1, p2);
                split3_val(v8[i + 1], r0, r1, r2);
                h[0][i / 2] = (uint32_t)p0 | ((uint32_t)r0 << 16);
                h[1][i / 2] = (uint32_t)p1 | ((uint32_t)r1 << 16);
                h[2][i / 2] = (uint32_t)p2 | ((uint32_t)r2 << 16);
            }
            bf16* dst = q.T2 + (long)(oc & 255) * D2p * q.ldo + (long)((oc >> 8) & 255) * q.D1p +
                        (long)(b0 + bl) * q.ldo + a0 + a8;
#pragma unroll
            for (int pl = 0; pl < 3; pl++) {
                u32x4 w;
                w.x = h[pl][0];
                w.y = h[pl][1];
                w.z = h[pl][2];
                w.w = h[pl][3];
                *(u32x4*)(dst + pl * q.ps2) = w;
            }
        }
    }
    // the left identity channel: y[a'][m][b], lanes along b
    {
        const int bl = tid & 31, ag = tid >> 5;
        for (int o = 0; o < q.nout; o++) {
            const int oc = s_ocode[o];
            if (!(oc >> 16)) continue;
            float v4[4];
            mixsums(o, ag, 8, bl, v4, std::integral_constant<int, 4>());
#pragma unroll
            for (int k = 0; k < 4; k++)
                q.y[((long)(a0 + ag + 8 * k) * P + (oc & 255)) * D2p + b0 + bl] = (double)v4[k];
        }
    }
}

bool x3_stage1_mix_ok(int p, int nR, const MixTable& t, int D1p, int D2p)
{
    return t.ocode && t.ecode && t.nout <= 32 && t.nnz <= 256 && D1p > 0 && D2p > 0 && D1p % 32 == 0 &&
           D2p % 32 == 0 && (p == 2 || p == 3) && nR >= 2 && nR <= 5;
}

hipError_t x3_stage1_mix(int p, int nR, const bf16* X, long psX, const bf16* R, long psR, const double* x,
                         bf16* T2, long ps2, long ldo, double* y, int D1p, int D2p, const MixTable& t,
                         hipStream_t s)
{
    if (!x3_stage1_mix_ok(p, nR, t, D1p, D2p)) return hipErrorInvalidValue;
    X3MixParams q;
    q.X = X; q.psX = psX; q.R = R; q.psR = psR; q.x = x; q.T2 = T2; q.ps2 = ps2; q.ldo = ldo; q.y = y;
    q.D1p = D1p; q.D2p = D2p;
    q.optr = t.optr; q.ocode = t.ocode; q.ecode = t.ecode; q.val = t.evalf; q.nout = t.nout; q.nnz = t.nnz;
    const dim3 grid((D1p / 32) * (D2p / 32));
#define X3M_CASE(PP, NN)                                                  \
    if (p == PP && nR == NN) {                                            \
        x3_stage1_mix_k<PP, NN><<<grid, 256, 0, s>>>(q);                  \
        return hipGetLastError();                                         \
    }
    X3M_CASE(2, 2) X3M_CASE(2, 3) X3M_CASE(2, 4) X3M_CASE(2, 5)
    X3M_CASE(3, 2) X3M_CASE(3, 3) X3M_CASE(3, 4) X3M_CASE(3, 5)
#undef X3M_CASE
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------
// The whole FP64 Heff apply of a small site in one launch (left bond padded to
// 32, right bond to 32 or 64).  A workgroup owns 16 of the b columns of y: stage 1
// for those b (T1 in LDS, one 16-column block per kept right channel, and x itself
// as one more block for the identity channel), then stage 3, whose right operand
// (the MPO stage's output) is formed in registers from T1 as the matrix
// instruction needs it.  16 waves: stage 1 wave = (row tile, channel group), stage
// 3 wave = (m, slice of the K sum over (w, a')), the slices summed through LDS.
// Bound by the latency of its loads and of the two stages; the three-kernel path
// pays that, a launch and a drain three times: D = 32, d = 2, four channels 9.4 us
// here; a host call at D = 8 (padded to 32) took 28 us with the three kernels and
// the two layout passes, 18.6 us with this one.  A left bond of 64 makes one
// workgroup's share of the work too large (measured at D = 64, d = 2: 26 us against
// 14 us of kernels and two launch gaps), so it keeps the three kernels.
constexpr int HS_LDS = 116 * 1024;
constexpr int HS_MAXO = 64, HS_MAXE = 256;

static inline int hs_pad(int p) { return p == 2 ? 2 : (p == 3 ? 4 : 1); }  // spreads the four lane groups over the banks
bool heff_small_ok(const HeffSmall& a)
{
    return a.p >= 2 && a.p <= 4 && a.D1p == 32 && (a.D2p == 32 || a.D2p == 64) && a.nR >= 1 && a.nL >= 1 &&
           a.t.ocode && a.t.ecode && a.t.nout <= HS_MAXO && a.t.nnz <= HS_MAXE &&
           32L * a.p * ((a.nR + 1) * 16 + hs_pad(a.p)) * 8 <= HS_LDS;
}

template <int P, int D2P, bool REF>
__global__ void __launch_bounds__(1024) heff_small_k(HeffSmall q)
{
    typedef MT<double> T;
    constexpr int NT = 1024, NW = 16, D1P = 32, RT = D1P * P / 16, KB = D2P / 16, AT = D1P / 16;
    constexpr int CG = NW / RT;  // channel groups of stage 1
    constexpr int PAD = P == 2 ? 2 : (P == 3 ? 4 : 1);
    constexpr int SL = NW / P;   // K slices of stage 3
    static_assert(SL * P * D1P * 16 * 8 <= HS_LDS, "partial sums");
    __shared__ __attribute__((aligned(16))) double sm[HS_LDS / 8];
    __shared__ int s_optr[HS_MAXO + 1], s_ecode[HS_MAXE];
    __shared__ double s_val[HS_MAXE];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int r = lane & 15, kq = lane >> 4;
    const int b0 = blockIdx.x * 16;
    const int ld1 = (q.nR + 1) * 16 + PAD;
    // element (row (a', n), b') of x
    auto xat = [&](int row, int b) -> double {
        if constexpr (REF) return row < P * q.D1 && b < q.D2 ? q.x[row + (long)P * q.D1 * b] : 0.0;
        else return q.x[(long)row * D2P + b];
    };
    // K index of a block's value e of lane group kq: two 16-byte units per lane,
    // the four groups side by side
    auto kof = [&](int e) { return ((e >> 1) * 4 + kq) * 2 + (e & 1); };
    // every first load is in flight before anything waits: the stage-1 operands,
    // stage 3's first block of L, x's own columns, the table
    double a[KB][4], bv[2][KB][4], la[AT][4];
    const int rt = wid % RT, cg = wid / RT;  // stage 1: row tile, channels cg, cg + CG, ...
    const int nkb = q.nL * AT;
    const int m = wid % P, sl = wid / P;  // stage 3: column block m, K blocks sl, sl + SL, ...
    auto loadR = [&](int ch, int h) {
        const double* Rw = q.R + ((long)ch * D2P + b0 + r) * D2P;
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int e = 0; e < 4; e++) bv[h][kb][e] = Rw[kb * 16 + kof(e)];
    };
    auto loadL = [&](int kb) {
        const double* Lw = q.L + (long)(kb / AT) * D1P + (kb % AT) * 16;
#pragma unroll
        for (int i = 0; i < AT; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) la[i][e] = Lw[(long)(i * 16 + r) * q.Dw1 * D1P + kof(e)];
    };
    const bool s1 = cg < CG && cg < q.nR;
    if (s1) {
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int e = 0; e < 4; e++) a[kb][e] = xat(rt * 16 + r, kb * 16 + kof(e));
        loadR(cg, 0);
        if (cg + CG < q.nR) loadR(cg + CG, 1);
    }
    if (sl < SL && sl < nkb) loadL(sl);
    constexpr int XN = (D1P * P * 16 + NT - 1) / NT;
    double xs[XN];
#pragma unroll
    for (int u = 0; u < XN; u++) {
        const int i = tid + u * NT;
        const int row = REF ? i % (D1P * P) : i >> 4, b = REF ? i / (D1P * P) : i & 15;
        if (i < D1P * P * 16) xs[u] = xat(row, b0 + b);
    }
    static_assert(HS_MAXO < NT && HS_MAXE <= NT, "one table entry per thread");
    const int to = tid <= q.t.nout ? q.t.optr[tid] : 0, te = tid < q.t.nnz ? q.t.ecode[tid] : 0;
    const double tv = tid < q.t.nnz ? q.t.eval[tid] : 0.0;
    if (tid <= q.t.nout) s_optr[tid] = to;
    if (tid < q.t.nnz) {
        s_ecode[tid] = te;
        s_val[tid] = tv;
    }
    // x's own 16 columns: the block after the kept channels
#pragma unroll
    for (int u = 0; u < XN; u++) {
        const int i = tid + u * NT;
        const int row = REF ? i % (D1P * P) : i >> 4, b = REF ? i / (D1P * P) : i & 15;
        if (i < D1P * P * 16) sm[row * ld1 + q.nR * 16 + b] = xs[u];
    }
    // stage 1: T1[(a', n)][(w', b)]
    auto step = [&](int ch, int h) {
        v4d acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc = mma(a[kb][e], bv[h][kb][e], acc);
        if (ch + 2 * CG < q.nR) loadR(ch + 2 * CG, h);
        double* d = sm + rt * 16 * ld1 + ch * 16 + r;
#pragma unroll
        for (int i = 0; i < 4; i++) d[T::crow(lane, i) * ld1] = acc[i];
    };
    if (s1) {
        for (int ch = cg; ch < q.nR; ch += 2 * CG) {
            step(ch, 0);
            if (ch + CG < q.nR) step(ch + CG, 1);
        }
    }
    __syncthreads();
    v4d acc[AT];
#pragma unroll
    for (int i = 0; i < AT; i++) acc[i] = v4d{0.0, 0.0, 0.0, 0.0};
    if (sl < SL) {
        if (sl == 0 && q.wl >= 0) {  // the left identity channel: a' = a
            const int o = q.wl * P + m;
            for (int e = s_optr[o]; e < s_optr[o + 1]; e++) {
                const int ec = s_ecode[e];
                const int ch = ec >> 16 ? q.nR : (ec >> 8) & 255;
                const double* src = sm + (ec & 255) * ld1 + ch * 16 + r;
                const double v = s_val[e];
#pragma unroll
                for (int i = 0; i < AT; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) acc[i][j] += v * src[(i * 16 + T::crow(lane, j)) * P * ld1];
            }
        }
        for (int kb = sl; kb < nkb; kb += SL) {
            const int w = kb / AT;
            const int o = (w + (q.wl == 0 ? 1 : 0)) * P + m;
            double b3[4] = {0.0, 0.0, 0.0, 0.0};
            const int a0 = (kb % AT) * 16;
            for (int e = s_optr[o]; e < s_optr[o + 1]; e++) {
                const int ec = s_ecode[e];
                const int ch = ec >> 16 ? q.nR : (ec >> 8) & 255;
                const double* src = sm + (ec & 255) * ld1 + ch * 16 + r;
                const double v = s_val[e];
#pragma unroll
                for (int u = 0; u < 4; u++) b3[u] += v * src[(a0 + kof(u)) * P * ld1];
            }
            double ca[AT][4];
#pragma unroll
            for (int i = 0; i < AT; i++)
#pragma unroll
                for (int u = 0; u < 4; u++) ca[i][u] = la[i][u];
            if (kb + SL < nkb) loadL(kb + SL);
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int i = 0; i < AT; i++) acc[i] = mma(ca[i][u], b3[u], acc[i]);
        }
    }
    __syncthreads();  // T1 is no longer read
    if (sl < SL) {
        double* d = sm + (sl * P + m) * D1P * 16 + r;
#pragma unroll
        for (int i = 0; i < AT; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) d[(i * 16 + T::crow(lane, j)) * 16] = acc[i][j];
    }
    __syncthreads();
    for (int i = tid; i < D1P * P * 16; i += NT) {
        const int row = REF ? i % (D1P * P) : i >> 4, b = REF ? i / (D1P * P) : i & 15;
        const int mm = row % P, aa = row / P;
        double s = 0.0;
#pragma unroll
        for (int z = 0; z < SL; z++) s += sm[((z * P + mm) * D1P + aa) * 16 + b];
        if constexpr (REF) {
            if (aa < q.D1 && b0 + b < q.D2) q.y[row + (long)P * q.D1 * (b0 + b)] = q.scale * s;
        } else {
            q.y[(long)row * D2P + b0 + b] = q.scale * s;
        }
    }
}

hipError_t heff_small(const HeffSmall& a, hipStream_t s)
{
    if (!heff_small_ok(a)) return hipErrorInvalidValue;
    const dim3 grid(a.D2p / 16);
#define HS_CASE(PP, B)                                                           \
    if (a.p == PP && a.D2p == B) {                                               \
        if (a.D1 > 0) heff_small_k<PP, B, true><<<grid, 1024, 0, s>>>(a);        \
        else heff_small_k<PP, B, false><<<grid, 1024, 0, s>>>(a);                \
        return hipGetLastError();                                                \
    }
    HS_CASE(2, 32) HS_CASE(2, 64) HS_CASE(3, 32) HS_CASE(3, 64) HS_CASE(4, 32) HS_CASE(4, 64)
#undef HS_CASE
    return hipErrorInvalidValue;
}

}  // namespace tn
