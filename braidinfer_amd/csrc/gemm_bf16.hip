// bf16 matrix products on the gfx950 matrix cores: C[M,N] (+)= A[M,K] * W[N,K]^T with
// bf16 inputs, float accumulation, and a bf16 or float output.  W is a weight matrix as
// checkpoints store it ([out, in], row-major), so both operands are read along k.
//
// Kernels:
//  * gemm_stream_tile: up to 16 rows (decode), and up to 128 against few weight rows: a workgroup a tile of 16 to 32 weight rows
//    over all of K, weights and activations brought into per-wave LDS rings by direct global-to-LDS loads.
//  * gemm_stream: up to 16 rows where tiles are many and K short or long, and with an RMS norm before or behind: the same streaming
//    by one resident workgroup per compute unit.
//  * gemm_tile: LDS-staged tiles for many rows (prompts): 4 waves, each a TM x TN grid of
//    v_mfma_f32_32x32x16_bf16 blocks; global loads of the next k-tile are issued before the
//    current one is multiplied and written to the other LDS buffer after it.
//  * gemm_narrow: more than 16 rows against at most 64 weight rows (a router): operands straight from memory, K
//    shared out over the waves of a workgroup.
//  * gemm_skinny: M <= 64 rows (decode): pure weight streaming.  A workgroup owns 16*RB
//    weight rows; its 4 waves take interleaved 128-element k-chunks, every lane reading
//    64 contiguous bytes of one weight row per chunk straight into v_mfma_f32_16x16x32_bf16
//    operands (the k-permutation inside a chunk is the same for both operands, so the dot
//    product is unchanged); the waves' partial sums are added in wave order in LDS.
//
// reference: op_linear_proj (GEMV per output row, kernels/megakernel_ops.hip:166-276) for
// what is computed; wmma_gemm_bf16 (kernels/wmma_gemm_bf16.hip:27-82, one wave32 per 16x16
// tile without LDS, used only by its tests) for the matrix-core form on RDNA3.
#include "common.h"

// output modes
#define OUT_BF16 0
#define OUT_F32 1
#define OUT_F32_ACC 2
// SwiGLU epilogue: W holds gate and up rows interleaved in blocks of 16 (8 gate rows, then
// the 8 up rows of the same outputs); the output is bf16 [M, N / 2] with
// out[m][8 b + j] = silu(gate) * up, silu(g) = g / (1 + exp(-g))
// (reference: kernels/megakernel_ops.hip:1538-1544, fused there too, per output row).
#define OUT_SWIGLU 3
#define SSQ_LD 64           // row stride of the sums of squares that a product leaves for the next RMS norm

__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.f + expf(-g)) * u; }

template <int MODE>
__device__ __forceinline__ void store_out(void* C, size_t idx, float v) {
    if (MODE == OUT_BF16) ((bf16*)C)[idx] = (bf16)v;
    else if (MODE == OUT_F32) ((float*)C)[idx] = v;
    else if (MODE == OUT_F32_ACC) ((float*)C)[idx] += v;
}

__device__ __forceinline__ bf16x8 zero8() {
    bf16x8 z;
#pragma unroll
    for (int i = 0; i < 8; ++i) z[i] = (bf16)0.f;
    return z;
}

// 8 consecutive bf16 of row `row` at k; zeros outside [0,rows) x [0,K).
template <bool ALIGNED>
__device__ __forceinline__ bf16x8 load8(const bf16* __restrict__ base, size_t ld, int row, int rows, int k, int K) {
    if (row >= rows || k >= K) return zero8();
    const bf16* p = base + (size_t)row * ld + k;
    if (ALIGNED) {
        if (k + 8 <= K) return *(const bf16x8*)p;
    }
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (k + i < K) ? p[i] : (bf16)0.f;
    return v;
}

// Store a wave's TM x TN grid of 32x32 accumulator blocks whose first element is (m1, n1).
// acc[i][j][r]: row = 8 (r / 4) + 4 (lane / 32) + r % 4, column = lane % 32 of the block.
template <int TM, int TN, int MODE>
__device__ __forceinline__ void tile_epilogue(f32x16 (&acc)[TM][TN], void* __restrict__ C, int M, int N, size_t ldc,
                                              int m1, int n1, int lane) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n1 + j * 32 + (lane & 31);
            if (MODE == OUT_SWIGLU) {
                // the up value of a gate column sits 8 columns on, in lane ^ 8
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float other = __shfl_xor(acc[i][j][r], 8, 64);
                    const int m = m1 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if ((lane & 8) == 0 && n < N && m < M)
                        ((bf16*)C)[(size_t)m * ldc + (n >> 4) * 8 + (n & 7)] = (bf16)silu_mul(acc[i][j][r], other);
                }
                continue;
            }
            if (n >= N) continue;
            // one 64-bit address per block; the 16 rows of a lane are reached by 32-bit offsets
            const int mb = m1 + i * 32 + 4 * (lane >> 5);
            const size_t base = (size_t)mb * ldc + n;
            const unsigned ld32 = (unsigned)ldc;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int dm = 8 * (r >> 2) + (r & 3);
                if (mb + dm < M) store_out<MODE>(C, base + (size_t)(dm * ld32), acc[i][j][r]);
            }
            // keep the blocks' stores apart: moving every accumulator out of the matrix-core
            // registers at once would not fit the register file of the large tiles
            __builtin_amdgcn_sched_barrier(0);
        }
}

// ------------------------------------------------------------------ gemm_tile -------
template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, int MODE, bool ALIGNED, bool KFULL>
__global__ __launch_bounds__(256) void gemm_tile_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                        void* __restrict__ C, int M, int N, int K,
                                                        size_t lda, size_t ldc, int tiles_m, int tiles_n) {
    static_assert(WAVES_M * WAVES_N == 4, "4 waves");
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;      // per-wave tile
    constexpr int TM = WM / 32, TN = WN / 32;
    constexpr int LDS_LD = BK + 8;                           // padded row, in bf16
    constexpr int A_CHUNKS = BM * BK / 8 / 256, B_CHUNKS = BN * BK / 8 / 256;
    constexpr int CPR = BK / 8;                              // 16-byte chunks per tile row
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    bf16* As = (bf16*)smem;                                  // [2][BM][LDS_LD]
    bf16* Bs = As + 2 * BM * LDS_LD;                         // [2][BN][LDS_LD]

    // Workgroups are dealt round-robin to the 8 XCDs; give each XCD a contiguous run of
    // tiles (n-major, m inner) so that the workgroups sharing an L2 share weight tiles.
    const int total = tiles_m * tiles_n;
    int pid = blockIdx.x;
    {
        const int per = total / 8, xcd = pid % 8, idx = pid / 8;
        if (pid < per * 8) pid = xcd * per + idx;
    }
    const int tile_n = pid / tiles_m, tile_m = pid - tile_n * tiles_m;
    const int m0 = tile_m * BM, n0 = tile_n * BN;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave / WAVES_N) * WM, wn = (wave % WAVES_N) * WN;
    const int lrow = lane & 31, lk = (lane >> 5) * 8;

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // Rows beyond M or N are read from the last valid row (and dropped at the store), so a
    // load needs a guard along k only; with K a multiple of BK and 16-byte aligned rows
    // (KFULL) it needs none.
    bf16x8 ra[A_CHUNKS], rb[B_CHUNKS];
    const bf16* ap[A_CHUNKS];
    const bf16* bp[B_CHUNKS];
    int akc[A_CHUNKS], bkc[B_CHUNKS];
#pragma unroll
    for (int c = 0; c < A_CHUNKS; ++c) {
        const int id = tid + c * 256;
        int r = m0 + id / CPR;
        if (r > M - 1) r = M - 1;
        akc[c] = (id % CPR) * 8;
        ap[c] = A + (size_t)r * lda + akc[c];
    }
#pragma unroll
    for (int c = 0; c < B_CHUNKS; ++c) {
        const int id = tid + c * 256;
        int r = n0 + id / CPR;
        if (r > N - 1) r = N - 1;
        bkc[c] = (id % CPR) * 8;
        bp[c] = W + (size_t)r * K + bkc[c];
    }
    auto gload = [&](int k0) {
#pragma unroll
        for (int c = 0; c < A_CHUNKS; ++c) {
            if (KFULL) ra[c] = *(const bf16x8*)(ap[c] + k0);
            else ra[c] = load8<ALIGNED>(ap[c] - akc[c], 0, 0, 1, k0 + akc[c], K);
        }
#pragma unroll
        for (int c = 0; c < B_CHUNKS; ++c) {
            if (KFULL) rb[c] = *(const bf16x8*)(bp[c] + k0);
            else rb[c] = load8<ALIGNED>(bp[c] - bkc[c], 0, 0, 1, k0 + bkc[c], K);
        }
    };
    auto sstore = [&](int buf) {
        bf16* a = As + buf * BM * LDS_LD;
        bf16* b = Bs + buf * BN * LDS_LD;
#pragma unroll
        for (int c = 0; c < A_CHUNKS; ++c) {
            const int id = tid + c * 256, r = id / CPR, kc = (id % CPR) * 8;
            *(bf16x8*)(a + r * LDS_LD + kc) = ra[c];
        }
#pragma unroll
        for (int c = 0; c < B_CHUNKS; ++c) {
            const int id = tid + c * 256, r = id / CPR, kc = (id % CPR) * 8;
            *(bf16x8*)(b + r * LDS_LD + kc) = rb[c];
        }
    };

    const int nk = (K + BK - 1) / BK;
    gload(0);
    sstore(0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk) gload((kt + 1) * BK);
        const bf16* a = As + buf * BM * LDS_LD + (wm + lrow) * LDS_LD + lk;
        const bf16* b = Bs + buf * BN * LDS_LD + (wn + lrow) * LDS_LD + lk;
#pragma unroll
        for (int kk = 0; kk < BK; kk += 16) {
            bf16x8 fa[TM], fb[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[i] = *(const bf16x8*)(a + i * 32 * LDS_LD + kk);
#pragma unroll
            for (int j = 0; j < TN; ++j) fb[j] = *(const bf16x8*)(b + j * 32 * LDS_LD + kk);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < nk) sstore(buf ^ 1);
        __syncthreads();
    }

    tile_epilogue<TM, TN, MODE>(acc, C, M, N, ldc, m0 + wm, n0 + wn, lane);
}

template <int BM, int BN, int BK, int WAVES_M, int WAVES_N>
static int launch_tile(const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc,
                       int mode, bool aligned, hipStream_t s) {
    const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
    const long long total = (long long)tm * tn;
    if (total > 0x7fffffffLL) return BR_BAD_ARG;
    const size_t lds = (size_t)2 * (BM + BN) * (BK + 8) * sizeof(bf16);
#define BR_LAUNCH_TILE_(MODE, AL, KF)                                                                    \
    do {                                                                                                \
        auto kern = gemm_tile_kernel<BM, BN, BK, WAVES_M, WAVES_N, MODE, AL, KF>;                       \
        if (lds > 48 * 1024) {                                                                          \
            static bool set = false;                                                                    \
            if (!set) {                                                                                 \
                if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,  \
                                        (int)lds) != hipSuccess) return BR_LAUNCH_FAILED;               \
                set = true;                                                                             \
            }                                                                                           \
        }                                                                                               \
        kern<<<(unsigned)total, 256, lds, s>>>(A, W, C, M, N, K, lda, ldc, tm, tn);                     \
    } while (0)
#define BR_LAUNCH_TILE(MODE)                                                 \
    do {                                                                     \
        if (aligned && K % BK == 0) BR_LAUNCH_TILE_(MODE, true, true);       \
        else if (aligned) BR_LAUNCH_TILE_(MODE, true, false);                \
        else BR_LAUNCH_TILE_(MODE, false, false);                            \
    } while (0)
    if (mode == OUT_BF16) BR_LAUNCH_TILE(OUT_BF16);
    else if (mode == OUT_F32) BR_LAUNCH_TILE(OUT_F32);
    else if (mode == OUT_F32_ACC) BR_LAUNCH_TILE(OUT_F32_ACC);
    else BR_LAUNCH_TILE(OUT_SWIGLU);
#undef BR_LAUNCH_TILE_
#undef BR_LAUNCH_TILE
    return br_check_launch();
}

// -------------------------------------------------------------- gemm_tile_dma -------
// The tile product for aligned shapes (K a multiple of 64, 16-byte aligned rows): tiles
// go from memory to LDS by direct global-to-LDS loads (global_load_lds_dwordx4: a wave
// writes 1 KB = 8 tile rows of 64 k, no registers, no ds_write), into a ring of S stages.
// A row's eight 16-byte columns are stored XOR-swizzled by (row / 2) % 8, which makes the
// operand reads of 16 consecutive rows conflict-free; the swizzle is applied by choosing
// the global column each lane fetches.  Rows beyond M or N are fetched from the last
// valid row and dropped at the store.
//
// The loads are issued from inline assembly and counted by hand: before a stage is
// read, `s_waitcnt vmcnt(n)` leaves only the younger stages' loads outstanding, then a
// barrier makes every wave's part of the stage visible (and says that the stage about to
// be overwritten has been read by all).  The kernel issues no other vector memory
// operation inside the loop, so the count is exact.
// Weight layouts (`wl`).  0: N rows of K.  1: blocks of 16 rows x 128 k, 4 KB contiguous each, ordered
// [row block][k block], rows padded to a multiple of 16 (K in steps of 128): a 16-row strip is one
// contiguous run along k.  A streaming product then reads 4 KB pieces, in order, instead of 256 bytes
// from every row, which the memory serves faster (bare loads of a 64-row tile by every workgroup: 5.4 to
// 5.9 against 4.1 to 4.6 TB/s; in the products: wide matrices at 17 to 128 rows gain 10 to 15 %, up to
// 16 rows 0 to 5 %, the rest nothing).  Blocks of 64 rows were tried: slower up to 16 rows.
#define WL_ROWS 0
#define WL_BLOCKED 1
#ifndef WL_BLOCK_ROWS
#define WL_BLOCK_ROWS 16
#endif
#define WL_BLOCK_ELEMS (WL_BLOCK_ROWS * 128)
__device__ __forceinline__ size_t w_row_base(int n, int K, int wl) {
    return wl ? (size_t)(n / WL_BLOCK_ROWS) * (size_t)(K >> 7) * WL_BLOCK_ELEMS + (size_t)((n % WL_BLOCK_ROWS) << 7)
              : (size_t)n * K;
}
#define DMA_BK 64
#define DMA_ISSUE(ST, kt)                                                                                      \
    do {                                                                                                       \
        _Pragma("unroll") for (int q = 0; q < INSTR; ++q) {                                                    \
            const unsigned lds_ = __builtin_amdgcn_readfirstlane(                                              \
                (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)(ST)) + dst[q]);          \
            if (once[q])                                   /* weights that no other row of tiles reads */      \
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds_), "v"(src[q]) \
                             : "m0");                                                                          \
            else                                                                                               \
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_), "v"(src[q]) \
                             : "m0");                                                                          \
            src[q] += (knext & 1) ? hop[q] : DMA_BK;       /* k-tiles are issued in order, (kt) is the next */ \
        }                                                                                                      \
        if (++knext == kwrap) {                            /* on to the run's first k-tile */                  \
            knext = kt0;                                                                                       \
            _Pragma("unroll") for (int q = 0; q < INSTR; ++q) src[q] -= (size_t)(nk_run >> 1) * (DMA_BK + hop[q]); \
        }                                                                                                      \
    } while (0)
#define DMA_COMPUTE(ST)                                                                                        \
    do {                                                                                                       \
        _Pragma("unroll") for (int kk = 0; kk < 4; ++kk) {                                                     \
            bf16x8 fa[TM], fb[TN];                                                                             \
            const int c = kk * 2 + g;                                                                          \
            _Pragma("unroll") for (int i = 0; i < TM; ++i) {                                                   \
                const int r = wm + i * 32 + lrow;                                                              \
                fa[i] = *(const bf16x8*)((ST) + r * 128 + ((c ^ ((r >> 1) & 7)) * 16));                        \
            }                                                                                                  \
            _Pragma("unroll") for (int j = 0; j < TN; ++j) {                                                   \
                const int r = BM + wn + j * 32 + lrow;                                                         \
                fb[j] = *(const bf16x8*)((ST) + r * 128 + ((c ^ ((r >> 1) & 7)) * 16));                        \
            }                                                                                                  \
            _Pragma("unroll") for (int i = 0; i < TM; ++i)                                                     \
                _Pragma("unroll") for (int j = 0; j < TN; ++j)                                                 \
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);     \
        }                                                                                                      \
    } while (0)
#define DMA_WAITBAR(N)                                              \
    do {                                                            \
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");    \
        __builtin_amdgcn_s_barrier();                               \
        asm volatile("" ::: "memory");                              \
    } while (0)

template <int BM, int BN, int WAVES_M, int WAVES_N, int S, int MODE>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) void gemm_tile_dma_kernel(
    const bf16* __restrict__ A, const bf16* __restrict__ W, void* __restrict__ C_, int M, int N, int K, size_t lda,
    size_t ldc, int tiles_m, int tiles_n, int kt_per_part, size_t part_stride, int wl) {
    constexpr int NW = WAVES_M * WAVES_N;
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, TM = WM / 32, TN = WN / 32;
    constexpr int STAGE_BYTES = (BM + BN) * DMA_BK * 2;
    // blockIdx.y: which run of k-tiles this workgroup sums (one run, or the parts of a split
    // product, each into a float matrix of its own `part_stride` elements on)
    void* C = MODE == OUT_F32 ? (void*)((float*)C_ + blockIdx.y * part_stride) : C_;
    constexpr int INSTR = (BM + BN) / 8 / NW;           // 1 KB wave-loads per wave and stage
    static_assert(S == 2 || S == 3, "2 or 3 stages");
    __shared__ __attribute__((aligned(1024))) unsigned char st0[STAGE_BYTES];
    __shared__ __attribute__((aligned(1024))) unsigned char st1[STAGE_BYTES];
    __shared__ __attribute__((aligned(1024))) unsigned char st2[S >= 3 ? STAGE_BYTES : 16];

    // each XCD takes a contiguous run of tiles, in groups of 8 tile columns by all tile rows
    const int total = tiles_m * tiles_n;
    int pid = blockIdx.x;
    {
        const int per = total / 8, xcd = pid % 8, idx = pid / 8;
        if (pid < per * 8) pid = xcd * per + idx;
    }
    const int grp = pid / (8 * tiles_m), in = pid - grp * 8 * tiles_m;
    int gn = tiles_n - grp * 8;
    if (gn > 8) gn = 8;
    const int tile_n = grp * 8 + in % gn, tile_m = in / gn;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave / WAVES_N) * WM, wn = (wave % WAVES_N) * WN;
    const int lrow = lane & 31, g = lane >> 5;

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // wave-load q of this wave covers rows (q NW + wave) 8 .. + 8 of the stacked tile [A rows | W rows]
    const bf16* src[INSTR];
    int dst[INSTR];
    int hop[INSTR];                                      // elements from an odd k-tile to the next (even) one
    bool once[INSTR];                                    // a load of weight rows that are read this once (non-temporal)
    const int kt0 = (int)blockIdx.y * kt_per_part;       // the run's first k-tile
    int nk_run = K / DMA_BK - kt0;                       // k-tiles of this run
    if (nk_run > kt_per_part) nk_run = kt_per_part;
    // Where in its run a workgroup starts (it wraps round): workgroups that walk k in step ask the same few
    // memory channels at the same time.  Only with a single row of tiles (3 to 6 % on wide matrices at
    // 65 to 128 rows): workgroups that share a tile live on reading the same k-tile at the same time (a start
    // of its own for each made 2,048 rows 50 % slower, one per tile column made 2 rows of tiles 5 to 12 %
    // slower).  An even start in an even run, so that pairs of k-tiles (one 128-wide block of the blocked
    // layout) stay together.
    const int rot = (tiles_m == 1 && nk_run % 2 == 0 && kt0 % 2 == 0)
                        ? 2 * (int)((((unsigned)tile_n * 2654435761u) >> 8) % (unsigned)(nk_run / 2)) : 0;
    const int kwrap = kt0 + nk_run;
    int knext = kt0 + rot;                               // the k-tile that src[] points at
#pragma unroll
    for (int q = 0; q < INSTR; ++q) {
        const int R = (q * NW + wave) * 8 + (lane >> 3);
        const int c = (lane & 7) ^ ((R >> 1) & 7);       // the global 16-byte column this lane fetches
        if (R < BM) {
            int r = m0 + R;
            if (r > M - 1) r = M - 1;
            src[q] = A + (size_t)r * lda + c * 8 + (size_t)(kt0 + rot) * DMA_BK;
            hop[q] = DMA_BK;
        } else {
            int r = n0 + R - BM;
            if (r > N - 1) r = N - 1;
            src[q] = W + w_row_base(r, K, wl) + c * 8 +
                     (wl ? (size_t)((kt0 + rot) >> 1) * WL_BLOCK_ELEMS + (kt0 & 1) * DMA_BK : (size_t)(kt0 + rot) * DMA_BK);
            hop[q] = wl ? WL_BLOCK_ELEMS - DMA_BK : DMA_BK;
        }
        hop[q] = __builtin_amdgcn_readfirstlane(hop[q]);             // the same for the 8 rows of a wave-load
        once[q] = __builtin_amdgcn_readfirstlane((int)((q * NW + wave) * 8 >= BM && tiles_m == 1)) != 0;
        dst[q] = (q * NW + wave) * 1024;
    }
    const int nk = nk_run;
    if (S == 2) {
        DMA_ISSUE(st0, 0);
        for (int kt = 0; kt < nk; kt += 2) {
            DMA_WAITBAR(0);
            if (kt + 1 < nk) DMA_ISSUE(st1, kt + 1);
            DMA_COMPUTE(st0);
            if (kt + 1 >= nk) break;
            DMA_WAITBAR(0);
            if (kt + 2 < nk) DMA_ISSUE(st0, kt + 2);
            DMA_COMPUTE(st1);
        }
    } else {
        DMA_ISSUE(st0, 0);
        if (nk > 1) DMA_ISSUE(st1, 1);
        int kt = 0;
        // steady state: two stages are in flight at every wait, the older one is waited for
        for (; kt + 5 <= nk; kt += 3) {
            DMA_WAITBAR(INSTR);
            DMA_ISSUE(st2, kt + 2);
            DMA_COMPUTE(st0);
            DMA_WAITBAR(INSTR);
            DMA_ISSUE(st0, kt + 3);
            DMA_COMPUTE(st1);
            DMA_WAITBAR(INSTR);
            DMA_ISSUE(st1, kt + 4);
            DMA_COMPUTE(st2);
        }
        // the last tiles: wait for everything in flight
        for (; kt < nk; kt += 3) {
            DMA_WAITBAR(0);
            if (kt + 2 < nk) DMA_ISSUE(st2, kt + 2);
            DMA_COMPUTE(st0);
            if (kt + 1 >= nk) break;
            DMA_WAITBAR(0);
            if (kt + 3 < nk) DMA_ISSUE(st0, kt + 3);
            DMA_COMPUTE(st1);
            if (kt + 2 >= nk) break;
            DMA_WAITBAR(0);
            if (kt + 4 < nk) DMA_ISSUE(st1, kt + 4);
            DMA_COMPUTE(st2);
        }
    }
    tile_epilogue<TM, TN, MODE>(acc, C, M, N, ldc, m0 + wm, n0 + wn, lane);
}

// ------------------------------------------------------------ gemm_tile_quad -------
// A BM x BN tile by four waves (2 x 2, or 4 x 1 for the 256x224 tile), one to a SIMD, each summing a quarter of it in the matrix-core
// registers (256x256: 16 blocks of 32x32, all 256 of them), with the operands of one k-step of 16 in
// vector registers, twice (the set in use and the set being read from LDS).  Per matrix instruction
// half the LDS operand bytes of the 64x64 wave tiles above.  With one wave per SIMD nothing fills a gap
// in that wave's instruction stream, so the order is written out: matrix instructions, LDS reads,
// direct loads and waits are inline assembly in program order.  The compiler keeps volatile statements
// in order, but it neither knows their latencies nor that they are matrix instructions: every wait is
// placed by hand, and so are the idle states that the hardware wants between a register's write and
// a matrix instruction's read of it (and the reverse).
// Each operand has a ring of two or three stages of 64 k (the layout and swizzle of gemm_tile_dma).  One
// barrier per k-tile, before its last k-step of 16: by then every wave has read the stages in use.  An
// operand with two stages is asked for after that barrier, into the stage just read; one with three
// during the k-steps before it, into the stage that the barrier before freed: a compute unit's path into
// LDS takes one 1 KB load per 16 cycles, so a k-tile's loads are spread over it, not bunched (bunched,
// the waves wait at their load instructions with the matrix cores idle behind them).
// The blocks hold the product transposed (weight rows are the instruction's first operand), which
// gives every lane four neighbouring columns of one output row: 16-byte accesses in the epilogue, and
// the up value of a gate column in the same lane.
typedef int i32x4 __attribute__((ext_vector_type(4)));
template <int I, int N_, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N_) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N_>(f);
    }
}
template <int OFF>
__device__ __forceinline__ void quad_read(i32x4& d, unsigned addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(d) : "v"(addr), "n"(OFF));
}
template <int IMM>
__device__ __forceinline__ void quad_load(unsigned lds_base, unsigned voff, unsigned long long sbase) {
    asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
                 ::"s"(lds_base), "n"(IMM), "v"(voff), "s"(sbase)
                 : "m0", "scc", "memory");
}
__device__ __forceinline__ void quad_mfma(f32x16& acc, const i32x4& a, const i32x4& b) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void quad_touch(f32x16& acc) { asm volatile("s_nop 1" : "+a"(acc)); }
template <int N_>
__device__ __forceinline__ void quad_wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N_) : "memory");
}

// Products of several experts in one launch (GROUPED): expert e's activation rows are the pairs first[e] .. first[e + 1] - 1
// (rows of A themselves, or with `order` the rows order[p] / top; `per` is 2^32 / top rounded up, or 0 where that is not exact), its weights lie N rows behind the expert before.  With
// the gated epilogue weight row v of a tile is gate row 8 (v / 16) + v % 16 or, from v % 16 = 8 on, the up row N / 2 behind
// it, so that the matrices stay as they are stacked; `alpha` > 0: the clamped unit.
struct QuadGroups {
    const int* first;
    const int* order;
    int experts, top;
    unsigned per;
    float limit, alpha;
};
// Several inputs by stacked weights in one launch (BRANCHES): the weight rows b * per .. of a column of tiles multiply the activations
// `a_step` elements behind the branch before; results leave `gap` columns alone in front of branch gap_at / per.
struct QuadBranches {
    int per;
    size_t a_step;
    int gap_at, gap;
    int whole;
};
// `whole`: the last tile of rows multiplies all of its blocks, also those without rows.  For products of one round of workgroups: what it saves
// ends no round earlier, and tiles that run ahead of the others read the weights from farther off than the L2 (gated 28,672 x 4,096 by
// 129 / 150 / 192 rows 65 / 60 / 55 us with its rows alone, 57 / 52 / 53 whole; 4,096 x 14,336 by 900 106 and 101).
struct QuadPlain {
    int whole;
};
enum { QUAD_PLAIN = 0, QUAD_EXPERTS = 1, QUAD_BRANCHES = 2 };
template <int KIND> struct QuadArg { typedef QuadPlain type; };
template <> struct QuadArg<QUAD_EXPERTS> { typedef QuadGroups type; };
template <> struct QuadArg<QUAD_BRANCHES> { typedef QuadBranches type; };
__device__ __forceinline__ float quad_glu(float g, float u, const QuadGroups& gr) {
    if (gr.alpha > 0.f) {
        g = fminf(g, gr.limit);
        u = fminf(fmaxf(u, -gr.limit), gr.limit);
        return g / (1.0f + expf(-gr.alpha * g)) * (u + 1.0f);
    }
    return silu_mul(g, u);
}

// acc[i][j][r]: weight row (output column) n1 + 32 i + 8 (r / 4) + 4 (lane / 32) + r % 4, activation
// row m1 + 32 ST j + lane % 32.  Needs ldc % 4 == 0 and C aligned to 16 bytes.
// What is only written goes through the wave's piece of LDS, 32 rows at a time, so that an instruction writes whole runs of rows: as
// the blocks lie, it would write 16 or 32 bytes of each of 32 rows, and 256 workgroups that end a round together wait for the L2's
// requests.  8,192 x 8,192 by K = 1,024 in bfloat16 153 -> 130 us; 6,144 x 4,096 by 3,625 rows 155.5 -> 150, by 7,001 rows 282 -> 272; float
// 12,288 x 4,096 by 7,001 rows 573 -> 565.  What is added to stays as the blocks lie: its reads and writes fill the memory's time
// either way, and through LDS (with up to half of the values asked for some k-tiles ahead) 4,096 x 4,096 by 3,625 and 5,018 rows took
// 112.5 and 167 us against 111.5 and 164, 4,096 x 14,336 by 7,001 rows 674 against 648.
template <int TI, int MODE>
struct QuadStrip {
    static constexpr int ES = MODE == OUT_BF16 || MODE == OUT_SWIGLU ? 2 : 4;            // bytes of an element
    static constexpr int RB = TI * 32 / (MODE == OUT_SWIGLU ? 2 : 1) * ES;                // of a row
    static constexpr int LD = RB + 16;                                                   // from row to row, off the banks' stride
    static constexpr int BYTES = MODE == OUT_F32_ACC ? 0 : 32 * LD;
};
template <int TI, int TJ, int ST, int MODE, bool GROUPED, class Arg>
__device__ __forceinline__ void quad_epilogue(f32x16 (&acc)[TI][TJ], void* __restrict__ C, int M, int N, size_t ldc, int m1, int n1, int lane,
                                              const Arg& gr, unsigned char* lds) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    if constexpr (MODE == OUT_F32_ACC) {
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int m = m1 + j * 32 * ST + (lane & 31);
            if (m >= M) continue;
#pragma unroll
            for (int i = 0; i < TI; ++i) {
                const int nb = n1 + i * 32 + 4 * (lane >> 5);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int n = nb + 8 * q;
                    const size_t at = (size_t)m * ldc + n;
                    if (n + 3 < N) {
                        f32x4 v = *(const f32x4*)((float*)C + at);
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] += acc[i][j][4 * q + e];
                        *(f32x4*)((float*)C + at) = v;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (n + e < N) store_out<MODE>(C, at + e, acc[i][j][4 * q + e]);
                    }
                }
            }
        }
    } else {
        struct __attribute__((packed, aligned(8))) Out { unsigned w[4]; };               // bfloat16 rows are aligned to 8 bytes
        typedef QuadStrip<TI, MODE> S;
        constexpr int CH = S::RB / 16, EL = 16 / S::ES;                                  // pieces of 16 bytes of a row, elements of one
        auto unit = [&](float x, float u) {
            if constexpr (GROUPED) return quad_glu(x, u, gr);
            else return silu_mul(x, u);
        };
        if (MODE == OUT_SWIGLU) {
            N >>= 1;
            n1 >>= 1;
        }
        unsigned char* const put = lds + (lane & 31) * S::LD + 4 * (lane >> 5) * S::ES;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int mj = m1 + j * 32 * ST;
            if (mj >= M) break;
#pragma unroll
            for (int i = 0; i < TI; ++i) {
                if (MODE == OUT_SWIGLU) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {                   // gate rows 32 i + 16 h + 4 (lane / 32) + 0 .. 3, up rows 8 on
                        bf16x4 v;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            v[e] = (bf16)unit(acc[i][j][8 * h + e], acc[i][j][8 * h + 4 + e]);
                        *(bf16x4*)(put + (16 * i + 8 * h) * 2) = v;
                    }
                    continue;
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (MODE == OUT_BF16) {
                        bf16x4 v;
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = (bf16)acc[i][j][4 * q + e];
                        *(bf16x4*)(put + (32 * i + 8 * q) * 2) = v;
                    } else {
                        f32x4 v;
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * q + e];
                        *(f32x4*)(put + (32 * i + 8 * q) * 4) = v;
                    }
                }
            }
            // (the wave's own writes and reads of LDS are executed in order)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int t = 0; t < CH / 2; ++t) {
                const int c = t * 64 + lane, row = c / CH, piece = c % CH, m = mj + row, n = n1 + piece * EL;
                if (m >= M || n >= N) continue;
                const unsigned char* from = lds + row * S::LD + piece * 16;
                const size_t at = (size_t)m * ldc + n;
                if (n + EL <= N) {
                    if (S::ES == 2) *(Out*)((bf16*)C + at) = *(const Out*)from;
                    else *(f32x4*)((float*)C + at) = *(const f32x4*)from;
                } else {
                    for (int e = 0; e < EL && n + e < N; ++e) {
                        if (S::ES == 2) ((bf16*)C)[at + e] = ((const bf16*)from)[e];
                        else ((float*)C)[at + e] = ((const float*)from)[e];
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
}

template <int BM, int BN, int NSA, int NSB, int WVM, int MODE, int KIND = QUAD_PLAIN>
__global__ __launch_bounds__(256) void gemm_tile_quad_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                              void* __restrict__ C_, int M, int N, int K, size_t lda,
                                                              size_t ldc, int tiles_m, int tiles_n, int kt_per_part,
                                                              size_t part_stride, int wl, typename QuadArg<KIND>::type gr) {
    constexpr bool GROUPED = KIND == QUAD_EXPERTS;
    // Branches by tiles of 128 rows: runs of kt_per_part k-tiles, one after another, whose sums are added up in registers in the order and with the
    // bits of gemm_split_sum_kernel (a tile of 256 rows has no registers left for them).
    constexpr bool RUNS = KIND == QUAD_BRANCHES && BM == 128;
    constexpr int SA = BM * 128, SB = BN * 128;          // bytes of a stage of activation rows, of weight rows
    constexpr int WVN = 4 / WVM;                         // the four waves: WVM along the activation rows x WVN
    constexpr int TI = BN / WVN / 32, TJ = BM / WVM / 32; // blocks of a wave: weight rows, activation rows
    constexpr int LA = BM / 32, LB = BN / 32;            // wave-loads per wave and stage
    // An operand with three stages is asked for during the first three k-steps of 16 of a k-tile, into the
    // stage that the barrier before freed, and has a whole k-tile more to arrive; one with two stages after
    // the barrier, into the stage just read.  Either way k-tile t asks for k-tile t + 2.
    constexpr bool EARLY_A = NSA == 3, EARLY_B = NSB == 3;
    static_assert((WVM == 2 || WVM == 4) && BM % (32 * WVM) == 0 && BN % (32 * WVN) == 0 && BM % 32 == 0 && BN % 32 == 0 &&
                      NSA * SA + NSB * SB <= 160 * 1024 && TI * TJ * 16 <= 256, "tile");
    static_assert((NSA == 2 || NSA == 3) && (NSB == 2 || NSB == 3), "two or three stages an operand");
    static_assert(TI + TJ <= TI * TJ, "schedule");
    static_assert(4 * QuadStrip<TI, MODE>::BYTES <= NSA * SA + NSB * SB, "the epilogue's strips");
    __shared__ __attribute__((aligned(1024))) unsigned char st[NSA * SA + NSB * SB];
    // blockIdx.y: which run of k-tiles this workgroup sums (one run, or the parts of a split product, each
    // into a float matrix of its own `part_stride` elements on; runs start at an even k-tile)
    void* C = MODE == OUT_F32 ? (void*)((float*)C_ + blockIdx.y * part_stride) : C_;
    const int kt0 = (int)blockIdx.y * kt_per_part;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // A wave's blocks of activation rows lie 32 ST apart: side by side where the product is added to what is there (a wave then reads and writes neighbouring
    // rows: 4,096 x 1,792 by 5,018 rows 89 us, 96 with the waves' blocks in turn), else the waves' blocks in turn, so that a last tile of few rows leaves
    // every wave as many.
    constexpr int ST = MODE == OUT_F32_ACC ? 1 : WVM;
    const int wm = (wave / WVN) * (ST == 1 ? BM / WVM : 32), wn = (wave % WVN) * (BN / WVN);
    const int lrow = lane & 31, g = lane >> 5;
    int nk = K / DMA_BK - kt0;                                         // k-tiles of this run
    if (nk > kt_per_part) nk = kt_per_part;
    const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)st);

    // One tile: rows m0 .. of A up to row m_end against the weight rows n0 .. of W_, k-tiles kt0 .. kt0 + nk.
    auto tile = [&](const bf16* A_, const bf16* W_, int m0, int n0, int m_end) {
    f32x16 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    f32x16 sum[RUNS ? TI : 1][RUNS ? TJ : 1];
    if constexpr (RUNS) {
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j) sum[i][j] = acc[i][j];
    }

    // wave-load q of this wave: rows (4 q + wave) 8 .. + 8 of the operand's tile, reached by a 32-bit byte
    // offset from the matrix's first element (the launcher checks that this suffices); the pairs of an expert
    // without `order`, of which a step may bring more than 4 GB, from the tile's first row
    int row0 = 0;
    if constexpr (GROUPED) {
        if (!gr.order) {
            A_ += (size_t)m0 * lda;
            row0 = m0;
        }
    }
    unsigned offA[LA], offB[LB];
#pragma unroll
    for (int q = 0; q < (LA > LB ? LA : LB); ++q) {
        const int R = (q * 4 + wave) * 8 + (lane >> 3);
        const int c = (lane & 7) ^ ((R >> 1) & 7);
        if (q < LA) {
            int r = m0 + R;
            if (r > m_end - 1) r = m_end - 1;
            if constexpr (GROUPED) {
                r = gr.order ? (gr.per ? (int)__umulhi((unsigned)gr.order[r], gr.per) : gr.order[r] / gr.top) : r - row0;
            }
            offA[q] = (unsigned)((size_t)r * lda * 2 + c * 16);
        }
        if (q < LB) {
            int r = n0 + R;
            if (r > N - 1) r = N - 1;
            if constexpr (GROUPED && MODE == OUT_SWIGLU) r = (r >> 4) * 8 + (r & 7) + ((r & 8) ? N / 2 : 0);
            offB[q] = (unsigned)(w_row_base(r, K, wl) * 2 + c * 16);
        }
    }
    // at the next k-tile to ask for
    unsigned long long baseA = (unsigned long long)A_ + (size_t)kt0 * 128;
    unsigned long long baseW = (unsigned long long)W_ + (wl ? (size_t)(kt0 >> 1) * (WL_BLOCK_ELEMS * 2) : (size_t)kt0 * 128);
    int knext = kt0;
    const unsigned hopW = wl ? WL_BLOCK_ELEMS * 2 - 128 : 128;                        // bytes from an odd k-tile on
    for (int rest = K / DMA_BK - nk;;) {                 // run by run (RUNS), or once
    // where this wave's loads of the next k-tile to ask for land, and which stage that is
    unsigned ldsA = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024);
    unsigned ldsB = __builtin_amdgcn_readfirstlane(lds0 + NSA * SA + wave * 1024);
    int slotA = 0, slotB = 0;
    // LDS addresses of this lane's operand pieces in the stage in use, per k-step of 16, and which stage that is
    unsigned ra[4], rb[4];
    int curA = 0, curB = 0;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        const int col = ((kk * 2 + g) ^ ((lrow >> 1) & 7)) * 16;
        ra[kk] = lds0 + (wm + lrow) * 128 + col;
        rb[kk] = lds0 + NSA * SA + (wn + lrow) * 128 + col;
    }
    i32x4 fa[2][TJ], fb[2][TI];

    auto loadA = [&](auto q_) {
        constexpr int q = decltype(q_)::value;
        quad_load<q * 4096>(ldsA, offA[q], baseA);
    };
    auto loadB = [&](auto q_) {
        constexpr int q = decltype(q_)::value;
        quad_load<q * 4096>(ldsB, offB[q], baseW);
    };
    auto next_tile = [&]() {                       // the pointers and the stages to load go on by a k-tile
        baseA += 128;
        baseW += (knext & 1) ? hopW : 128;
        ++knext;
        ldsA += slotA == NSA - 1 ? (unsigned)(-(NSA - 1) * SA) : (unsigned)SA;
        slotA = slotA == NSA - 1 ? 0 : slotA + 1;
        ldsB += slotB == NSB - 1 ? (unsigned)(-(NSB - 1) * SB) : (unsigned)SB;
        slotB = slotB == NSB - 1 ? 0 : slotB + 1;
    };
    // The k-loop over TV blocks of activation rows a wave: all of a tile's, or fewer where its rows end.
    auto run = [&](auto tv_) {
        constexpr int TV = decltype(tv_)::value;
        constexpr int NM = TI * TV, NR = TI + TV;  // matrix instructions and operand reads per k-step of 16
        constexpr int LV = LA / TJ * TV;           // wave-loads of activation rows per wave and stage
        constexpr int NEARLY = (EARLY_A ? LV : 0) + (EARLY_B ? LB : 0), NLATE = LV + LB - NEARLY;
        static_assert(NLATE <= (TV == TJ ? 2 : 4) * NM, "schedule");
        // the x-th early load (A's first where both operands are early), the x-th late load
        auto early = [&](auto x_) {
            constexpr int x = decltype(x_)::value;
            if constexpr (EARLY_A && x < LV) loadA(x_);
            else loadB(std::integral_constant<int, x - (EARLY_A ? LV : 0)>{});
        };
        auto late = [&](auto x_) {
            constexpr int x = decltype(x_)::value;
            if constexpr (!EARLY_A && x < LV) loadA(x_);
            else loadB(std::integral_constant<int, x - (!EARLY_A ? LV : 0)>{});
        };
        // One k-step of 16 from operand set `use`: NM matrix instructions, and between them the LDS reads of set
        // `use ^ 1` (k-step rk of the stage that ra/rb point into) and the direct loads [E0, E1) of the early
        // ones or [L0, L1) of the late ones, evenly.
        auto substep = [&](auto use_, auto rd_, auto rk_, auto e0_, auto e1_, auto l0_, auto l1_) {
            constexpr int use = decltype(use_)::value, rk = decltype(rk_)::value;
            constexpr bool RD = decltype(rd_)::value;
            constexpr int E0 = decltype(e0_)::value, E1 = decltype(e1_)::value, L0 = decltype(l0_)::value, L1 = decltype(l1_)::value;
            static_for<0, NM>([&](auto n_) {
                constexpr int n = decltype(n_)::value;
                // block (i, j): weight rows i (the instruction's first operand, so the result's rows), activation rows j
                constexpr int i = n / TV, j = (i & 1) ? TV - 1 - n % TV : n % TV;
                quad_mfma(acc[i][j], fb[use][i], fa[use][j]);
                constexpr int R0 = NM >= NR ? (n < NR ? n : NR) : n * NR / NM, R1 = NM >= NR ? (n < NR ? n + 1 : NR) : (n + 1) * NR / NM;
                static_for<R0, R1>([&](auto r_) {
                    constexpr int r = decltype(r_)::value;
                    if constexpr (RD && r < TV) quad_read<r * ST * 4096>(fa[use ^ 1][r], ra[rk]);
                    if constexpr (RD && r >= TV) quad_read<(r - TV) * 4096>(fb[use ^ 1][r - TV], rb[rk]);
                });
                static_for<E0 + n * (E1 - E0) / NM, E0 + (n + 1) * (E1 - E0) / NM>(early);
                static_for<L0 + n * (L1 - L0) / NM, L0 + (n + 1) * (L1 - L0) / NM>(late);
            });
            if constexpr (RD) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        };
        using T = std::true_type;
        using F = std::false_type;
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I3 = std::integral_constant<int, 3>;
        // One k-tile from the stages in use.  Not LAST: before its last k-step every wave waits for its own
        // loads of the next k-tile (the early ones of the one after may be on their way) and for the others at
        // a barrier, which also says that all have read these stages; then it reads the next k-tile's first
        // operands.  LOADS: it asks for the k-tile two on, the early loads before the barrier, the late ones after.
        auto step = [&](auto loads_, auto last_) {
            constexpr bool LOADS = decltype(loads_)::value, LAST = decltype(last_)::value;
            constexpr int NE = LOADS ? NEARLY : 0, NL = LOADS ? NLATE : 0;
            using Z = std::integral_constant<int, 0>;
            substep(I0{}, T{}, I1{}, Z{}, std::integral_constant<int, NE / 3>{}, Z{}, Z{});
            substep(I1{}, T{}, I2{}, std::integral_constant<int, NE / 3>{}, std::integral_constant<int, 2 * NE / 3>{}, Z{}, Z{});
            substep(I0{}, T{}, I3{}, std::integral_constant<int, 2 * NE / 3>{}, std::integral_constant<int, NE>{}, Z{}, Z{});
            if constexpr (LAST) {
                substep(I1{}, F{}, I0{}, Z{}, Z{}, Z{}, Z{});
            } else {
                quad_wait_loads<NE>();
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                const unsigned da = curA == NSA - 1 ? (unsigned)(-(NSA - 1) * SA) : (unsigned)SA;
                const unsigned db = curB == NSB - 1 ? (unsigned)(-(NSB - 1) * SB) : (unsigned)SB;
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {                       // reads: the next stages
                    ra[kk] += da;
                    rb[kk] += db;
                }
                curA = curA == NSA - 1 ? 0 : curA + 1;
                curB = curB == NSB - 1 ? 0 : curB + 1;
                substep(I1{}, T{}, I0{}, Z{}, Z{}, Z{}, std::integral_constant<int, NL>{});
                if constexpr (LOADS) next_tile();
            }
        };

        static_for<0, LV>(loadA);                                      // the first two k-tiles
        static_for<0, LB>(loadB);
        next_tile();
        if (nk > 1) {
            static_for<0, LV>(loadA);
            static_for<0, LB>(loadB);
            next_tile();
            quad_wait_loads<LV + LB>();
        } else {
            quad_wait_loads<0>();
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        static_for<0, TV>([&](auto n_) {
            constexpr int n = decltype(n_)::value;
            quad_read<n * ST * 4096>(fa[0][n], ra[0]);
        });
        static_for<0, TI>([&](auto n_) {
            constexpr int n = decltype(n_)::value;
            quad_read<n * 4096>(fb[0][n], rb[0]);
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        // Statements that name the accumulators: what the compiler wrote into one (the zeroes) is written before
        // its statement, and a matrix instruction must not read a register in the states right after its write.
        static_for<0, TI * TJ>([&](auto n_) { quad_touch(acc[decltype(n_)::value / TJ][decltype(n_)::value % TJ]); });
        int t = 0;
        for (; t + 2 < nk; ++t) step(T{}, F{});
        for (; t + 1 < nk; ++t) step(F{}, F{});
        step(F{}, T{});
    };
    int blocks = (m_end - m0 + 32 * WVM - 1) / (32 * WVM);             // of 32 rows a wave
    if constexpr (!GROUPED) {
        if (gr.whole) blocks = TJ;
    }
    if (ST == 1 || blocks >= TJ) run(std::integral_constant<int, TJ>{});
    else if (TJ > 3 && blocks == 3) run(std::integral_constant<int, (TJ > 3 ? 3 : 1)>{});
    else if (TJ > 2 && blocks == 2) run(std::integral_constant<int, (TJ > 2 ? 2 : 1)>{});
    else run(std::integral_constant<int, 1>{});
    // the last matrix instructions' results are not in their registers yet; the epilogue's reads of an
    // accumulator stay behind the statement that names it
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    static_for<0, TI * TJ>([&](auto n_) { quad_touch(acc[decltype(n_)::value / TJ][decltype(n_)::value % TJ]); });
    if (MODE != OUT_F32_ACC) {                                         // (which leaves LDS alone)
        __builtin_amdgcn_s_barrier();                                  // every wave has read its last operands
        asm volatile("" ::: "memory");
    }
    if constexpr (!RUNS) {
        break;
    } else {
        static_for<0, TI * TJ>([&](auto n_) {
            constexpr int i = decltype(n_)::value / TJ, j = decltype(n_)::value % TJ;
            sum[i][j] += acc[i][j];
            acc[i][j] = f32x16(0.f);
            quad_touch(acc[i][j]);                                     // block by block: no second copy of them all
        });
        if (!rest) break;
        nk = rest < kt_per_part ? rest : kt_per_part;
        rest -= nk;
    }
    }
    unsigned char* const strip = st + wave * QuadStrip<TI, MODE>::BYTES;
    if constexpr (RUNS) quad_epilogue<TI, TJ, ST, MODE, GROUPED>(sum, C, m_end, N, ldc, m0 + wm, n0 + wn, lane, gr, strip);
    else quad_epilogue<TI, TJ, ST, MODE, GROUPED>(acc, C, m_end, N, ldc, m0 + wm, n0 + wn, lane, gr, strip);
    };

    if constexpr (!GROUPED) {
        const int total = tiles_m * tiles_n;
        int pid = blockIdx.x;
        const int per = total / 8, xcd = pid % 8, idx = pid / 8;
        if (pid < per * 8) pid = xcd * per + idx;
        const int grp = pid / (8 * tiles_m), in = pid - grp * 8 * tiles_m;
        int gn = tiles_n - grp * 8;
        if (gn > 8) gn = 8;
        const int tile_n = grp * 8 + in % gn, tile_m = in / gn;
        if constexpr (KIND == QUAD_BRANCHES) {                         // (no tile lies across two branches)
            const int n0 = tile_n * BN;
            if (n0 >= gr.gap_at) C = (float*)C + gr.gap;
            tile(A + (size_t)(n0 / gr.per) * gr.a_step, W, tile_m * BM, n0, M);
        } else {
            tile(A, W, tile_m * BM, tile_n * BN, M);
        }
    } else {
        // Expert by expert, column of tiles by column, an expert's row tiles of the same weights in turn; eight runs of as many tiles, one to an
        // XCD.  (Runs of columns of about equal cost, by what a tile of few rows costs beside a whole one, left some XCDs a round more than the
        // others: 32 experts of 1,792 by 4,096, 450 rows on average, gated 485 us against 446; 8 experts of 2,048 by 1,024, 400 rows, 73 against 43.)
        // this lane's expert of a block of 64: its pairs, its tiles of one column and those before them in the block
        struct Lane { int a, b, nt, nt0; };
        auto lane_of = [&](int e0) {
            Lane v;
            const int e = e0 + lane;
            v.a = e < gr.experts ? gr.first[e] : 0;
            v.b = e < gr.experts ? gr.first[e + 1] : 0;
            v.nt = (v.b - v.a + BM - 1) / BM;
            int sum = v.nt;                                            // of this lane and all before
            sum += __builtin_amdgcn_update_dpp(0, sum, 0x111, 0xf, 0xf, false);        // row_shr 1, 2, 4, 8
            sum += __builtin_amdgcn_update_dpp(0, sum, 0x112, 0xf, 0xf, false);
            sum += __builtin_amdgcn_update_dpp(0, sum, 0x114, 0xf, 0xf, false);
            sum += __builtin_amdgcn_update_dpp(0, sum, 0x118, 0xf, 0xf, false);
            sum += __builtin_amdgcn_update_dpp(0, sum, 0x142, 0xa, 0xf, false);        // row_bcast 15, 31
            sum += __builtin_amdgcn_update_dpp(0, sum, 0x143, 0xc, 0xf, false);
            v.nt0 = sum - v.nt;
            return v;
        };
        auto tiles_of = [](const Lane& v) { return __builtin_amdgcn_readlane(v.nt0 + v.nt, 63); };
        Lane v = lane_of(0);
        long long total = tiles_of(v);
        for (int e0 = 64; e0 < gr.experts; e0 += 64) total += tiles_of(lane_of(e0));
        total *= tiles_n;
        const int xcd = blockIdx.x % 8, job = (int)(total * xcd / 8) + (int)(blockIdx.x / 8);
        if (job >= (int)(total * (xcd + 1) / 8)) return;               // the grid is a bound
        int e = 0, p0 = 0, end = 0, nt = 1, before = 0;
        for (int e0 = 0, nt0 = 0; e0 < gr.experts; e0 += 64) {
            if (e0) v = lane_of(e0);
            const unsigned long long here = __ballot((nt0 + v.nt0) * tiles_n <= job && job < (nt0 + v.nt0 + v.nt) * tiles_n);
            if (here) {
                const int l = __ffsll(here) - 1;
                e = e0 + l;
                p0 = __builtin_amdgcn_readlane(v.a, l);
                end = __builtin_amdgcn_readlane(v.b, l);
                nt = __builtin_amdgcn_readlane(v.nt, l);
                before = (nt0 + __builtin_amdgcn_readlane(v.nt0, l)) * tiles_n;
                break;
            }
            nt0 += tiles_of(v);
        }
        const int in = job - before;
        tile(A, W + (size_t)e * N * K, p0 + in % nt * BM, in / nt * BN, end);
    }
}

static int launch_split_sum(const float* scratch, int parts, void* C, int M, int N, size_t ldc, int mode, hipStream_t s);

// What the quad tiles ask of a product beyond K % 64 == 0 and aligned rows: the loads reach a row by a
// 32-bit byte offset from the matrix's first element, and the epilogue stores 16 bytes at a time.
static bool quad_takes(const void* C, int M, int N, int K, size_t lda, size_t ldc) {
    return (unsigned long long)M * lda * 2 < (1ull << 32) && ((unsigned long long)N + 16) * K * 2 < (1ull << 32) &&
           ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
}

// parts > 1: the k-tiles are cut into runs of an even number of k-tiles, every (tile, run) workgroup writes
// its float sums to a matrix of its own in `scratch`, and gemm_split_sum_kernel adds the runs in run order
// and applies the epilogue.
#ifndef QUAD12
#define QUAD12 2, 3
#endif
#ifndef QUAD13
#define QUAD13 3, 3
#endif
#ifndef QUAD14
#define QUAD14 2, 3
#endif
template <int BM, int BN, int NSA, int NSB, int WVM = 2>
static int launch_tile_quad(const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc,
                            int mode, hipStream_t s, int wl, int parts = 1, float* scratch = nullptr, int* leave = nullptr) {
    const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
    const long long total = (long long)tm * tn;
    if (total > 0x7fffffffLL || !quad_takes(C, M, N, K, lda, ldc)) return BR_BAD_ARG;
    const int nk = K / DMA_BK;
    if (parts > 1) {
        if (N % 4 != 0 || (uintptr_t)scratch % 16 != 0) return BR_BAD_ARG;
        int kpp = (nk + parts - 1) / parts;
        kpp += kpp & 1;
        parts = (nk + kpp - 1) / kpp;                                 // no empty run
        dim3 grid((unsigned)total, (unsigned)parts);
        const QuadPlain whole = {total * parts <= br_device_cus()};
        gemm_tile_quad_kernel<BM, BN, NSA, NSB, WVM, OUT_F32><<<grid, 256, 0, s>>>(A, W, scratch, M, N, K, lda, (size_t)N, tm, tn, kpp,
                                                                        (size_t)M * N, wl, whole);
        int rc = br_check_launch();
        if (rc != BR_OK) return rc;
        if (leave) {                                                  // the runs' sums are the caller's
            *leave = parts;
            return rc;
        }
        return launch_split_sum(scratch, parts, C, M, N, ldc, mode, s);
    }
    if (leave) return BR_BAD_ARG;
    const QuadPlain whole = {total <= br_device_cus()};
    if (mode == OUT_BF16)
        gemm_tile_quad_kernel<BM, BN, NSA, NSB, WVM, OUT_BF16><<<(unsigned)total, 256, 0, s>>>(A, W, C, M, N, K, lda, ldc, tm, tn, nk, 0, wl, whole);
    else if (mode == OUT_F32)
        gemm_tile_quad_kernel<BM, BN, NSA, NSB, WVM, OUT_F32><<<(unsigned)total, 256, 0, s>>>(A, W, C, M, N, K, lda, ldc, tm, tn, nk, 0, wl, whole);
    else if (mode == OUT_F32_ACC)
        gemm_tile_quad_kernel<BM, BN, NSA, NSB, WVM, OUT_F32_ACC><<<(unsigned)total, 256, 0, s>>>(A, W, C, M, N, K, lda, ldc, tm, tn, nk, 0, wl, whole);
    else
        gemm_tile_quad_kernel<BM, BN, NSA, NSB, WVM, OUT_SWIGLU><<<(unsigned)total, 256, 0, s>>>(A, W, C, M, N, K, lda, ldc, tm, tn, nk, 0, wl, whole);
    return br_check_launch();
}

// Which quad tile (12: 256x256, 13: 128x256, 14: 256x192, 15: 256x224, whose 128 tile columns over 28,672
// weight rows make whole rounds where 112 of 256 do not) and how many runs of k-tiles: the least time by a
// count in microseconds.  A k-tile takes 1.50, 0.85, 1.20 and 1.39 us with every compute unit at work and 1.08,
// 0.80, 0.92 and 1.00 us with few (measured; in between, the cube of the share at work fits: at half the chip
// the tiles hardly feel each other yet); whole rounds of workgroups over the chip, then the rest of them,
// which after whole rounds take nearly what a whole round takes (2,048 x 28,672 by 896 tiles of 256x256,
// three and a half rounds: 390 us, the half round 1.41 us a k-tile); plus what a launch costs besides and,
// when split along k, the second launch and the traffic of the partial sums.  Returns the count.
static const double QUAD_FULL[4] = {1.50, 0.85, 1.20, 1.39}, QUAD_FEW[4] = {1.08, 0.80, 0.92, 1.00};
static double quad_count(int M, int N, int K, int mode, int cus, int k, int p) {       // tile 12 + k in p runs
    static const int bm[4] = {256, 128, 256, 256}, bn[4] = {256, 256, 192, 224};
    int kpp = (K / DMA_BK + p - 1) / p;
    kpp += kpp & 1;
    const long long units = (long long)((M + bm[k] - 1) / bm[k]) * ((N + bn[k] - 1) / bn[k]) * p, whole = units / cus;
    const double share = (double)(units % cus) / cus;
    const double rest = units % cus == 0 ? 0.0
                        : whole        ? QUAD_FULL[k] * (0.9 + 0.1 * share)
                                       : QUAD_FEW[k] + (QUAD_FULL[k] - QUAD_FEW[k]) * share * share * share;
    const double t = kpp * ((double)whole * QUAD_FULL[k] + rest) + (mode == OUT_BF16 ? 8.0 : 12.0);
    return p > 1 ? t + 5.0 + (double)p * M * N * 8.0 / 4e6 : t;
}
static double choose_quad(int M, int N, int K, int mode, int cus, size_t scratch_bytes, int* kernel, int* parts) {
    double best = 1e30;
    *kernel = 13;
    *parts = 1;
    for (int k = 0; k < 4; ++k) {
        for (int p = 1; p <= 16; p *= 2) {
            if (p > 1 && (p * 4 > K / DMA_BK || N % 4 != 0 || (size_t)p * M * N * sizeof(float) > scratch_bytes)) break;
            const double t = quad_count(M, N, K, mode, cus, k, p);
            if (t < best - 1e-9) { best = t; *kernel = 12 + k; *parts = p; }
        }
    }
    return best;
}

// Weight rows that the 256x256 tile covers in whole rounds of workgroups over the chip, where the count says that
// these rounds and the best tile for the rest (`kernel`, `parts`, chosen over N - n1 weight rows) take less than
// the best single tile over all rows (`single`); 0 where not.  n1 is a multiple of 256.
static int quad_whole_rounds(int M, int N, int K, int mode, int cus, size_t scratch_bytes, double single, int* kernel,
                             int* parts) {
    const int tm = (M + 255) / 256, nk = K / DMA_BK;
    const int cols = cus / tm;                                        // tile columns of one round
    if (cols < 1) return 0;
    const long long rounds = (long long)(N / 256) / cols, n1 = rounds * cols * 256;
    if (rounds < 1 || n1 >= N || (mode == OUT_SWIGLU && (N - n1) % 16 != 0)) return 0;
    const long long used = (long long)tm * cols;                      // workgroups of such a round
    const double share = (double)used / cus;
    const double per = used == cus ? QUAD_FULL[0] : QUAD_FEW[0] + (QUAD_FULL[0] - QUAD_FEW[0]) * share * share * share;
    int k2, p2;
    const double t = (double)rounds * nk * per + (mode == OUT_BF16 ? 8.0 : 12.0) +
                     choose_quad(M, (int)(N - n1), K, mode, cus, scratch_bytes, &k2, &p2);
    if (t >= 0.97 * single) return 0;
    *kernel = k2;
    *parts = p2;
    return (int)n1;
}

// parts > 1: the k-tiles are cut into `parts` runs, every (tile, run) workgroup writes its
// float sums to a matrix of its own in `scratch`, and gemm_split_sum_kernel adds the runs in
// run order and applies the epilogue (for products with too few tiles to fill the chip).
template <int BM, int BN, int WAVES_M, int WAVES_N, int S>
static int launch_tile_dma(const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc,
                           int mode, hipStream_t s, int parts = 1, float* scratch = nullptr, int wl = 0, int* leave = nullptr) {
    const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
    const long long total = (long long)tm * tn;
    if (total > 0x7fffffffLL) return BR_BAD_ARG;
    constexpr int NT = 64 * WAVES_M * WAVES_N;
    const int nk = K / DMA_BK;
    if (parts > 1) {
        const int kpp = (nk + parts - 1) / parts;
        parts = (nk + kpp - 1) / kpp;                                 // no empty run
        dim3 grid((unsigned)total, (unsigned)parts);
        gemm_tile_dma_kernel<BM, BN, WAVES_M, WAVES_N, S, OUT_F32><<<grid, NT, 0, s>>>(
            A, W, scratch, M, N, K, lda, (size_t)N, tm, tn, kpp, (size_t)M * N, wl);
        int rc = br_check_launch();
        if (rc != BR_OK) return rc;
        if (leave) {                                                  // the runs' sums are the caller's
            *leave = parts;
            return rc;
        }
        return launch_split_sum(scratch, parts, C, M, N, ldc, mode, s);
    }
    if (leave) return BR_BAD_ARG;
    if (mode == OUT_BF16)
        gemm_tile_dma_kernel<BM, BN, WAVES_M, WAVES_N, S, OUT_BF16><<<(unsigned)total, NT, 0, s>>>(A, W, C, M, N, K, lda, ldc, tm, tn, nk, 0, wl);
    else if (mode == OUT_F32)
        gemm_tile_dma_kernel<BM, BN, WAVES_M, WAVES_N, S, OUT_F32><<<(unsigned)total, NT, 0, s>>>(A, W, C, M, N, K, lda, ldc, tm, tn, nk, 0, wl);
    else if (mode == OUT_F32_ACC)
        gemm_tile_dma_kernel<BM, BN, WAVES_M, WAVES_N, S, OUT_F32_ACC><<<(unsigned)total, NT, 0, s>>>(A, W, C, M, N, K, lda, ldc, tm, tn, nk, 0, wl);
    else
        gemm_tile_dma_kernel<BM, BN, WAVES_M, WAVES_N, S, OUT_SWIGLU><<<(unsigned)total, NT, 0, s>>>(A, W, C, M, N, K, lda, ldc, tm, tn, nk, 0, wl);
    return br_check_launch();
}

// Which direct-to-LDS tile (5: 128x256, one workgroup per CU; 6: 128x128, two; 10: 256x192, one, two
// stages, not split) and how many runs of k-tiles for a product of more than 64 rows: the least time by
// a rough count in microseconds (rounds of workgroups over the chip times k-tiles times 1.0-1.7 us a
// k-tile, plus, when split, a launch and the traffic of the partial sums), runs of at least 4 k-tiles
// that fit the scratch memory.  The 256x192 tile is there for shapes that it covers in fewer rounds:
// 2,048 x 6,144 is 256 of them, one round, against 384 tiles of 128x256 (measured 103-118 against
// 129-134 us); with equal rounds it loses (two stages, 1.5 times the work a k-tile for 1.5 times the time).
static void choose_tile(int M, int N, int K, int mode, int cus, size_t scratch_bytes, int* kernel, int* parts) {
    const int nk = K / DMA_BK;
    double best = 1e30;
    *kernel = 5;
    *parts = 1;
    {
        const long long tiles = (long long)((M + 255) / 256) * ((N + 191) / 192);
        const double t = (double)((tiles + cus - 1) / cus) * nk * 1.72;
        if (tiles > cus / 2) { best = t; *kernel = 10; }             // with fewer tiles a split product fills the chip better
    }
    if (mode == OUT_SWIGLU) {
        // 256x256, SwiGLU epilogue only (the other epilogues run out of registers around its 128 accumulators a
        // wave): 8 % faster than 128x256 where its rounds fit (4,096 x 28,672: 920 against 1,000 us)
        const long long tiles = (long long)((M + 255) / 256) * ((N + 255) / 256);
        const double t = (double)((tiles + cus - 1) / cus) * nk * 2.1;
        if (tiles > cus / 2 && t < best - 1e-9) { best = t; *kernel = 11; }
    }
    for (int k = 5; k <= 6; ++k) {
        const long long tiles = (long long)((M + 127) / 128) * ((N + (k == 5 ? 255 : 127)) / (k == 5 ? 256 : 128));
        const long long slots = (long long)cus * (k == 5 ? 1 : 2);
        for (int p = 1; p <= 16; p *= 2) {
            if (p > 1 && (p * 4 > nk || (size_t)p * M * N * sizeof(float) > scratch_bytes)) break;
            const long long units = tiles * p, rounds = (units + slots - 1) / slots;
            const int kpp = (nk + p - 1) / p;
            const double per = k == 5 ? 1.14 : (units > cus ? 1.33 : 1.0);
            double t = (double)rounds * kpp * per;
            if (p > 1) t += 5.0 + (double)p * M * N * 8.0 / 4e6;
            if (t < best - 1e-9) { best = t; *kernel = k; *parts = p; }
        }
    }
}

// ----------------------------------------------------------------- gemm_skinny ------
// grid = ceil(N / (16 RB)); block = 64 NW.  Needs K % 8 == 0 and 16-byte aligned rows.
// Every wave keeps U chunks of 128 k in flight (the loads of all U are issued before the
// first product), which is what fills the memory pipeline; rows beyond N or M are read
// from the last valid row instead of being masked, and dropped at the store.
template <int MB, int RB, int U, int NW, int MODE>
__global__ __launch_bounds__(NW * 64) void gemm_skinny_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                              void* __restrict__ C, int M, int N, int K,
                                                              size_t lda, size_t ldc) {
    constexpr int ROWS = 16 * RB, COLS = 16 * MB;
    __shared__ float red[NW][ROWS][COLS + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * ROWS;

    f32x4 acc[RB][MB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;
    const bf16* wp[RB];
    const bf16* xp[MB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        int row = n0 + i * 16 + r16;
        if (row > N - 1) row = N - 1;
        wp[i] = W + (size_t)row * K + g * 8;
    }
#pragma unroll
    for (int j = 0; j < MB; ++j) {
        int row = j * 16 + r16;
        if (row > M - 1) row = M - 1;
        xp[j] = A + (size_t)row * lda + g * 8;
    }
    // lane (row r16, group g) holds k = chunk * 128 + s * 32 + g * 8 + [0, 8) for s = 0..3
    const int nfull = K / 128;
    int c = wave * U;
    for (; c + U <= nfull; c += NW * U) {
        bf16x8 fw[U][RB][4], fx[U][MB][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kb = (c + u) * 128;
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int s = 0; s < 4; ++s) fw[u][i][s] = *(const bf16x8*)(wp[i] + kb + s * 32);
#pragma unroll
            for (int j = 0; j < MB; ++j)
#pragma unroll
                for (int s = 0; s < 4; ++s) fx[u][j][s] = *(const bf16x8*)(xp[j] + kb + s * 32);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < RB; ++i)
#pragma unroll
                    for (int j = 0; j < MB; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[u][i][s], fx[u][j][s], acc[i][j], 0, 0, 0);
    }
    // this wave's leftover chunks (fewer than U, or the partial last chunk), guarded along k
    const int nch = (K + 127) / 128;
    for (int u = 0; u < U; ++u) {
        const int cc = c + u;
        if (cc >= nch) break;
        const int kb = cc * 128;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const bool in = kb + s * 32 + g * 8 + 8 <= K;
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                const bf16x8 a = in ? *(const bf16x8*)(wp[i] + kb + s * 32) : zero8();
#pragma unroll
                for (int j = 0; j < MB; ++j) {
                    const bf16x8 b = in ? *(const bf16x8*)(xp[j] + kb + s * 32) : zero8();
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[i][j], 0, 0, 0);
                }
            }
        }
    }
    // acc[i][j][r]: weight row = 16 i + 4 (lane / 16) + r, batch row = 16 j + lane % 16
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][i * 16 + 4 * g + r][j * 16 + r16] = acc[i][j][r];
    __syncthreads();
    if (MODE == OUT_SWIGLU) {
        for (int e = tid; e < (ROWS / 2) * COLS; e += NW * 64) {
            const int m = e / (ROWS / 2), jl = e - m * (ROWS / 2);
            const int gl = (jl >> 3) * 16 + (jl & 7);            // gate row in the tile; its up row is 8 on
            if (m < M && n0 + gl + 8 < N) {
                float gv = 0.f, uv = 0.f;
#pragma unroll
                for (int w = 0; w < NW; ++w) { gv += red[w][gl][m]; uv += red[w][gl + 8][m]; }
                ((bf16*)C)[(size_t)m * ldc + n0 / 2 + jl] = (bf16)silu_mul(gv, uv);
            }
        }
        return;
    }
    for (int e = tid; e < ROWS * COLS; e += NW * 64) {
        const int m = e / ROWS, nl = e - m * ROWS;   // consecutive threads: consecutive weight rows
        const int n = n0 + nl;
        if (m < M && n < N) {
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) v += red[w][nl][m];     // in wave order, always
            store_out<MODE>(C, (size_t)m * ldc + n, v);
        }
    }
}

template <int MB, int RB, int U, int NW>
static int launch_skinny(const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc,
                         int mode, hipStream_t s) {
    const unsigned grid = (unsigned)((N + 16 * RB - 1) / (16 * RB));
    if (mode == OUT_BF16)
        gemm_skinny_kernel<MB, RB, U, NW, OUT_BF16><<<grid, NW * 64, 0, s>>>(A, W, C, M, N, K, lda, ldc);
    else if (mode == OUT_SWIGLU)
        gemm_skinny_kernel<MB, RB, U, NW, OUT_SWIGLU><<<grid, NW * 64, 0, s>>>(A, W, C, M, N, K, lda, ldc);
    else if (mode == OUT_F32)
        gemm_skinny_kernel<MB, RB, U, NW, OUT_F32><<<grid, NW * 64, 0, s>>>(A, W, C, M, N, K, lda, ldc);
    else
        gemm_skinny_kernel<MB, RB, U, NW, OUT_F32_ACC><<<grid, NW * 64, 0, s>>>(A, W, C, M, N, K, lda, ldc);
    return br_check_launch();
}

// ------------------------------------------------------------- gemm_narrow ----------
// More than 16 rows against at most 64 weight rows (a router's scores, the narrow half of a low-rank pair).  The tiles above
// give such a product one workgroup to 128 rows, 15 compute units for 1,801 rows that each walk all of K.  Here a workgroup takes 16 rows
// of A and 16 NB weight rows, its eight waves U chunks of 128 k each at a time straight into operands (with K = 4,096 all of a
// wave's loads are under way at once), and the waves' sums meet in LDS in wave order.  The weights come from the L2, once per
// workgroup.  grid (ceil(M / 16), ceil(N / (16 NB))).  Needs K % 8 == 0 and 16-byte aligned rows; rows beyond M or N are
// read from the last one and dropped at the store.
// 32 weight rows of 4,096 (us, launch to launch): 64 rows 10.2 -> 8.7, 300 rows 14.3 -> 8.7, 1,801 rows 39.0 -> 9.2, 7,000 rows
// 39.6 -> 23.2; the error against 64 bits 1.0e-7 of the result (before 1.0e-7 to 4.0e-7).  Bound by the latency of one
// round of loads and the sum of the waves; each further round of workgroups costs the same again.
template <int NB, int U, int MODE>
__global__ __launch_bounds__(512) void gemm_narrow_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W, void* __restrict__ C,
                                                          int M, int N, int K, size_t lda, size_t ldc) {
    constexpr int NW = 8, COLS = 16 * NB;
    __shared__ float red[NW][16][COLS + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int m0 = blockIdx.x * 16, n0 = blockIdx.y * COLS;
    f32x4 acc[2][NB];                                         // two chains each: shorter sums round less
    const bf16* wp[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        acc[0][j] = acc[1][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        wp[j] = W + (size_t)min(n0 + 16 * j + r16, N - 1) * K + g * 8;
    }
    const bf16* ap = A + (size_t)min(m0 + r16, M - 1) * lda + g * 8;
    // lane (row r16, group g) holds k = chunk * 128 + s * 32 + g * 8 + [0, 8) for s = 0..3
    const int nfull = K / 128, nch = (K + 127) / 128;
    int c = wave * U;
    for (; c + U <= nfull; c += NW * U) {
        bf16x8 fa[U][4], fw[U][NB][4];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int kb = (c + u) * 128 + s * 32;
                fa[u][s] = *(const bf16x8*)(ap + kb);
#pragma unroll
                for (int j = 0; j < NB; ++j) fw[u][j][s] = *(const bf16x8*)(wp[j] + kb);
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int j = 0; j < NB; ++j) acc[s & 1][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[u][s], fw[u][j][s], acc[s & 1][j], 0, 0, 0);
    }
    // this wave's leftover chunks (fewer than U, or the partial last chunk), guarded along k
    for (int u = 0; u < U && c + u < nch; ++u) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int kb = (c + u) * 128 + s * 32;
            const bool in = kb + g * 8 + 8 <= K;
            const bf16x8 a = in ? *(const bf16x8*)(ap + kb) : zero8();
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                const bf16x8 b = in ? *(const bf16x8*)(wp[j] + kb) : zero8();
                acc[s & 1][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[s & 1][j], 0, 0, 0);
            }
        }
    }
    // acc[..][j][r]: row 4 g + r, weight row 16 j + r16
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wave][4 * g + r][16 * j + r16] = acc[0][j][r] + acc[1][j][r];
    __syncthreads();
    for (int e = tid; e < 16 * COLS; e += NW * 64) {
        const int m = e / COLS, n = e % COLS;
        if (m0 + m < M && n0 + n < N) {
            float v[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w) v[w] = red[w][m][n];
#pragma unroll
            for (int h = 1; h < NW; h *= 2)
#pragma unroll
                for (int w = 0; w < NW; w += 2 * h) v[w] += v[w + h];
            store_out<MODE>(C, (size_t)(m0 + m) * ldc + n0 + n, v[0]);
        }
    }
}

template <int NB, int U>
static int launch_narrow(const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc, int mode, hipStream_t s) {
    const dim3 grid((unsigned)((M + 15) / 16), (unsigned)((N + 16 * NB - 1) / (16 * NB)));
    if (mode == OUT_BF16) gemm_narrow_kernel<NB, U, OUT_BF16><<<grid, 512, 0, s>>>(A, W, C, M, N, K, lda, ldc);
    else if (mode == OUT_F32) gemm_narrow_kernel<NB, U, OUT_F32><<<grid, 512, 0, s>>>(A, W, C, M, N, K, lda, ldc);
    else gemm_narrow_kernel<NB, U, OUT_F32_ACC><<<grid, 512, 0, s>>>(A, W, C, M, N, K, lda, ldc);
    return br_check_launch();
}

// The longest K that the narrow kernel takes where scratch lets the kernels it stands for cut the product into runs along k (without, they
// are at least 1.1 times as long at every K).  It brings all of K to each of its few workgroups, 2 us and 1.65 for every 1,000 of K (one block
// of 16 weight rows), and the runs spread K over the chip.  Runs against it, us, 32 weight rows: 32 rows, K = 3,072 / 3,584 / 4,096 /
// 8,192 / 14,336: 8.1 / 8.0 / 8.2 / 10.0 / 12.3 against 7.0 / 7.8 / 8.6 / 15.6 / 25.7; 64 rows, 4,096 / 5,120 / 8,192: 9.8 / 10.3 /
// 11.9 against 8.8 / 10.5 / 15.7; 128 rows 12.8 / 13.8 / 15.9 and, at 7,168, 15.5 against 8.9 / 10.6 / 15.9 and 14.1, 1,000 rows 14.9 / 15.6 / 17.2 and 16.5 against
// 9.0 / 10.7 / 16.0 and 14.2.
// Above 1,024 rows (no caller here brings scratch then) it is ahead up to 3,072 rows of K = 3,072 (64 weight rows, 3,000 rows: 1.1 times, 5,000: 0.8).
static int narrow_longest(int M, int N, int K, size_t room) {
    if (room < (size_t)8 * M * N * sizeof(float) || (M > 64 && K % DMA_BK)) return 0x7fffffff;
    return M <= 32 ? 3584 : M <= 64 ? 4608 : M <= 1024 ? 7168 : M <= 3072 ? 3072 : 0;
}

// How many blocks of 16 weight rows a workgroup takes (1, 2 or 4), or 0 where the tiles are as fast: rounds of workgroups
// over the compute units times what a round takes, 7, 10.5 and 17.5 us with K = 4,096 and nearly in proportion otherwise (one block: 2.4,
// 5.4, 15.6 and 25.8 us at K = 256, 2,048, 8,192 and 14,336), against the 37 of the tiles' single round, which go with K in the same way
// (9, 23, 71 and 121; measured, us; K = 4,096, 64 weight rows: 1,801 rows 17 / 13 / 20 by 1 / 2 / 4 blocks and 39 by the
// tiles, 3,000 rows 23 / 23 / 20 and 39, 5,000 rows 37 / 34 / 37 and 39, 7,000 rows 51 / 44 / 37 and 40).
static int narrow_blocks(int M, int N, int K, int mode, int cus, size_t room) {
    if (M <= 16 || N > 64 || K < 256 || mode == OUT_SWIGLU || cus <= 0 || K > narrow_longest(M, N, K, room)) return 0;
    static const double round_us[3] = {7.0, 10.5, 17.5};
    int best = 0;
    double least = 32.0;
    for (int i = 0; i < 3 && (i == 0 || 16 << (i - 1) < N); ++i) {
        const long long units = (long long)((M + 15) / 16) * ((N + (16 << i) - 1) / (16 << i));
        const double t = (double)((units + cus - 1) / cus) * round_us[i];
        if (t < least) { least = t; best = 1 << i; }
    }
    return best;
}

static int launch_narrow_blocks(int blocks, const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc, int mode,
                                hipStream_t s) {
    // a wave's share of K in one go where it has four chunks, two where it has fewer
    if (blocks == 1) return K >= 4096 ? launch_narrow<1, 4>(A, W, C, M, N, K, lda, ldc, mode, s) : launch_narrow<1, 2>(A, W, C, M, N, K, lda, ldc, mode, s);
    if (blocks == 2) return K >= 4096 ? launch_narrow<2, 4>(A, W, C, M, N, K, lda, ldc, mode, s) : launch_narrow<2, 2>(A, W, C, M, N, K, lda, ldc, mode, s);
    return launch_narrow<4, 2>(A, W, C, M, N, K, lda, ldc, mode, s);
}

// ------------------------------------------------------------- gemm_skinny_lds ------
// 16 < M <= 64: the activations of a 512-wide k-slab are staged in LDS once per workgroup
// with direct global-to-LDS loads (one 1 KB row per wave-load, no registers), because at
// these M the activation fragments, not the weights, dominate the load instructions.
// A row's 16-byte columns are stored XOR-swizzled by the row number, so that the 16 rows
// an operand read touches fall into different banks; the swizzle is applied by choosing
// which global column each lane fetches.  Weights stream from memory into the operands
// as in gemm_skinny; the 4 waves split the slab's k and are added in wave order.
#define SLAB_K 512
template <int MB, int RB, int MODE>
__global__ __launch_bounds__(256) void gemm_skinny_lds_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                              void* __restrict__ C_, int M, int N, int K,
                                                              size_t lda, size_t ldc, int slabs_per_part,
                                                              size_t part_stride) {
    constexpr int ROWS = 16 * RB, COLS = 16 * MB;
    constexpr int SLAB_BYTES = COLS * SLAB_K * 2;
    constexpr int RED_BYTES = 4 * ROWS * (COLS + 1) * 4;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[SLAB_BYTES > RED_BYTES ? SLAB_BYTES : RED_BYTES];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * ROWS;
    f32x4 acc[RB][MB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;
    const bf16* wp[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        int row = n0 + i * 16 + r16;
        if (row > N - 1) row = N - 1;
        wp[i] = W + (size_t)row * K + wave * 128 + g * 8;
    }
    // blockIdx.y: which run of k-slabs this workgroup sums (one run, or the parts of a split
    // product, each into its own float matrix `part_stride` elements on)
    const int nslab = (K + SLAB_K - 1) / SLAB_K;
    const int sl0 = blockIdx.y * slabs_per_part;
    const int sl1 = sl0 + slabs_per_part < nslab ? sl0 + slabs_per_part : nslab;
    void* C = MODE == OUT_F32 ? (void*)((float*)C_ + blockIdx.y * part_stride) : C_;
    for (int sl = sl0; sl < sl1; ++sl) {
        const int k0 = sl * SLAB_K;
        bf16x8 fw[RB][4];                                  // this wave's weight fragments of the slab
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int k = k0 + wave * 128 + s * 32 + g * 8;
                fw[i][s] = (k + 8 <= K) ? *(const bf16x8*)(wp[i] + k0 + s * 32) : zero8();
            }
#pragma unroll
        for (int rr = 0; rr < COLS / 4; ++rr) {
            const int row = rr * 4 + wave;                 // slab row = batch row; lane l fetches column l ^ (row & 15)
            int grow = row;
            if (grow > M - 1) grow = M - 1;
            int kk = k0 + ((lane ^ (row & 15)) * 8);
            if (kk + 8 > K) kk = 0;                        // never multiplied: the weight fragment there is zero
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(A + (size_t)grow * lda + kk),
                                             (__attribute__((address_space(3))) void*)(smem + row * 1024), 16, 0, 0);
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int c = wave * 16 + s * 4 + g;
#pragma unroll
            for (int j = 0; j < MB; ++j) {
                const bf16x8 fx = *(const bf16x8*)(smem + (j * 16 + r16) * 1024 + ((c ^ r16) * 16));
#pragma unroll
                for (int i = 0; i < RB; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[i][s], fx, acc[i][j], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    float (*red)[ROWS][COLS + 1] = (float (*)[ROWS][COLS + 1])smem;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][i * 16 + 4 * g + r][j * 16 + r16] = acc[i][j][r];
    __syncthreads();
    if (MODE == OUT_SWIGLU) {
        for (int e = tid; e < (ROWS / 2) * COLS; e += 256) {
            const int m = e / (ROWS / 2), jl = e - m * (ROWS / 2);
            const int gl = (jl >> 3) * 16 + (jl & 7);
            if (m < M && n0 + gl + 8 < N) {
                float gv = 0.f, uv = 0.f;
#pragma unroll
                for (int w = 0; w < 4; ++w) { gv += red[w][gl][m]; uv += red[w][gl + 8][m]; }
                ((bf16*)C)[(size_t)m * ldc + n0 / 2 + jl] = (bf16)silu_mul(gv, uv);
            }
        }
        return;
    }
    for (int e = tid; e < ROWS * COLS; e += 256) {
        const int m = e / ROWS, nl = e - m * ROWS;
        const int n = n0 + nl;
        if (m < M && n < N) {
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) v += red[w][nl][m];
            store_out<MODE>(C, (size_t)m * ldc + n, v);
        }
    }
}

template <int MB, int RB>
static int launch_skinny_lds(const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc,
                             int mode, hipStream_t s) {
    const unsigned grid = (unsigned)((N + 16 * RB - 1) / (16 * RB));
    const int nslab = (K + SLAB_K - 1) / SLAB_K;
    if (mode == OUT_BF16) gemm_skinny_lds_kernel<MB, RB, OUT_BF16><<<grid, 256, 0, s>>>(A, W, C, M, N, K, lda, ldc, nslab, 0);
    else if (mode == OUT_F32) gemm_skinny_lds_kernel<MB, RB, OUT_F32><<<grid, 256, 0, s>>>(A, W, C, M, N, K, lda, ldc, nslab, 0);
    else if (mode == OUT_F32_ACC) gemm_skinny_lds_kernel<MB, RB, OUT_F32_ACC><<<grid, 256, 0, s>>>(A, W, C, M, N, K, lda, ldc, nslab, 0);
    else gemm_skinny_lds_kernel<MB, RB, OUT_SWIGLU><<<grid, 256, 0, s>>>(A, W, C, M, N, K, lda, ldc, nslab, 0);
    return br_check_launch();
}

// ---------------------------------------------------------------- split product ------
// 16 < M <= 64 and so few weight rows that 64-row workgroups would leave most of the chip
// idle (N = 4096: 64 of them): the k-slabs are cut into `parts` runs, every (tile, run)
// workgroup writes its sums to a float matrix of its own in `scratch`, and a second kernel
// adds the runs in run order and applies the epilogue.  Nothing is added atomically: the
// result does not depend on which workgroup finishes first.
// VEC neighbouring results a thread, 4 where rows of 16 bytes (8 of bf16) allow, with eight runs asked for at a time.  A thread a result,
// one run after the other, took (with the product, us): 6,144 x 4,096 by 150 and 300 rows 29.4 and 40.0 (now 28.5 and 38.2), 4,096 x 14,336
// added into float rows by 700 and 1,000 rows 102.6 and 126.5 (98.7 and 122.3), with the next norm prepared by 24 rows 27.5 (26.4).
template <int VEC>
__device__ __forceinline__ void add_runs(const float* __restrict__ at, int parts, size_t part_stride, float* v) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) v[e] = 0.f;
    for (int p0 = 0; p0 < parts; p0 += 8) {
        float t[8][VEC];
#pragma unroll
        for (int p = 0; p < 8; ++p)
            if (p0 + p < parts) ew_load<float, VEC>(at + (size_t)(p0 + p) * part_stride, t[p]);
#pragma unroll
        for (int p = 0; p < 8; ++p)
            if (p0 + p < parts)
#pragma unroll
                for (int e = 0; e < VEC; ++e) v[e] += t[p][e];
    }
}
template <int MODE, int VEC>
__global__ __launch_bounds__(256) void gemm_split_sum_kernel(const float* __restrict__ part, int parts, size_t part_stride, void* __restrict__ C,
                                                             int M, int N, size_t ldc) {
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * VEC;
    const size_t width = MODE == OUT_SWIGLU ? (size_t)N / 2 : (size_t)N;
    if (i >= (size_t)M * width) return;
    const size_t m = i / width, n = i - m * width;
    float v[VEC];
    if (MODE == OUT_SWIGLU) {
        // output n of a row: gate column 16 (n / 8) + n % 8, its up value 8 columns on
        const float* at = part + m * N + (n >> 3) * 16 + (n & 7);
        float u[VEC];
        add_runs<VEC>(at, parts, part_stride, v);
        add_runs<VEC>(at + 8, parts, part_stride, u);
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] = silu_mul(v[e], u[e]);
        ew_store<bf16, VEC>((bf16*)C + m * ldc + n, v);
        return;
    }
    add_runs<VEC>(part + i, parts, part_stride, v);
    if (MODE == OUT_BF16) ew_store<bf16, VEC>((bf16*)C + m * ldc + n, v);
    else {
        float* to = (float*)C + m * ldc + n;
        if (MODE == OUT_F32_ACC) {
            float c[VEC];
            ew_load<float, VEC>(to, c);
#pragma unroll
            for (int e = 0; e < VEC; ++e) v[e] = c[e] + v[e];
        }
        ew_store<float, VEC>(to, v);
    }
}

// The sum of the runs added into the residual rows C, with the next RMS norm prepared as by
// gemm_stream's NORM = 1 form: a wave takes 256 consecutive columns of one row, four a lane (N in
// steps of 256), writes h = C + sum back, bf16(h * gain) to xg, and the sum of its 256
// squares to ssq[(column / 256) * SSQ_LD + row].
template <int VEC>
__global__ __launch_bounds__(256) void gemm_split_sum_prep_kernel(const float* __restrict__ part, int parts,
                                                                  size_t part_stride, float* __restrict__ C, int N,
                                                                  size_t ldc, const float* __restrict__ gain,
                                                                  bf16* __restrict__ xg, size_t ldx,
                                                                  float* __restrict__ ssq, size_t segments) {
    const size_t seg = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (seg >= segments) return;
    const int lane = threadIdx.x & 63;
    const size_t m = seg * 256 / N, n0 = seg * 256 - m * N;
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < 4 / VEC; ++j) {                  // VEC 1: a lane's four columns lie 64 apart
        const size_t n = n0 + j * 64 + (size_t)lane * VEC;
        float v[VEC], c[VEC], g[VEC], o[VEC];
        ew_load<float, VEC>(C + m * ldc + n, c);
        ew_load<float, VEC>(gain + n, g);
        add_runs<VEC>(part + m * N + n, parts, part_stride, v);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            v[e] = c[e] + v[e];
            o[e] = v[e] * g[e];
            q += v[e] * v[e];
        }
        ew_store<float, VEC>(C + m * ldc + n, v);
        ew_store<bf16, VEC>(xg + m * ldx + n, o);
    }
    q = wave_sum(q);
    if (lane == 0) ssq[(n0 / 256) * SSQ_LD + m] = q;
}

// The sum of the runs added into the residual rows C, and the RMS norm that reads them next in the same pass: h = bf16(C gain /
// rms(C)).  A workgroup takes a row and keeps it in registers, 4 NV columns a thread; the runs are asked for eight at a time and added in
// run order.  The sum and the norm are two launches otherwise, each reading and writing the rows (us, 4,096 columns): 100 rows in 8 runs
// 5.9 + 4.1 -> 5.8, 400 rows in 4 runs 10.6 + 5.0 -> 8.6, 700 rows 14.4 + 5.3 -> 11.5.
template <int NV>
__global__ __launch_bounds__(1024) void gemm_split_sum_norm_kernel(const float* __restrict__ part, int parts, size_t part_stride,
                                                                   float* __restrict__ C, int N, size_t ldc, const float* __restrict__ gain,
                                                                   float eps, bf16* __restrict__ h, size_t ldh) {
    __shared__ float scratch[16];
    const size_t m = blockIdx.x;
    const int nv = N >> 2;
    const float* pr = part + m * N;
    f32x4* cr = (f32x4*)(C + m * ldc);
    f32x4 v[NV], c[NV], g[NV];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int i = threadIdx.x + blockDim.x * j;
        v[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (i < nv) { c[j] = cr[i]; g[j] = ((const f32x4*)gain)[i]; }
    }
    for (int p0 = 0; p0 < parts; p0 += 8) {
        f32x4 t[8][NV];
#pragma unroll
        for (int p = 0; p < 8; ++p)
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const int i = threadIdx.x + blockDim.x * j;
                if (p0 + p < parts && i < nv) t[p][j] = *(const f32x4*)(pr + (size_t)(p0 + p) * part_stride + 4 * i);
            }
#pragma unroll
        for (int p = 0; p < 8; ++p)
#pragma unroll
            for (int j = 0; j < NV; ++j)
                if (p0 + p < parts && (int)(threadIdx.x + blockDim.x * j) < nv) v[j] += t[p][j];
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int i = threadIdx.x + blockDim.x * j;
        if (i < nv) {
            v[j] = c[j] + v[j];
            cr[i] = v[j];
            ss += (v[j][0] * v[j][0] + v[j][1] * v[j][1]) + (v[j][2] * v[j][2] + v[j][3] * v[j][3]);
        }
    }
    const float inv = rsqrtf(block_sum(ss, scratch) / (float)N + eps);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int i = threadIdx.x + blockDim.x * j;
        if (i < nv) {
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (bf16)(v[j][e] * inv * g[j][e]);
            *(bf16x4*)(h + m * ldh + 4 * i) = o;
        }
    }
}

static int launch_split_sum(const float* scratch, int parts, void* C, int M, int N, size_t ldc, int mode, hipStream_t s) {
    const size_t stride = (size_t)M * N, results = mode == OUT_SWIGLU ? stride / 2 : stride;
    const bool half = mode == OUT_BF16 || mode == OUT_SWIGLU;
    // Up to 2,048 columns a result a thread: a row's eight workgroups of 256 columns then lie on the XCDs that wrote these columns, whose L2
    // still has them; four a thread spread a row over fewer (128 x 128 tiles with their sum, K 4,096, us by one and by four: 2,048 columns in 16
    // runs by 66, 96 and 128 rows 12.8 / 16.4, 13.4 / 18.7, 14.3 / 21.0, in 8 runs 15.5 / 17.0, 15.7 / 18.3, 16.0 / 19.2; 1,024 by 200 rows in 8 runs
    // 16.0 / 17.2.  8,192 columns in 4 runs by 96 rows 31.3 / 26.2, where four a thread make the eight; between them alike.)
    const int vec = (mode == OUT_SWIGLU ? N / 2 : N) > 2048 && N % 4 == 0 && ldc % 4 == 0 && (uintptr_t)C % (half ? 8 : 16) == 0 && (uintptr_t)scratch % 16 == 0 ? 4 : 1;
    const unsigned blocks = (unsigned)((results / vec + 255) / 256);
#define BR_SUM(MODE_)                                                                                                          \
    do {                                                                                                                       \
        if (vec == 4) gemm_split_sum_kernel<MODE_, 4><<<blocks, 256, 0, s>>>(scratch, parts, stride, C, M, N, ldc);            \
        else gemm_split_sum_kernel<MODE_, 1><<<blocks, 256, 0, s>>>(scratch, parts, stride, C, M, N, ldc);                     \
    } while (0)
    if (mode == OUT_BF16) BR_SUM(OUT_BF16);
    else if (mode == OUT_F32) BR_SUM(OUT_F32);
    else if (mode == OUT_F32_ACC) BR_SUM(OUT_F32_ACC);
    else BR_SUM(OUT_SWIGLU);
#undef BR_SUM
    return br_check_launch();
}

template <int MB>
static int launch_split(const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc, int mode,
                        int parts, float* scratch, hipStream_t s) {
    constexpr int RB = 4;
    const int nslab = (K + SLAB_K - 1) / SLAB_K;
    const int spp = (nslab + parts - 1) / parts;
    parts = (nslab + spp - 1) / spp;                                   // no empty run
    const size_t stride = (size_t)M * N;
    dim3 grid((unsigned)((N + 16 * RB - 1) / (16 * RB)), (unsigned)parts);
    gemm_skinny_lds_kernel<MB, RB, OUT_F32><<<grid, 256, 0, s>>>(A, W, scratch, M, N, K, lda, (size_t)N, spp, stride);
    int rc = br_check_launch();
    if (rc != BR_OK) return rc;
    return launch_split_sum(scratch, parts, C, M, N, ldc, mode, s);
}

// How many runs of k-slabs a product of 16 < M <= 64 rows is cut into when the caller gives
// scratch memory: enough (tile, run) workgroups of 64 weight rows for the chip, at least two
// slabs a run; 1 = not split.
static int split_parts(int M, int N, int K, int mode, size_t scratch_bytes) {
    if (M <= 16 || M > 64 || mode == OUT_SWIGLU) return 1;
    const int tiles = (N + 63) / 64, nslab = (K + SLAB_K - 1) / SLAB_K;
    int parts = 256 / tiles;
    if (parts > nslab / 2) parts = nslab / 2;
    if (parts > 8) parts = 8;
    if (parts < 2 || (size_t)parts * M * N * sizeof(float) > scratch_bytes) return 1;
    return parts;
}

// ------------------------------------------------------------------ gemm_stream ------
// M <= 16, K in steps of 128: weight streaming by workgroups that stay.  One workgroup per
// compute unit walks over tiles of 16 weight rows (tile t of workgroup b is b + t * grid);
// its 8 waves take the tile's 128-wide k-chunks in turn.  A wave brings a chunk of the
// tile (16 rows x 256 bytes) and the same chunk of the activations (8 or 16 rows) into a
// ring of LDS stages of its own with direct global-to-LDS loads: whole 256-byte row
// pieces per request, no registers, and the loads of the next chunk (of the next tile,
// at a tile's end) are in flight while this one is multiplied.  No wave waits for another
// inside a tile; at a tile's end the waves' sums meet in LDS (one barrier, two buffers)
// and are added in wave order.  The 16-byte columns of a row are XOR-swizzled by the row
// number through the choice of the global column a lane fetches.
//
// Two forms serve the RMS norm between a product that adds into the residual stream and the
// product that reads the normed rows, so that single-token steps launch no norm kernel
// (reference: op_rmsnorm, kernels/megakernel_ops.hip:1421-1446, a step of its own there):
//  * NORM = 1, the producer (with the accumulate epilogue): it reads the element it adds to,
//    writes the sum h back, writes bf16(h * g) (g: the next norm's weights) to `xg`, and the
//    sum of h^2 over its tile's 16 columns to ssq[tile * SSQ_LD + row].
//  * NORM = 2, the consumer: its activations are those bf16(h * g) rows; before its first
//    tile it adds the `ssq_tiles` sums of every row in a fixed order, and 1 / rms, the same
//    for a whole row, multiplies the sums at a tile's end:
//    y = rsqrt(mean(h^2) + eps) * sum_k W[n,k] (h[k] g[k]).
struct StreamNorm {
    const float* gain;     // producer: the next norm's weights [N]
    bf16* xg;              // producer: [M, ldx]
    size_t ldx;
    float* ssq;            // producer writes, consumer reads: [tiles, SSQ_LD]
    int ssq_tiles;         // consumer: tiles of the producer
    float inv_k, eps;      // consumer: 1 / width of the normed rows, the norm's eps
};
// Branches: weight rows b per .. + per multiply the activations b a_step elements on; output columns from gap_at on lie `gap`
// further on.  (A type of its own, so that the arguments of the other forms stay as short as they are.)
// Weight rows from tail_at on are one more branch, whose sums' tanh goes to bf16 rows of their own (the first half of a low-rank pair).
struct StreamBranches {
    int per;
    size_t a_step;
    int gap_at, gap;
    int tail_at;
    bf16* tail;
    size_t tail_ld;
};
template <int NORM> struct StreamArg { typedef StreamNorm type; };
template <> struct StreamArg<3> { typedef StreamBranches type; };
__device__ __forceinline__ size_t branch_rows(const StreamNorm&, int) { return 0; }
__device__ __forceinline__ size_t branch_rows(const StreamBranches& b, int n) { return (size_t)(n / b.per) * b.a_step; }
__device__ __forceinline__ int branch_gap(const StreamNorm&, int) { return 0; }
__device__ __forceinline__ int branch_gap(const StreamBranches& b, int n) { return n >= b.gap_at ? b.gap : 0; }

template <int RT, int XR, int KC, int S, int NW, int MODE, int NORM>
__global__ __launch_bounds__(NW * 64) void gemm_stream_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                              void* __restrict__ C, int M, int N, int K, size_t lda,
                                                              size_t ldc, int ntiles, StreamNorm nrm, int wl) {
    static_assert(NORM == 0 || (NORM == 1 && MODE == OUT_F32_ACC) || (NORM == 2 && MODE != OUT_F32_ACC), "norm forms");
    constexpr int STEPS = KC / 32;
    constexpr int ROWB = KC * 2;
    constexpr int STAGE = (RT + XR) * ROWB;
    constexpr int WDMA = RT * ROWB / 1024;
    constexpr int NDMA = STAGE / 1024;
    constexpr int CPL = ROWB / 16;          // 16-byte columns per row
    constexpr int RPI = 64 / CPL;           // rows per DMA instruction
    constexpr int LPI = NDMA;
    constexpr int D = S - 1;
    static_assert(RPI >= 1 && (D - 1) * LPI <= 63, "wait count");
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    float* red = (float*)(smem + NW * S * STAGE);       // [2][NW][16][17]
    float* rstd = red + 2 * NW * 16 * 17;               // NORM 2: [16]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    unsigned char* ring = smem + wave * (S * STAGE);
    const unsigned ring_lds = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)ring);

    const int nch = K / KC;
    const int ncw = (nch - wave + NW - 1) / NW;
    // Where in k this workgroup starts: workgroups that walk their rows in step ask the same few memory
    // channels at the same time; a start of its own for each spreads them (measured: 4 to 9 % on the
    // products of 4,096 to 6,144 weight rows).  The order of a column's sum depends on the column only.
    const int rot = (int)(((unsigned)blockIdx.x * 2654435761u) >> 8) % nch;
    const int my_tiles = (ntiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
    const int nitems = my_tiles * ncw;

    // DMA lane mapping
    const int drow = lane / CPL, dcol = lane % CPL;
    const int wstep = wl ? WL_BLOCK_ELEMS : KC;        // elements from a chunk of a weight row to the next
    f32x4 acc = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};

    int is_t = 0, is_c = 0;      // issue cursor: local tile index, local chunk index
    int cp_t = 0, cp_c = 0;      // compute cursor
    int buf = 0;

#define ISSUE(J)                                                                                         \
    do {                                                                                                 \
        int chunk_ = wave + is_c * NW + rot;                                                             \
        if (chunk_ >= nch) chunk_ -= nch;                                                                \
        const int n0_ = ((int)blockIdx.x + is_t * (int)gridDim.x) * RT;                                  \
        _Pragma("unroll") for (int q_ = 0; q_ < NDMA; ++q_) {                                            \
            const int row_ = q_ * RPI + drow;                                                            \
            const bf16* gp_;                                                                             \
            if (q_ < WDMA) {                                                                             \
                int nrow_ = n0_ + row_;                                                                  \
                if (nrow_ > N - 1) nrow_ = N - 1;                                                        \
                gp_ = W + w_row_base(nrow_, K, wl) + (size_t)chunk_ * wstep + ((dcol ^ (row_ & 7)) * 8);  \
            } else {                                                                                     \
                int m_ = row_ - RT;                                                                      \
                if (m_ > M - 1) m_ = M - 1;                                                              \
                gp_ = A + (size_t)m_ * lda + (size_t)chunk_ * KC + ((dcol ^ (row_ & 7)) * 8);            \
            }                                                                                            \
            const unsigned lds_ = __builtin_amdgcn_readfirstlane(ring_lds + (J) * STAGE + q_ * 1024);    \
            if (q_ < WDMA)                              /* weights pass once: non-temporal */            \
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds_), "v"(gp_) : "m0"); \
            else                                        /* activations are every workgroup's: they stay cached */ \
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_), "v"(gp_) : "m0"); \
        }                                                                                                \
        if (++is_c == ncw) {                                                                             \
            is_c = 0;                                                                                    \
            ++is_t;                                                                                      \
        }                                                                                                \
    } while (0)

    // prologue
#pragma unroll
    for (int j = 0; j < D; ++j)
        if (j < nitems) ISSUE(j);
    // NORM 2: row m = tid / 32, its 32 lanes take the tiles' sums in turn.  The first eight a lane are requested
    // here and added at the first tile's end, so that their way from memory runs under the first tile.
    float ssq_pre[8];
    if constexpr (NORM == 2) {
        const int m = tid >> 5, l = tid & 31;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            ssq_pre[j] = (m < M && l + 32 * j < nrm.ssq_tiles) ? nrm.ssq[(size_t)(l + 32 * j) * SSQ_LD + m] : 0.f;
    }

    for (int base = 0; base < nitems; base += S) {
#pragma unroll
        for (int j = 0; j < S; ++j) {
            const int it = base + j;
            if (it < nitems) {
                // wait for item `it`
                if (it + D - 1 < nitems) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * LPI) : "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                if (it + D < nitems) ISSUE((j + D) % S);
                // compute
                const unsigned char* st = ring + j * STAGE;
                const int rr = RT == 8 ? (r16 & 7) : r16;
                const int xr = XR == 8 ? (r16 & 7) : r16;
                bf16x8 wf[STEPS], xv[STEPS];
#pragma unroll
                for (int s = 0; s < STEPS; ++s) {
                    wf[s] = *(const bf16x8*)(st + rr * ROWB + (((4 * s + g) ^ (rr & 7)) * 16));
                    xv[s] = *(const bf16x8*)(st + (RT + xr) * ROWB + (((4 * s + g) ^ (xr & 7)) * 16));
                }
#pragma unroll
                for (int s = 0; s < STEPS; s += 2) {
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s], xv[s], acc, 0, 0, 0);
                    acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s + 1], xv[s + 1], acc1, 0, 0, 0);
                }
                if (++cp_c == ncw) {
                    cp_c = 0;
                    const int n0 = ((int)blockIdx.x + cp_t * (int)gridDim.x) * RT;
                    ++cp_t;
                    float* rb = red + buf * (NW * 16 * 17);
                    if constexpr (NORM == 2) if (cp_t == 1) {
                        const int m = tid >> 5, l = tid & 31;
                        float t = 0.f;
#pragma unroll
                        for (int j = 0; j < 8; ++j) t += ssq_pre[j];
                        if (m < M)
                            for (int c = l + 256; c < nrm.ssq_tiles; c += 32) t += nrm.ssq[(size_t)c * SSQ_LD + m];
#pragma unroll
                        for (int o = 16; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
                        if (l == 0) rstd[m] = m < M ? rsqrtf(t * nrm.inv_k + nrm.eps) : 0.f;
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) rb[(wave * 16 + 4 * g + r) * 17 + r16] = acc[r] + acc1[r];
                    acc = {0.f, 0.f, 0.f, 0.f};
                    acc1 = {0.f, 0.f, 0.f, 0.f};
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    if constexpr (MODE == OUT_SWIGLU) {
                        for (int e = tid; e < 8 * 16; e += NW * 64) {
                            const int m = e >> 3, jl = e & 7;
                            if (m < M && n0 + jl + 8 < N) {
                                float gv = 0.f, uv = 0.f;
#pragma unroll
                                for (int w = 0; w < NW; ++w) { gv += rb[(w * 16 + jl) * 17 + m]; uv += rb[(w * 16 + jl + 8) * 17 + m]; }
                                if (NORM == 2) { gv *= rstd[m]; uv *= rstd[m]; }
                                ((bf16*)C)[(size_t)m * ldc + n0 / 2 + jl] = (bf16)silu_mul(gv, uv);
                            }
                        }
                    } else if constexpr (NORM == 1) {
                        // whole waves (16 lanes a row): the row's 16 squares of this tile are added by shuffles
                        if (tid < 16 * XR) {
                            const int m = tid >> 4, nl = tid & 15, n = n0 + nl;
                            const bool ok = m < M && n < N;
                            float h = 0.f;
                            if (ok) {
                                float v = 0.f;
#pragma unroll
                                for (int w = 0; w < NW; ++w) v += rb[(w * 16 + nl) * 17 + m];
                                const size_t idx = (size_t)m * ldc + n;
                                h = ((float*)C)[idx] + v;
                                ((float*)C)[idx] = h;
                                nrm.xg[(size_t)m * nrm.ldx + n] = (bf16)(h * nrm.gain[n]);
                            }
                            float sq = h * h;
#pragma unroll
                            for (int o = 8; o > 0; o >>= 1) sq += __shfl_xor(sq, o, 64);
                            if (nl == 0 && m < M) nrm.ssq[(size_t)(n0 / 16) * SSQ_LD + m] = sq;
                        }
                    } else {
                        for (int e = tid; e < RT * 16; e += NW * 64) {
                            const int m = e / RT, nl = e % RT, n = n0 + nl;
                            if (m < M && n < N) {
                                float v = 0.f;
#pragma unroll
                                for (int w = 0; w < NW; ++w) v += rb[(w * 16 + nl) * 17 + m];
                                if (NORM == 2) v *= rstd[m];
                                const size_t idx = (size_t)m * ldc + n;
                                if (MODE == OUT_BF16) ((bf16*)C)[idx] = (bf16)v;
                                else if (MODE == OUT_F32) ((float*)C)[idx] = v;
                                // one add per element and product, without a read that this wave would
                                // have to wait for behind its loads in flight
                                else unsafeAtomicAdd((float*)C + idx, v);
                            }
                        }
                    }
                    buf ^= 1;
                }
            }
        }
    }
#undef ISSUE
}



#define STREAM_KC 128
#define STREAM_NW 8
template <int XR, int NORM>
static int launch_stream(const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc,
                         int mode, hipStream_t s, const StreamNorm& nrm, int wl) {
    constexpr int RT = 16, KC = STREAM_KC, S = 2, NW = STREAM_NW;
    static_assert(KC == 128, "the blocked weight layout has 128 k a block");
    const int cus = br_device_cus();
    if (!cus) return BR_LAUNCH_FAILED;
    const int ntiles = (N + RT - 1) / RT;
    const int grid = ntiles < cus ? ntiles : cus;
    constexpr size_t lds = (size_t)NW * S * (RT + XR) * KC * 2 + 2 * NW * 16 * 17 * 4 + 16 * 4;
#define BR_STREAM(MODE_)                                                                                        \
    do {                                                                                                        \
        auto kern = gemm_stream_kernel<RT, XR, KC, S, NW, MODE_, NORM>;                                         \
        static bool set = false;                                                                                \
        if (!set) {                                                                                             \
            if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != \
                hipSuccess)                                                                                     \
                return BR_LAUNCH_FAILED;                                                                        \
            set = true;                                                                                         \
        }                                                                                                       \
        kern<<<grid, NW * 64, lds, s>>>(A, W, C, M, N, K, lda, ldc, ntiles, nrm, wl);                           \
    } while (0)
    if constexpr (NORM == 1) {
        BR_STREAM(OUT_F32_ACC);
    } else {
        if (mode == OUT_BF16) BR_STREAM(OUT_BF16);
        else if (mode == OUT_F32) BR_STREAM(OUT_F32);
        else if (mode == OUT_SWIGLU) BR_STREAM(OUT_SWIGLU);
        else if constexpr (NORM == 0) BR_STREAM(OUT_F32_ACC);
        else return BR_BAD_ARG;
    }
#undef BR_STREAM
    return br_check_launch();
}

// ------------------------------------------------------------- gemm_stream_tile ------
// Few rows (up to 128) against few enough weight rows that a tile of 16, 24 or 32 of them for every workgroup covers the matrix in
// one round: K in steps of 128, the whole of it in one workgroup, shared over its waves (wave w takes the 64-wide chunks w, w + NW,
// ..), so that no sums of runs are written, read and added by another launch.  A wave brings its chunk of the tile's weights and the
// same chunk of all activations (16 MB rows) into two LDS stages of its own by direct loads; what has landed goes to registers at
// once and the stage is asked for again before the matrix instructions, so that two stages are in flight all but a few
// cycles.  At the end the waves' sums meet in LDS and are added in wave order.
//
// Up to 16 rows the memory bounds it: what counts is that all compute units stream the same share (6,144 weight rows are 256 tiles of
// 24; 384 tiles of 16 leave half of the units with twice the work of the others), and that two workgroups share a unit where there are
// more tiles than units.  With more rows it is the compute unit's path from the L2, 62 to 70 GB/s here, which carries 16 MB activation
// rows for the tile's 16 to 32: gemm_stream_wide shares them over more weight rows and pays with runs along k and their sum, and wins
// where K is long (see tile_rows).
// us, weights in no cache, before -> now (before: resident workgroups that walk tiles of 16 rows up to 16 rows, gemm_stream_wide with the
// sum of its runs up to 64, the eight-wave tiles with theirs beyond): 6,144 x 4,096 by 8 rows 12.7 -> 10.9; 4,096 x 4,096, 2,048 x 2,048,
// 8,192 x 4,096 by 24 rows 14.3 -> 9.2, 9.5 -> 5.6, 18.7 -> 13.6, by 64 rows 14.9 -> 13.3, 11.6 -> 7.8, 19.9 -> 18.3, by 80 rows
// 22.4 -> 15.3, 11.5 -> 8.8, 28.1 -> 20.9.
// Chunks of 128 in one stage took 0 to 10 % longer; rows of activations further apart than a power of two changed nothing.
//
// NORM 1, 2: as gemm_stream's forms (the tile's columns as sums of squares by 16); C, or the sums of squares, are asked for
// before the first weights and used at the end.  NORM 3: products of several inputs by stacked weights in one launch
// (br_gemm_bf16_branches); a tile lies in one branch.  NORM 4: float rows that 16-byte stores can take are added to, and asked for ahead
// as NORM 1 does (added in memory instead, a column at a time, it took, us: 64 rows, 6,144 x 4,096 22.8, now 17.4; 96 rows 30.4,
// 22.3; 128 rows, 6,144 x 1,024 24.6, 12.7; 8,192 x 4,096 by 64 rows 22.8, 18.8).  A form of its own: asked for under a test of `mode`, the
// products that add to nothing waited 0.2 us for it.
constexpr int tile_waves(int RT, int MB) { return 640 / (RT + 16 * MB) < 8 ? 640 / (RT + 16 * MB) : 8; }     // 160 KB of LDS
#define TILE_KC 64
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <int RT, int MB, int NORM>
__global__ __launch_bounds__(64 * tile_waves(RT, MB)) void gemm_stream_tile_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                                                   void* __restrict__ C, int M, int N, int K, size_t lda,
                                                                                   size_t ldc, int mode, int vec, typename StreamArg<NORM>::type nrm, int wl) {
    static_assert(NORM != 1 || RT % 16 == 0, "sums of squares by 16 columns");
    constexpr int NW = tile_waves(RT, MB), RB = (RT + 15) / 16, ROWS = RT + 16 * MB, STAGE = ROWS * TILE_KC * 2, NL = STAGE / 1024;
    constexpr int WL_LOADS = RT / 8;   // loads of 8 rows by 128 bytes: the weights', then the activations'
    constexpr int GROUPS = RB * MB, PER = (GROUPS + NW - 1) / NW;        // blocks of 16 x 16 results; those of a wave
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = uniform((int)threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
    unsigned char* ring = smem + wave * (2 * STAGE);
    const unsigned ring_lds = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)ring);
    const int nch = K / TILE_KC, ncw = (nch - wave + NW - 1) / NW;
    const int n0 = (int)blockIdx.x * RT;
    // where in k the workgroup starts: see gemm_stream
    const int rot = uniform((int)((((unsigned)blockIdx.x * 2654435761u) >> 8) % (unsigned)nch));

    // blocks of results: block t = wave + i NW of this wave; lane (r16, g) holds row 16 j + r16, columns col .. col + 3
    auto block_of = [&](int i) { return wave + i * NW; };
    auto row_of = [&](int t) { return 16 * (t % MB) + r16; };
    auto col_of = [&](int t) {          // -1: columns of another block (the last block of 24 weight rows begins at the eighth)
        const int b = t / MB;
        if (RT % 16 && b == RB - 1) return g < 2 ? -1 : n0 + RT - 16 + 4 * g;
        return n0 + 16 * b + 4 * g;
    };
    // sums of squares: a lane a row, and where rows are few its wave's other lanes the next tiles; 32 loads or less for 256 tiles
    constexpr int QR = MB == 1 ? 16 : MB == 2 ? 32 : 64, QT = 64 / QR, QN = 32 / QT;
    const int q_row = lane % QR, q_tile = wave * QT + lane / QR;
    f32x4 c_pre[PER], g_pre[PER];
    float q_pre[QN];
    if constexpr (NORM == 4) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int t = block_of(i), m = row_of(t), n = col_of(t);
            c_pre[i] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (t < GROUPS && m < M && n >= 0 && n < N) c_pre[i] = *(const f32x4*)((const float*)C + (size_t)m * ldc + n);
        }
    }
    if constexpr (NORM == 1) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int t = block_of(i), m = row_of(t), n = col_of(t);
            c_pre[i] = g_pre[i] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (t >= GROUPS || m >= M || n >= N) continue;
            if (vec) {
                c_pre[i] = *(const f32x4*)((const float*)C + (size_t)m * ldc + n);
                g_pre[i] = *(const f32x4*)(nrm.gain + n);
            } else
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    c_pre[i][e] = ((const float*)C)[(size_t)m * ldc + n + e];
                    g_pre[i][e] = nrm.gain[n + e];
                }
        }
    }
    if constexpr (NORM == 2) {
#pragma unroll
        for (int i = 0; i < QN; ++i) {
            const int t = q_tile + i * NW * QT;
            q_pre[i] = t < nrm.ssq_tiles && q_row < M ? nrm.ssq[(size_t)t * SSQ_LD + q_row] : 0.f;
        }
    }

    // A lane's 16 bytes of each load.  Rows beyond M or N are fetched from the last valid row and dropped at the store.
    const bf16* src[NL];
    const size_t w_k128 = wl ? WL_BLOCK_ELEMS : 128;                     // elements from 128 k of a weight row to the next
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int row = 8 * i + (lane >> 3), col = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
        if (i < WL_LOADS) {
            const int n = n0 + row < N ? n0 + row : N - 1;
            src[i] = W + w_row_base(n, K, wl) + col;
        } else {
            const int m = row - RT < M ? row - RT : M - 1;
            src[i] = A + branch_rows(nrm, n0) + (size_t)m * lda + col;
        }
    }
    int asked = 0;
    auto ask = [&](int st) {
        int c = wave + asked * NW + rot;
        if (c >= nch) c -= nch;
        const size_t w_at = (size_t)(c >> 1) * w_k128 + (c & 1) * TILE_KC, a_at = (size_t)c * TILE_KC;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const unsigned to = uniform((int)(ring_lds + st * STAGE + i * 1024));
            if (i < WL_LOADS)          // weights pass once: non-temporal
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(to), "v"(src[i] + w_at) : "m0", "memory");
            else
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(to), "v"(src[i] + a_at) : "m0", "memory");
        }
        ++asked;
    };
    f32x4 acc[2][RB][MB];
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int j = 0; j < MB; ++j) acc[0][b][j] = acc[1][b][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (0 < ncw) ask(0);
    if (1 < ncw) ask(1);
    for (int base = 0; base < ncw; base += 2) {
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            if (base + st >= ncw) continue;
            if (base + st + 1 < ncw) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NL) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            const unsigned char* at = ring + st * STAGE;
            bf16x8 wf[RB][2], xv[MB][2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    const int row = (b == RB - 1 ? RT - 16 : 16 * b) + r16;
                    wf[b][s] = *(const bf16x8*)(at + row * 128 + (((4 * s + g) ^ ((row >> 1) & 7)) * 16));
                }
#pragma unroll
                for (int j = 0; j < MB; ++j) {
                    const int row = RT + 16 * j + r16;
                    xv[j][s] = *(const bf16x8*)(at + row * 128 + (((4 * s + g) ^ ((row >> 1) & 7)) * 16));
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (base + st + 2 < ncw) ask(st);
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int b = 0; b < RB; ++b)
#pragma unroll
                    for (int j = 0; j < MB; ++j) acc[s][b][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[b][s], xv[j][s], acc[s][b][j], 0, 0, 0);
        }
    }
    // the waves' sums meet where the stages were
    f32x4* red = (f32x4*)smem;                         // [NW][GROUPS][64]
    float* sq = (float*)(smem + NW * GROUPS * 1024);   // NORM 2: [NW][64]
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int j = 0; j < MB; ++j) red[(wave * GROUPS + b * MB + j) * 64 + lane] = acc[0][b][j] + acc[1][b][j];
    if constexpr (NORM == 2) {
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < QN; ++i) t += q_pre[i];
        if (q_row < M)
            for (int c = q_tile + QN * NW * QT; c < nrm.ssq_tiles; c += NW * QT) t += nrm.ssq[(size_t)c * SSQ_LD + q_row];
#pragma unroll
        for (int o = QR; o < 64; o <<= 1) t += __shfl_xor(t, o, 64);
        sq[wave * 64 + lane] = t;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int t = block_of(i), m = row_of(t), n = col_of(t);
        if (t >= GROUPS) break;
        f32x4 v = red[t * 64 + lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += red[(w * GROUPS + t) * 64 + lane];
        if constexpr (NORM == 2) {
            float q = sq[m];
#pragma unroll
            for (int w = 1; w < NW; ++w) q += sq[w * 64 + m];
            v *= rsqrtf(q * nrm.inv_k + nrm.eps);
        }
        if (NORM != 4 && mode == OUT_SWIGLU) {
            // 16 weight rows are 8 gates, then the 8 up values of the same outputs
            f32x4 up;
#pragma unroll
            for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(v[e], 32, 64);
            if (m < M && g < 2 && n < N) {
                bf16x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = (bf16)silu_mul(v[e], up[e]);
                bf16* to = (bf16*)C + (size_t)m * ldc + (n0 + 16 * (t / MB)) / 2 + 4 * g;
                if (vec) *(bf16x4*)to = o;
                else
#pragma unroll
                    for (int e = 0; e < 4; ++e) to[e] = o[e];
            }
            continue;
        }
        if constexpr (NORM == 1) {
            // whole waves: a row's 16 squares of this block are added by shuffles
            const f32x4 h = c_pre[i] + v;
            float q = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) q += h[e] * h[e];
            q += __shfl_xor(q, 16, 64);
            q += __shfl_xor(q, 32, 64);
            if (m >= M || (RT > 16 && n >= N)) continue;   // a tile of 32 rows may end 16 columns behind the last one
            if (g == 0) nrm.ssq[(size_t)(n / 16) * SSQ_LD + m] = q;
            float* to = (float*)C + (size_t)m * ldc + n;
            bf16* xg = nrm.xg + (size_t)m * nrm.ldx + n;
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (bf16)(h[e] * g_pre[i][e]);
            if (vec) {
                *(f32x4*)to = h;
                *(bf16x4*)xg = o;
            } else
#pragma unroll
                for (int e = 0; e < 4; ++e) { to[e] = h[e]; xg[e] = o[e]; }
            continue;
        }
        if (m >= M || n < 0 || n >= N) continue;
        if constexpr (NORM == 3) if (n0 >= nrm.tail_at) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < N) nrm.tail[(size_t)m * nrm.tail_ld + n - nrm.tail_at + e] = (bf16)tanhf(v[e]);
            continue;
        }
        float* to = (float*)C + (size_t)m * ldc + n + branch_gap(nrm, n0);
        bf16* to16 = (bf16*)C + (size_t)m * ldc + n;
        if (NORM == 4 || (vec && mode != OUT_F32_ACC)) {   // N in steps of 4: all four columns
            if constexpr (NORM == 4) v = c_pre[i] + v;
            if (NORM != 4 && mode == OUT_BF16) {
                bf16x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = (bf16)v[e];
                *(bf16x4*)to16 = o;
            } else *(f32x4*)to = v;
            continue;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (n + e >= N) break;
            if (mode == OUT_BF16) to16[e] = (bf16)v[e];
            else if (mode == OUT_F32) to[e] = v[e];
            else unsafeAtomicAdd(to + e, v[e]);        // one add per element, no read to wait for
        }
    }
}

// rt: weight rows of a workgroup (16, 24, 32).  norm as NORM above; 1 and 2 up to 64 rows, 1 with N and rt in steps of 16.
template <int RT, int MB, int NORM>
static int launch_tile_form(const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc, int mode, hipStream_t s,
                            const typename StreamArg<NORM>::type& nrm, int wl) {
    constexpr int lds = tile_waves(RT, MB) * 2 * (RT + 16 * MB) * TILE_KC * 2;
    static_assert(lds <= 160 * 1024, "LDS of a compute unit");
    auto kern = gemm_stream_tile_kernel<RT, MB, NORM>;
    static bool set = false;
    if (!set) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return BR_LAUNCH_FAILED;
        set = true;
    }
    // rows that 16-byte stores (8 of bf16) can take
    const bool half = mode == OUT_BF16 || mode == OUT_SWIGLU;
    int vec = N % 4 == 0 && ldc % 4 == 0 && (uintptr_t)C % (half ? 8 : 16) == 0;
    if constexpr (NORM == 1) vec = vec && (nrm.ldx % 4 == 0 && (uintptr_t)nrm.xg % 8 == 0 && (uintptr_t)nrm.gain % 16 == 0);
    if constexpr (NORM == 3) vec = vec && nrm.gap % 4 == 0;
    if constexpr (NORM == 0) if (vec && mode == OUT_F32_ACC) return launch_tile_form<RT, MB, 4>(A, W, C, M, N, K, lda, ldc, mode, s, nrm, wl);
    kern<<<(N + RT - 1) / RT, 64 * tile_waves(RT, MB), lds, s>>>(A, W, C, M, N, K, lda, ldc, mode, vec, nrm, wl);
    return br_check_launch();
}
template <int MB>
static int launch_tile_rows(int rt, int norm, const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc, int mode, hipStream_t s,
                            const StreamNorm& nrm, int wl) {
#define BR_TILE(RT_, NORM_) return launch_tile_form<RT_, MB, NORM_>(A, W, C, M, N, K, lda, ldc, mode, s, nrm, wl)
    if (norm == 0) {
        if (rt == 16) BR_TILE(16, 0);
        if (rt == 24) BR_TILE(24, 0);
        if (rt == 32) BR_TILE(32, 0);
    }
    if constexpr (MB <= 4) {
        if (norm == 1 && rt == 16) BR_TILE(16, 1);
        if (norm == 1 && rt == 32) BR_TILE(32, 1);
        if (norm == 2 && rt == 16) BR_TILE(16, 2);
        if (norm == 2 && rt == 24) BR_TILE(24, 2);
        if (norm == 2 && rt == 32) BR_TILE(32, 2);
    }
#undef BR_TILE
    return BR_BAD_ARG;
}
#define TILE_MAX_ROWS 128
static int launch_stream_tile(int rt, int norm, const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc, int mode, hipStream_t s,
                              const StreamNorm& nrm, int wl) {
    if (rt == 24 && (mode == OUT_SWIGLU || norm == 1)) return BR_BAD_ARG;
    switch ((M + 15) / 16) {
        case 1: return launch_tile_rows<1>(rt, norm, A, W, C, M, N, K, lda, ldc, mode, s, nrm, wl);
        case 2: return launch_tile_rows<2>(rt, norm, A, W, C, M, N, K, lda, ldc, mode, s, nrm, wl);
        case 3: return launch_tile_rows<3>(rt, norm, A, W, C, M, N, K, lda, ldc, mode, s, nrm, wl);
        case 4: return launch_tile_rows<4>(rt, norm, A, W, C, M, N, K, lda, ldc, mode, s, nrm, wl);
        case 5: return launch_tile_rows<5>(rt, norm, A, W, C, M, N, K, lda, ldc, mode, s, nrm, wl);
        case 6: return launch_tile_rows<6>(rt, norm, A, W, C, M, N, K, lda, ldc, mode, s, nrm, wl);
        case 7: return launch_tile_rows<7>(rt, norm, A, W, C, M, N, K, lda, ldc, mode, s, nrm, wl);
        case 8: return launch_tile_rows<8>(rt, norm, A, W, C, M, N, K, lda, ldc, mode, s, nrm, wl);
    }
    return BR_BAD_ARG;
}
// The weight rows of a workgroup (16, 24 or 32) where gemm_stream_tile is the faster kernel, else 0.
// Up to 16 rows always (K in steps of 128 from 1,024; but see resident_pays): the fewest weight rows for the busiest compute unit, the same for every number
// of rows, so that a row's bits do not depend on the others'; of two that are alike the taller where one round covers the matrix
// (8,192 x 4,096: 12.6 us by 32, 13.7 by 16), else the lower, of which two workgroups share a unit (32,768 x 4,096 by 8 rows:
// 43.9 by 16, 46.0 by 24, 46.5 by 32).  One resident workgroup a unit that walked tiles of 16 rows, as gemm_stream does, took, at 1, 8
// and 16 rows: 6,144 x 4,096 12.2 / 12.7 / 13.8 (now 10.6 / 10.9 / 11.0), 32,768 x 4,096 45.3 / 47.0 / 54.3 (43.3 / 43.9 / 49.2),
// 5,120 x 13,824 32.0 / 32.9 / 36.8 (25.5 / 27.2 / 28.0), 4,096 x 14,336 21.2 / 21.4 / 24.3 (20.7 / 21.5 / 23.5), 2,048 x 8,192
// 10.7 / 9.9 / 11.2 (9.9 / 9.8 / 11.6).  Against up to 4,096 weight rows, where 16 balance one round either way, tiles gain 2 to 10 % at one row
// and lose 2 to 5 % at 9 to 16 (2,048 x 8,192 added into rows 12.3 and 11.8).
// More rows, by counts in microseconds.  Up to 64, fitted to 18 shapes (512 to 12,288 weight rows, K 1,024 to 14,336) at rows from 17
// to 64, mean error 5 %: a tile's rows and activations over a unit's path at 69 GB/s, and its share of the memory's, against gemm_stream_wide
// with the sum of its runs.  Single rounds only: matrices of more (32,768 x 4,096 by 32 rows: 47 us shared, 50 by tiles) have no sums to save.
// Beyond 64, fitted to 143 shapes (256 to 8,192 weight rows, K 512 to 14,336) at six numbers of rows, mean error 5 %, against the
// eight-wave tiles with the sum of theirs, 7 % and less 8 %, since these differ by up to a fifth from card to card: 8,192 x 14,336 by
// 65 rows 49 to 54 us on three cards, 62 by tiles on each; 7,168 x 11,008 38 and 48; 8,192 x 4,096 28 and 20; 4,096 x 4,096 21 and 15.
// The lines gain 1.25 in the mean over these shapes and lose 6 % at most.  by16: whole blocks of 16 columns only (NORM 1).
static int tile_rows(int M, int N, int K, int mode, int cus, bool by16 = false) {
    if (M <= 0 || M > TILE_MAX_ROWS || K % 128 || K < (M <= 16 ? 1024 : 256) || cus <= 0 || (M > 16 && N > 32 * cus)) return 0;
    int best_rt = 0;
    double best = 1e30;
    const bool low = M <= 16 && N > 32 * cus;
    const int m16 = (M + 15) / 16 * 16;
    for (int i = 0; i < 3; ++i) {
        const int rt = low ? 16 + 8 * i : 32 - 8 * i;
        if (rt == 24 && (mode == OUT_SWIGLU || by16)) continue;
        const int rounds = (N + rt * cus - 1) / (rt * cus);
        const double t = M <= 16   ? (double)rounds * rt
                         : M <= 64 ? 3.1 + rounds * (double)(rt + M) * K * 2.9e-5 + (double)N * K * 1.27e-7
                                   : 2.6 + rounds * ((double)(rt + m16) * K * 2.83e-5 + 0.016 * m16) + (double)N * K * 1.09e-7;
        if (t < best * (1.0 - 1e-9)) { best = t; best_rt = rt; }
    }
    if (M <= 16) return best_rt;
    const double mb = (double)N * K * 2e-7;                              // weights in 10 MB
    const double other = M <= 64 ? 0.96 * (6.2 + 0.043 * M + 1.61 * mb + 1.6e-6 * M * N + 4.7e-6 * M * K - (mode == OUT_SWIGLU ? 2.4 : 0.0))
                                 : 8.2 + 1.04 * mb + 0.63e-3 * K + 0.59e-3 * N + 0.025 * M;
    return best < other ? best_rt : 0;
}

// Where products of up to 16 rows without a norm stay with gemm_stream's resident workgroups (the same for every number of rows): a chunk
// a wave, or two and an add into rows, is over before the tile's two stages have anything to hide, so that many tiles pay a workgroup's start each
// (K 1,024 by 8 rows, us, tiles and resident: 16,384 weight rows 8.7 / 8.2, 65,536 27.9 / 23.1, gated 28,672 14.4 / 12.3, added into float rows 2,048
// 4.2 / 3.9; K 2,048 added 2,048 5.2 / 4.9), but not where 24 or 32 rows balance one round (6,144 5.0 / 5.4, 8,192 5.5 / 5.7) nor from K 1,152
// on, of which resident waves take two uneven shares (65,536 by 8 rows 29.5 / 34.4); and long K over more than one round (K 12,288 to 14,336,
// 10,240 to 16,384 weight rows by 8 rows 45.0 / 43.4 to 73.8 / 70.5; K 11,008 41.2 / 41.0).
static bool resident_pays(int N, int K, int mode, int cus) {
    if (N > 32 * cus) return K == 1024 || K >= 12288;
    return N <= 16 * cus && (K == 1024 || (mode == OUT_F32_ACC && K <= 2048 && N <= 12 * cus));
}

// Whether the norm forms of up to 16 rows, too, leave gemm_stream: one round of tiles (every workgroup reads all sums of squares:
// 28,672 x 4,096 by 8 rows 38.7 us by tiles, 37.2 by resident workgroups; 6,144 x 4,096 11.5 and 12.9), and K below 8,192 (4,096 x 14,336
// by 8 and 16 rows 21.4 and 24.0 against 20.9 and 23.2; 4,096 x 4,096 8.1 and 9.0 against 8.6 and 9.0).  Resident over tiles, K 1,024 to
// 7,168: a norm prepared by 1, 8 and 16 rows 1.02 to 1.10, 1.00 to 1.05 and 0.97 to 1.05 against up to 4,096 weight rows, 1.03 to 1.26 against
// 5,120 to 8,192; one used 1.00 to 1.13 and 1.01 to 1.37 (6,144 the most).
static bool tile_norms(int M, int N, int K, int cus) { return M > 16 || (N <= 32 * cus && K < 8192); }

// What launch_stream_tile needs of its operands beside aligned rows.
static bool tile_takes(int M, int K, size_t lda) { return M > 0 && M <= TILE_MAX_ROWS && K % 128 == 0 && K >= 256 && lda >= (size_t)K; }

// ------------------------------------------------------------- gemm_stream_wide ------
// 16 < M <= 64, K in steps of 128: the same streaming by workgroups that stay, with the
// activations shared.  A unit of work is a tile of 16 HB weight rows (64 to 128) over one run of
// k-chunks (the whole K, or one of `parts` runs); height and runs are chosen so that the units
// fill the compute units in whole rounds (wide_shape below: 28,672 rows are 256 tiles of 112).
// Unit u of workgroup b is b + u * grid.  A stage of the workgroup's 3-stage LDS ring holds one
// 128-wide chunk of the tile and of the activations (16 MB rows), brought by all 8 waves with
// direct global-to-LDS loads, two chunks ahead; one barrier per chunk.  Wave w multiplies the
// weight rows 16 (w % 4) .. + 16 (and 64 + 16 (w % 4) .. + 16 where the tile has them) with
// k-steps 2 (w / 4), 2 (w / 4) + 1 of the chunk; the two k-halves are added in LDS at the
// unit's end (half 0 + half 1), in the stage that was multiplied last.  With `parts` > 1 the
// unit's float sums go to a matrix of its run (`part_stride` elements apart) for
// gemm_split_sum_kernel; else the epilogue (`mode`) is applied here.  The epilogue's form is
// chosen at run time: it runs once per unit, the chunk loop is the same for all.
// scale: the activations are the bf16(h * g) rows that the product before left for an RMS norm
// (see gemm_stream's NORM forms); the sums are multiplied by 1 / rms of their row, run by run.
#define WIDE_S 3
// BRANCHES: products of several inputs by stacked weights in one launch (br_gemm_bf16_branches); a unit lies in one branch.
template <int MB, int HB, bool BRANCHES = false>
__global__ __launch_bounds__(512) void gemm_stream_wide_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                               void* __restrict__ C, int M, int N, int K, size_t lda,
                                                               size_t ldc, int mode, int partial, int scale,
                                                               int ntiles, int parts, int cpp, size_t part_stride,
                                                               typename StreamArg<BRANCHES ? 3 : 0>::type nrm, int wl) {
    constexpr int S = WIDE_S, D = S - 1, NW = 8, H = 16 * HB;
    constexpr int ROWS = H + 16 * MB;                // stacked rows of a stage: weights, then activations
    constexpr int STAGE = ROWS * 256;
    constexpr int NLD = ROWS / 4;                    // wave-loads of a chunk: 4 rows of 256 bytes each
    constexpr int NDMA = (NLD + NW - 1) / NW;        // of each wave; surplus ones repeat the chunk's last load
    constexpr int RLD = 16 * MB + 1;
    constexpr bool TWO = HB > 4;
    static_assert(HB >= 4 && HB <= 8 && (D - 1) * NDMA <= 63 && H * RLD * 4 <= STAGE, "stage");
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    float* rstd = (float*)(smem + S * STAGE);        // scale: [64]
    float* sq = rstd + 64;                           // scale: [NW][64], see below
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int rb = wave & 3, khalf = wave >> 2;
    const bool has1 = TWO && rb + 4 < HB;
    const unsigned ring_lds = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)smem);
    const int nch = K / 128;
    const int nunits = ntiles * parts;
    const int my_units = (nunits - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;

    f32x4 acc[TWO ? 2 : 1][MB];
#pragma unroll
    for (int t = 0; t < (TWO ? 2 : 1); ++t)
#pragma unroll
        for (int j = 0; j < MB; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    f32x4 far[TWO ? 2 : 1][MB];                             // BRANCHES: the sums of the runs of four chunks before
    if (BRANCHES) {
#pragma unroll
        for (int t = 0; t < (TWO ? 2 : 1); ++t)
#pragma unroll
            for (int j = 0; j < MB; ++j) far[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // Cursors over this workgroup's chunks in order.  What depends on the unit only (its tile, its run
    // of chunks, each lane's addresses) is worked out once per unit, so that a chunk costs each wave its
    // loads, an address step and a count.
    int is_u = 0, is_left = 0, cp_u = 0, cp_left = 0;       // units begun, chunks of the current one to go
    int is_wrap = 0, is_len = 0;                            // chunks to go before the run's first chunk is next; the run's length
    // Where in its run of chunks a workgroup starts (it wraps round to the run's first chunk): workgroups
    // that walk their rows in step ask the same few memory channels at the same time.
    const unsigned start_hash = ((unsigned)blockIdx.x * 2654435761u) >> 8;
    int issued = 0, done = 0;
    unsigned is_off = 0, cp_off = 0;                        // the ring's stage to fill, to multiply (bytes)
    const bf16* src[NDMA];                                  // this lane's 16 bytes of each of its loads
    const int wstep = wl ? WL_BLOCK_ELEMS : 128;                      // elements from a chunk of a weight row to the next
#define WIDE_RUN_LENGTH(U, LEN)                                                                               \
    do {                                                                                                      \
        const int c0_ = (((int)blockIdx.x + (U) * (int)gridDim.x) % parts) * cpp;                             \
        LEN = (c0_ + cpp < nch ? c0_ + cpp : nch) - c0_;                                                      \
    } while (0)
#define WIDE_LOAD_INDEX(Q) ((wave * NDMA + (Q)) < NLD - 1 ? (wave * NDMA + (Q)) : NLD - 1)
#define WIDE_SETUP()                                                                                          \
    do {                                                                                                      \
        const int unit_ = (int)blockIdx.x + is_u * (int)gridDim.x;                                            \
        const int tile_ = unit_ / parts, c0_ = (unit_ % parts) * cpp;                                         \
        is_left = (c0_ + cpp < nch ? c0_ + cpp : nch) - c0_;                                                  \
        is_len = is_left;                                                                                     \
        const int rot_ = (int)(start_hash % (unsigned)is_left);                                               \
        is_wrap = is_left - rot_;                                                                             \
        _Pragma("unroll") for (int q_ = 0; q_ < NDMA; ++q_) {                                                 \
            const int row_ = WIDE_LOAD_INDEX(q_) * 4 + (lane >> 4);                                           \
            const bf16* gp_;                                                                                  \
            if (row_ < H) {                                                                                   \
                int n_ = tile_ * H + row_;                                                                    \
                if (n_ > N - 1) n_ = N - 1;                                                                   \
                gp_ = W + w_row_base(n_, K, wl) + (size_t)(c0_ + rot_) * wstep;                               \
            } else {                                                                                          \
                int m_ = row_ - H;                                                                            \
                if (m_ > M - 1) m_ = M - 1;                                                                   \
                gp_ = A + (size_t)m_ * lda + (size_t)(c0_ + rot_) * 128;                                      \
                gp_ += branch_rows(nrm, tile_ * H);                                                           \
            }                                                                                                 \
            src[q_] = gp_ + (((lane & 15) ^ (row_ & 7)) * 8);                                                 \
        }                                                                                                     \
    } while (0)
#define WIDE_ISSUE()                                                                                          \
    do {                                                                                                      \
        _Pragma("unroll") for (int q_ = 0; q_ < NDMA; ++q_) {                                                 \
            const unsigned lds_ = __builtin_amdgcn_readfirstlane(ring_lds + is_off + WIDE_LOAD_INDEX(q_) * 1024); \
            if (WIDE_LOAD_INDEX(q_) * 4 < H)                /* weights pass once: non-temporal */             \
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds_), "v"(src[q_]) : "m0"); \
            else                                                                                              \
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_), "v"(src[q_]) : "m0"); \
            src[q_] += WIDE_LOAD_INDEX(q_) * 4 < H ? wstep : 128;                                             \
        }                                                                                                     \
        if (--is_wrap == 0) {                              /* on to the run's first chunk */                  \
            _Pragma("unroll") for (int q_ = 0; q_ < NDMA; ++q_)                                               \
                src[q_] -= (size_t)is_len * (WIDE_LOAD_INDEX(q_) * 4 < H ? wstep : 128);                      \
        }                                                                                                     \
        ++issued;                                                                                             \
        is_off = is_off + STAGE == S * STAGE ? 0 : is_off + STAGE;                                            \
        if (--is_left == 0 && ++is_u < my_units) WIDE_SETUP();                                                \
    } while (0)

    if (my_units > 0) WIDE_SETUP();
    for (int j = 0; j < D; ++j)
        if (is_u < my_units) WIDE_ISSUE();
    if constexpr (!BRANCHES) if (scale) {
        // wave w takes the tiles w, w + 8, .. of all rows, a lane a row; the first wave adds the eight sums
        float t = 0.f;
        if (lane < M) {
#pragma unroll 8
            for (int c = wave; c < nrm.ssq_tiles; c += NW) t += nrm.ssq[(size_t)c * SSQ_LD + lane];
        }
        sq[tid] = t;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (wave == 0) {
            t = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) t += sq[w * 64 + lane];
            rstd[lane] = rsqrtf(t * nrm.inv_k + nrm.eps);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the barrier in front of the first chunk publishes it
        }
    }
    if (my_units > 0) WIDE_RUN_LENGTH(0, cp_left);
    while (cp_u < my_units) {
        // the chunk to multiply has landed when at most the loads of the chunks issued after it are in flight
        if (issued - done - 1 >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NDMA) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();            // every wave's part of it is there; the chunk before is done with
        asm volatile("" ::: "memory");
        if (is_u < my_units) WIDE_ISSUE();
        unsigned char* st = smem + cp_off;
        cp_off = cp_off + STAGE == S * STAGE ? 0 : cp_off + STAGE;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int col = 4 * (2 * khalf + ks) + g;
            const int wr = 16 * rb + r16;
            const bf16x8 wf0 = *(const bf16x8*)(st + wr * 256 + ((col ^ (wr & 7)) * 16));
            bf16x8 wf1 = wf0;
            if (TWO && has1) wf1 = *(const bf16x8*)(st + (64 + wr) * 256 + ((col ^ (wr & 7)) * 16));
#pragma unroll
            for (int j = 0; j < MB; ++j) {
                const int xr = H + 16 * j + r16;
                const bf16x8 xv = *(const bf16x8*)(st + xr * 256 + ((col ^ (xr & 7)) * 16));
                acc[0][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf0, xv, acc[0][j], 0, 0, 0);
                if (TWO && has1) acc[TWO ? 1 : 0][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf1, xv, acc[TWO ? 1 : 0][j], 0, 0, 0);
            }
        }
        ++done;
        --cp_left;
        if (BRANCHES && (cp_left == 0 || (done & 3) == 0)) {
            // a product that is cut into runs otherwise: sums of four chunks, added up, round no more than those (4,096 by 4,096,
            // 24 and 64 rows: error against 64 bits 1.06e-7 of the result, cut into runs 1.06e-7 and 1.34e-7, one chain 2.7e-7)
#pragma unroll
            for (int t = 0; t < (TWO ? 2 : 1); ++t)
#pragma unroll
                for (int j = 0; j < MB; ++j) {
                    far[t][j] += acc[t][j];
                    acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
        if (cp_left > 0) continue;
        if (BRANCHES) {
#pragma unroll
            for (int t = 0; t < (TWO ? 2 : 1); ++t)
#pragma unroll
                for (int j = 0; j < MB; ++j) {
                    acc[t][j] = far[t][j];
                    far[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
        // The unit's end: acc[t][j][r] is weight row 64 t + 16 rb + 4 g + r of the tile, batch row 16 j + r16.
        // The sums meet in the stage that was multiplied last: the next loads into it are issued after
        // the next chunk's barrier, which a wave reaches after its part of the epilogue.
        const int unit = (int)blockIdx.x + cp_u * (int)gridDim.x;
        const int part = unit % parts;
        const int n0 = (unit / parts) * H;
        if (++cp_u < my_units) WIDE_RUN_LENGTH(cp_u, cp_left);
        float* red = (float*)st;                 // [H][RLD]
        __builtin_amdgcn_s_barrier();            // every wave has read its operands of the stage
        asm volatile("" ::: "memory");
        if (khalf == 1) {
#pragma unroll
            for (int t = 0; t < (TWO ? 2 : 1); ++t)
                if (t == 0 || has1)
#pragma unroll
                    for (int j = 0; j < MB; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r) red[(64 * t + 16 * rb + 4 * g + r) * RLD + 16 * j + r16] = acc[t][j][r];
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (khalf == 0) {
#pragma unroll
            for (int t = 0; t < (TWO ? 2 : 1); ++t)
                if (t == 0 || has1)
#pragma unroll
                    for (int j = 0; j < MB; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            float* p = red + (64 * t + 16 * rb + 4 * g + r) * RLD + 16 * j + r16;
                            *p = acc[t][j][r] + *p;
                        }
        }
#pragma unroll
        for (int t = 0; t < (TWO ? 2 : 1); ++t)
#pragma unroll
            for (int j = 0; j < MB; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (mode == OUT_SWIGLU && !partial) {
            // blocks of 16 tile rows: 8 gates, then the 8 up values of the same outputs
            for (int e = tid; e < (H / 2) * 16 * MB; e += 512) {
                const int m = e / (H / 2), jl = e % (H / 2);
                const int gr = (jl >> 3) * 16 + (jl & 7);
                if (m < M && n0 + gr + 8 < N) {
                    float gv = red[gr * RLD + m];
                    float uv = red[(gr + 8) * RLD + m];
                    if (scale) { gv *= rstd[m]; uv *= rstd[m]; }
                    ((bf16*)C)[(size_t)m * ldc + n0 / 2 + jl] = (bf16)silu_mul(gv, uv);
                }
            }
        } else {
            for (int e = tid; e < H * 16 * MB; e += 512) {
                const int m = e / H, nl = e % H, n = n0 + nl;
                if (m < M && n < N) {
                    float v = red[nl * RLD + m];
                    if (scale) v *= rstd[m];
                    const size_t idx = (size_t)m * ldc + n + branch_gap(nrm, n0);
                    if (partial) ((float*)C)[part * part_stride + (size_t)m * N + n] = v;
                    else if (mode == OUT_BF16) ((bf16*)C)[idx] = (bf16)v;
                    else if (mode == OUT_F32) ((float*)C)[idx] = v;
                    else unsafeAtomicAdd((float*)C + idx, v);         // one add per element, no read to wait for
                }
            }
        }
    }
#undef WIDE_ISSUE
#undef WIDE_SETUP
#undef WIDE_LOAD_INDEX
#undef WIDE_RUN_LENGTH
}

// The shape of gemm_stream_wide's units: tile height (64 to 128 rows in steps of 16) and runs
// along k (1 to 8), the least time by a simple count: rounds of units over the compute
// units, times the run's chunks, times what a chunk costs (its weight rows and a constant for
// the activations, which come from the L2, and the barrier), plus the traffic of the partial
// sums.  Ties go to fewer runs, then to lower tiles.
static void wide_shape(int M, int N, int K, int mode, int cus, size_t scratch_bytes, int* hb_out, int* parts_out) {
    const int nch = K / 128;
    double best_cost = 1e30;
    *hb_out = 4;
    *parts_out = 1;
    for (int parts = 1; parts <= 8; ++parts) {
        if (parts > 1 && (mode == OUT_SWIGLU || parts * 2 > nch || (size_t)parts * M * N * sizeof(float) > scratch_bytes))
            break;
        const int cpp = (nch + parts - 1) / parts;
        if ((nch + cpp - 1) / cpp != parts) continue;                // it would leave a run empty
        for (int hb = 4; hb <= 8; ++hb) {
            const int h = 16 * hb;
            const long long tiles = (N + h - 1) / h;
            const long long rounds = (tiles * parts + cus - 1) / cus;
            double cost = (double)rounds * cpp * (h + 16.0);
            if (parts > 1) cost *= 1.0 + 4.0 * parts * M / K;
            if (cost < best_cost * (1.0 - 1e-9)) { best_cost = cost; *hb_out = hb; *parts_out = parts; }
        }
    }
}

// norm: 0 none; 1 the product is added into the residual rows C and prepares the next RMS norm
// (needs a split product: the sum kernel does it; refused otherwise); 2 the activations were so
// prepared and the sums are scaled (modes 0, 1, 3).  force_hb, force_parts: a tile height (in
// blocks of 16 rows) and a number of runs other than wide_shape's (tests and measurements).
// leave: the runs' sums stay in `scratch` ([runs][M][N] floats) for a consumer that adds them
// in run order itself, and *leave says how many runs; refused (nothing launched) when the
// product is not cut.
template <int MB>
static int launch_stream_wide(const bf16* A, const bf16* W, void* C, int M, int N, int K, size_t lda, size_t ldc,
                              int mode, float* scratch, size_t scratch_bytes, hipStream_t s, int norm = 0,
                              StreamNorm nrm = StreamNorm{}, int force_hb = 0, int force_parts = 0, int wl = 0,
                              int* leave = nullptr) {
    const int cus = br_device_cus();
    if (!cus) return BR_LAUNCH_FAILED;
    const int nch = K / 128;
    int hb, parts;
    wide_shape(M, N, K, mode, cus, scratch ? scratch_bytes : 0, &hb, &parts);
    if (leave && (parts < 2 || norm == 1 || force_hb || force_parts)) return BR_BAD_ARG;
    if (force_hb) {
        if (force_hb < 4 || force_hb > 8) return BR_BAD_ARG;
        hb = force_hb;
    }
    if (force_parts) {
        const int cpp_ = (nch + force_parts - 1) / force_parts;
        if (force_parts > 1 && (!scratch || mode == OUT_SWIGLU || force_parts > 8 || force_parts * 2 > nch ||
                                (nch + cpp_ - 1) / cpp_ != force_parts ||
                                (size_t)force_parts * M * N * sizeof(float) > scratch_bytes))
            return BR_BAD_ARG;
        parts = force_parts;
    }
    if (norm == 1 && (parts < 2 || N % 256 || mode != OUT_F32_ACC)) return BR_BAD_ARG;
    if (norm == 2 && mode == OUT_F32_ACC) return BR_BAD_ARG;
    const int cpp = (nch + parts - 1) / parts;
    const int h = 16 * hb, ntiles = (N + h - 1) / h;
    const long long nunits = (long long)ntiles * parts;
    const int grid = nunits < cus ? (int)nunits : cus;
    const size_t stride = (size_t)M * N;
    const int partial = parts > 1;
    void* out = partial ? (void*)scratch : C;
#define BR_WIDE(HB_)                                                                                            \
    do {                                                                                                        \
        auto kern = gemm_stream_wide_kernel<MB, HB_>;                                                           \
        constexpr size_t lds = (size_t)WIDE_S * (16 * HB_ + 16 * MB) * 256 + 9 * 64 * 4;                            \
        static_assert(lds <= 160 * 1024, "LDS of a compute unit");                                              \
        static bool set = false;                                                                                \
        if (!set) {                                                                                             \
            if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != \
                hipSuccess)                                                                                     \
                return BR_LAUNCH_FAILED;                                                                        \
            set = true;                                                                                         \
        }                                                                                                       \
        kern<<<grid, 512, lds, s>>>(A, W, out, M, N, K, lda, ldc, mode, partial, norm == 2, ntiles, parts, cpp, \
                                    stride, nrm, wl);                                                           \
    } while (0)
    switch (hb) {
        case 4: BR_WIDE(4); break;
        case 5: BR_WIDE(5); break;
        case 6: BR_WIDE(6); break;
        case 7: BR_WIDE(7); break;
        default: BR_WIDE(8); break;
    }
#undef BR_WIDE
    int rc = br_check_launch();
    if (rc != BR_OK || !partial) return rc;
    if (leave) {
        *leave = parts;
        return rc;
    }
    if (norm == 1) {
        const size_t segments = stride / 256;
        const unsigned blocks = (unsigned)((segments + 3) / 4);
        if (ldc % 4 == 0 && nrm.ldx % 4 == 0 && ((uintptr_t)C | (uintptr_t)nrm.gain) % 16 == 0 && (uintptr_t)nrm.xg % 8 == 0)
            gemm_split_sum_prep_kernel<4><<<blocks, 256, 0, s>>>(scratch, parts, stride, (float*)C, N, ldc, nrm.gain, nrm.xg, nrm.ldx, nrm.ssq, segments);
        else
            gemm_split_sum_prep_kernel<1><<<blocks, 256, 0, s>>>(scratch, parts, stride, (float*)C, N, ldc, nrm.gain, nrm.xg, nrm.ldx, nrm.ssq, segments);
        return br_check_launch();
    }
    return launch_split_sum(scratch, parts, C, M, N, ldc, mode, s);
}

// kernel: 0 = choose, 1 = tile 128x128 through registers (any shape; plus 16 b: the narrow kernel with b blocks of 16 weight rows a
// workgroup, 1, 2 or 4, aligned rows), 2 = the same 256x128,
// 3 = skinny (M <= 64), 4..6 = direct-to-LDS tiles 256x128, 128x256, 128x128 (K a multiple
// of 64, aligned rows), 7 = gemm_stream_tile (M <= 16, K a multiple of 128 and at least 1024, aligned
// rows; plus 16 b: 8 (b + 1) weight rows a workgroup, M <= 128, K from 256), 8 = stream wide (16 < M <= 64, K a multiple of 128), 9 = direct-to-LDS tile 64x128
// (M <= 64), 10 = direct-to-LDS tile 256x192, 11 = the same 256x256 (SwiGLU epilogue only), 12..15 = the tiles of
// four waves, one to a SIMD: 256x256, 128x256, 256x192, 256x224 (K a multiple of 64, aligned rows, output rows in steps
// of 16 bytes; plus 16 p: with p runs along k); tests force one.  (A 256x256 tile of 8 waves for every epilogue
// was tried: it runs out of registers in three of the four and was no faster in the fourth.)
// `wl`: the layout of W (see WL_BLOCKED; K in steps of 128 then, kernels 4 to 15).
// `scratch` (float, `scratch_bytes`; may be null) lets a product of 16 < M <= 64 rows with few
// weight rows be split along k (see gemm_split_sum_kernel); BR_GEMM_SCRATCH_BYTES always suffices.
extern "C" int br_gemm_bf16_ex(const void* A_, const void* W_, void* C, int M, int N, int K, size_t lda,
                               size_t ldc, int mode, int kernel, void* scratch, size_t scratch_bytes, int wl,
                               hipStream_t s) {
    if (M <= 0 || N <= 0) return BR_OK;
    if (K <= 0 || lda < (size_t)K || mode < 0 || mode > 3) return BR_BAD_ARG;
    if (mode == OUT_SWIGLU ? (N % 16 != 0 || ldc < (size_t)N / 2) : ldc < (size_t)N) return BR_BAD_ARG;
    // kernel / 16: a forced number of runs along k for kernels 5 and 6, or for kernel 8 a forced tile
    // height in blocks of 16 rows plus 16 times a forced number of runs (measurements and tests), 0 = by shape
    const int forced_parts = kernel >= 16 ? kernel / 16 : 0;
    kernel %= 16;
    const bf16* A = (const bf16*)A_;
    const bf16* W = (const bf16*)W_;
    const bool aligned = (K % 8 == 0) && (lda % 8 == 0) && (((uintptr_t)A | (uintptr_t)W) % 16 == 0);
    if (kernel == 3 && (!aligned || M > 64)) return BR_BAD_ARG;
    const bool dma_ok = aligned && K % DMA_BK == 0;
    const bool stream_ok = aligned && M <= 16 && K % STREAM_KC == 0 && K / STREAM_KC >= STREAM_NW;
    if (kernel >= 4 && kernel <= 6 && !dma_ok) return BR_BAD_ARG;
    const bool wide_ok = aligned && M > 16 && M <= 64 && K % 128 == 0 && K >= 256 &&
                         (!scratch || (uintptr_t)scratch % 16 == 0);
    if ((kernel == 7 && (forced_parts ? !(aligned && tile_takes(M, K, lda)) : !stream_ok)) || (kernel == 8 && !wide_ok) || kernel > 15 || kernel < 0 || (kernel >= 10 && !dma_ok) ||
        (kernel == 11 && mode != OUT_SWIGLU) ||
        (kernel == 9 && (!dma_ok || M > 64)))
        return BR_BAD_ARG;
    if (wl != WL_ROWS) {
        if (wl != WL_BLOCKED || !aligned || K % 128 || (kernel != 0 && kernel < 4)) return BR_BAD_ARG;
        if (kernel == 0 && M <= 16 && !stream_ok) return BR_BAD_ARG;      // blocked weights have K from 1024
    }
    const bool chosen = kernel == 0;
    if (chosen && wl == WL_ROWS && aligned) {
        const int blocks = narrow_blocks(M, N, K, mode, br_device_cus(), (scratch && (uintptr_t)scratch % 16 == 0) ? scratch_bytes : 0);
        if (blocks) return launch_narrow_blocks(blocks, A, W, C, M, N, K, lda, ldc, mode, s);
    }
    // Beyond 64 rows the tile kernel where it is the faster; 17 to 64 rows only when asked for a product without runs
    // (kernel 16): the sums of runs that br_gemm_bf16_wide_partial leaves are those of the product that is chosen without being asked.
    if (chosen && aligned && M > 16 && tile_takes(M, K, lda) && (M > 64 || forced_parts == 1)) {
        const int rt = tile_rows(M, N, K, mode, br_device_cus());
        if (rt) return launch_stream_tile(rt, 0, A, W, C, M, N, K, lda, ldc, mode, s, StreamNorm{}, wl);
    }
    if (kernel == 1 && forced_parts) {
        if (!aligned || wl != WL_ROWS || mode == OUT_SWIGLU || (forced_parts != 1 && forced_parts != 2 && forced_parts != 4)) return BR_BAD_ARG;
        return launch_narrow_blocks(forced_parts, A, W, C, M, N, K, lda, ldc, mode, s);
    }
    if (kernel == 0)
        kernel = stream_ok ? 7
                 : wide_ok ? 8
                 : (aligned && M <= 64) ? (wl ? 9 : 3) : (!dma_ok ? 1 : (N > 128 ? 5 : 6));
    if (kernel == 9) return launch_tile_dma<64, 128, 1, 4, 3>(A, W, C, M, N, K, lda, ldc, mode, s, 1, nullptr, wl);
    if (kernel == 8) {
        const int fh = chosen ? 0 : forced_parts % 16, fp = chosen ? 0 : forced_parts / 16;
        return M <= 32 ? launch_stream_wide<2>(A, W, C, M, N, K, lda, ldc, mode, (float*)scratch, scratch_bytes, s, 0,
                                               StreamNorm{}, fh, fp, wl)
                       : launch_stream_wide<4>(A, W, C, M, N, K, lda, ldc, mode, (float*)scratch, scratch_bytes, s, 0,
                                               StreamNorm{}, fh, fp, wl);
    }
    if (kernel == 7 && !chosen && forced_parts) {      // 7 + 16 b: a workgroup a tile of 8 (b + 1) weight rows, b = 1, 2, 3
        return launch_stream_tile(8 * (forced_parts + 1), 0, A, W, C, M, N, K, lda, ldc, mode, s, StreamNorm{}, wl);
    }
    if (kernel == 7) {
        const int cus = br_device_cus();
        if (resident_pays(N, K, mode, cus))
            return M <= 8 ? launch_stream<8, 0>(A, W, C, M, N, K, lda, ldc, mode, s, StreamNorm{}, wl)
                          : launch_stream<16, 0>(A, W, C, M, N, K, lda, ldc, mode, s, StreamNorm{}, wl);
        return launch_stream_tile(tile_rows(M, N, K, mode, cus), 0, A, W, C, M, N, K, lda, ldc, mode, s, StreamNorm{}, wl);
    }
    int parts = 1;
    if (chosen && M > 128 && (kernel == 5 || kernel == 6) && quad_takes(C, M, N, K, lda, ldc)) {
        // More than 128 rows, K in steps of 64: the tiles of one wave per SIMD, where the product's addresses
        // allow.  (Up to 128 rows the tiles of eight waves below stream the weights faster: 7B shapes at 128
        // rows, gate/up 59 against 69 us, the 32,768-row head 71 against 85, down 39 against 45.)
        const int cus = br_device_cus();
        const size_t room = (scratch && (uintptr_t)scratch % 16 == 0) ? scratch_bytes : 0;
        if (cus > 0) {
            const double single = choose_quad(M, N, K, mode, cus, room, &kernel, &parts);
            int k2, p2;
            const int n1 = quad_whole_rounds(M, N, K, mode, cus, room, single, &k2, &p2);
            if (n1 > 0) {
                // whole rounds of the 256x256 tile over the first n1 weight rows, then the rest; n1 rows on
                // is the same number of elements in either weight layout (n1 is a multiple of 16)
                int rc = launch_tile_quad<256, 256, QUAD12>(A, W, C, M, n1, K, lda, ldc, mode, s, wl);
                if (rc != BR_OK) return rc;
                const bf16* W2 = W + (size_t)n1 * K;
                void* C2 = mode == OUT_SWIGLU ? (void*)((bf16*)C + n1 / 2)
                           : mode == OUT_BF16 ? (void*)((bf16*)C + n1) : (void*)((float*)C + n1);
                const int N2 = N - n1;
                if (k2 == 12) return launch_tile_quad<256, 256, QUAD12>(A, W2, C2, M, N2, K, lda, ldc, mode, s, wl, p2, (float*)scratch);
                if (k2 == 13) return launch_tile_quad<128, 256, QUAD13>(A, W2, C2, M, N2, K, lda, ldc, mode, s, wl, p2, (float*)scratch);
                if (k2 == 15) return launch_tile_quad<256, 224, 2, 3, 4>(A, W2, C2, M, N2, K, lda, ldc, mode, s, wl, p2, (float*)scratch);
                return launch_tile_quad<256, 192, QUAD14>(A, W2, C2, M, N2, K, lda, ldc, mode, s, wl, p2, (float*)scratch);
            }
        }
    }
    if (chosen && (kernel == 5 || kernel == 6)) {
        const int cus = br_device_cus();
        if (cus > 0) choose_tile(M, N, K, mode, cus, (scratch && (uintptr_t)scratch % 16 == 0) ? scratch_bytes : 0, &kernel, &parts);
    }
    if (chosen && mode == OUT_SWIGLU && kernel == 5 && parts == 1) {
        // The 256x256 tile over as many weight rows as make whole rounds of it, the 128x256 tile over the rest,
        // where the count says that this is faster than 128x256 over all of them (2,048 x 28,672: three
        // rounds of 256x256 over 24,576 rows and one round of 128x256 over 4,096, instead of seven of 128x256).
        const int cus = br_device_cus();
        const int tm11 = (M + 255) / 256, nk = K / DMA_BK;
        const int cols = cus > 0 ? cus / tm11 : 0;                   // tile columns of one round
        if (cols > 0) {
            const long long n_round = (long long)cols * 256;
            const long long r11 = N / n_round, n1 = r11 * n_round, n2 = N - n1;
            const long long t5_all = ((long long)((M + 127) / 128) * ((N + 255) / 256) + cus - 1) / cus;
            const long long t5_rest = ((long long)((M + 127) / 128) * ((n2 + 255) / 256) + cus - 1) / cus;
            const double whole = (double)t5_all * nk * 1.14;
            const double split = (double)r11 * nk * 2.05 + (double)t5_rest * nk * 1.14 + 5.0;
            if (r11 >= 1 && n2 > 0 && n2 % 16 == 0 && split < 0.97 * whole) {
                gemm_tile_dma_kernel<256, 256, 2, 4, 2, OUT_SWIGLU><<<(unsigned)(tm11 * (int)(n1 / 256)), 512, 0, s>>>(
                    A, W, C, M, (int)n1, K, lda, ldc, tm11, (int)(n1 / 256), nk, 0, wl);
                int rc = br_check_launch();
                if (rc != BR_OK) return rc;
                // n1 rows on: the same number of elements in either weight layout (n1 is a multiple of 16)
                return launch_tile_dma<128, 256, 2, 4, 3>(A, W + (size_t)n1 * K, (bf16*)C + n1 / 2, M, (int)n2, K, lda, ldc,
                                                          mode, s, 1, nullptr, wl);
            }
        }
    }
    if (kernel >= 12 && forced_parts > 1) {
        if (!scratch || (uintptr_t)scratch % 16 || (size_t)forced_parts * M * N * sizeof(float) > scratch_bytes ||
            forced_parts * 2 > K / DMA_BK)
            return BR_BAD_ARG;
        parts = forced_parts;
    }
    if (kernel == 12) return launch_tile_quad<256, 256, QUAD12>(A, W, C, M, N, K, lda, ldc, mode, s, wl, parts, (float*)scratch);
    if (kernel == 13) return launch_tile_quad<128, 256, QUAD13>(A, W, C, M, N, K, lda, ldc, mode, s, wl, parts, (float*)scratch);
    if (kernel == 14) return launch_tile_quad<256, 192, QUAD14>(A, W, C, M, N, K, lda, ldc, mode, s, wl, parts, (float*)scratch);
    if (kernel == 15) return launch_tile_quad<256, 224, 2, 3, 4>(A, W, C, M, N, K, lda, ldc, mode, s, wl, parts, (float*)scratch);
    if (kernel == 10) return launch_tile_dma<256, 192, 4, 2, 2>(A, W, C, M, N, K, lda, ldc, mode, s, 1, nullptr, wl);
    if (kernel == 11) {
        gemm_tile_dma_kernel<256, 256, 2, 4, 2, OUT_SWIGLU><<<(unsigned)(((M + 255) / 256) * ((N + 255) / 256)), 512, 0, s>>>(
            A, W, C, M, N, K, lda, ldc, (M + 255) / 256, (N + 255) / 256, K / DMA_BK, 0, wl);
        return br_check_launch();
    }
    if (forced_parts > 1 && (kernel == 5 || kernel == 6)) {
        if (!scratch || (uintptr_t)scratch % 16 || (size_t)forced_parts * M * N * sizeof(float) > scratch_bytes ||
            forced_parts > K / DMA_BK)
            return BR_BAD_ARG;
        parts = forced_parts;
    }
    if (kernel == 4) return launch_tile_dma<256, 128, 4, 2, 3>(A, W, C, M, N, K, lda, ldc, mode, s, 1, nullptr, wl);
    if (kernel == 5) return launch_tile_dma<128, 256, 2, 4, 3>(A, W, C, M, N, K, lda, ldc, mode, s, parts, (float*)scratch, wl);
    if (kernel == 6) return launch_tile_dma<128, 128, 2, 2, 2>(A, W, C, M, N, K, lda, ldc, mode, s, parts, (float*)scratch, wl);
    if (kernel == 3) {
        // shapes measured on cold weights (cycled through more than the 256 MB cache)
        const bool wide = N >= 16384;
        if (M <= 16) return (wide && M > 4) ? launch_skinny<1, 1, 2, 8>(A, W, C, M, N, K, lda, ldc, mode, s)
                                            : launch_skinny<1, 1, 4, 8>(A, W, C, M, N, K, lda, ldc, mode, s);
        const int parts = (scratch && (uintptr_t)scratch % 16 == 0) ? split_parts(M, N, K, mode, scratch_bytes) : 1;
        if (parts > 1)
            return M <= 32 ? launch_split<2>(A, W, C, M, N, K, lda, ldc, mode, parts, (float*)scratch, s)
                           : launch_split<4>(A, W, C, M, N, K, lda, ldc, mode, parts, (float*)scratch, s);
        if (M <= 32) return wide ? launch_skinny_lds<2, 4>(A, W, C, M, N, K, lda, ldc, mode, s)
                                 : launch_skinny_lds<2, 1>(A, W, C, M, N, K, lda, ldc, mode, s);
        if (wide) return dma_ok ? launch_tile_dma<64, 128, 1, 4, 3>(A, W, C, M, N, K, lda, ldc, mode, s)
                                : launch_skinny_lds<4, 4>(A, W, C, M, N, K, lda, ldc, mode, s);
        return (N >= 6144) ? launch_skinny_lds<4, 2>(A, W, C, M, N, K, lda, ldc, mode, s)
                           : launch_skinny_lds<4, 1>(A, W, C, M, N, K, lda, ldc, mode, s);
    }
    if (kernel == 2) return launch_tile<256, 128, 32, 2, 2>(A, W, C, M, N, K, lda, ldc, mode, aligned, s);
    return launch_tile<128, 128, 64, 2, 2>(A, W, C, M, N, K, lda, ldc, mode, aligned, s);
}

extern "C" int br_gemm_bf16(const void* A, const void* W, void* C, int M, int N, int K, size_t lda, size_t ldc,
                            int mode, hipStream_t s) {
    return br_gemm_bf16_ex(A, W, C, M, N, K, lda, ldc, mode, 0, nullptr, 0, WL_ROWS, s);
}

// What br_gemm_bf16_ex picks for a product of more than 64 rows with K in steps of 64, aligned rows of the plain layout and a
// contiguous, aligned output (tests and benchmarks ask): the kernel and its runs along k; and, where the product is
// cut along its weight rows, `n1` > 0 rows by the 256x256 tile first and `kernel`, `parts` for the rest.  The narrow kernel is
// kernel 1 with its blocks of 16 weight rows as `parts`.
extern "C" int br_gemm_bf16_tile_choice(int M, int N, int K, int mode, size_t scratch_bytes, int* kernel, int* parts,
                                        int* n1) {
    const int cus = br_device_cus();
    if (!cus) return BR_LAUNCH_FAILED;
    *n1 = 0;
    *parts = narrow_blocks(M, N, K, mode, cus, scratch_bytes);
    if (*parts) {
        *kernel = 1;
        return BR_OK;
    }
    if (M > 64 && tile_takes(M, K, (size_t)K) && tile_rows(M, N, K, mode, cus)) {
        *kernel = 7;
        *parts = 1;
        return BR_OK;
    }
    if (M > 128 && quad_takes(nullptr, M, N, K, (size_t)K, (size_t)(mode == OUT_SWIGLU ? N / 2 : N))) {
        const double single = choose_quad(M, N, K, mode, cus, scratch_bytes, kernel, parts);
        int k2, p2;
        const int rows = quad_whole_rounds(M, N, K, mode, cus, scratch_bytes, single, &k2, &p2);
        if (rows > 0) {
            *n1 = rows;
            *kernel = k2;
            *parts = p2;
        }
        return BR_OK;
    }
    choose_tile(M, N, K, mode, cus, scratch_bytes, kernel, parts);
    return BR_OK;
}

// Whether a product of up to 128 aligned rows goes to gemm_stream_tile (17 to 64 rows: when asked for one without runs).
extern "C" int br_gemm_bf16_whole_pays(int M, int N, int K, int by16) {
    const int cus = br_device_cus();
    return tile_rows(M, N, K, OUT_BF16, cus, by16 != 0) != 0 && (M > 16 || !resident_pays(N, K, OUT_BF16, cus));
}

static bool stream_takes(const void* A, const void* W, int M, int K, size_t lda) {
    return M > 0 && M <= 16 && K % STREAM_KC == 0 && K / STREAM_KC >= STREAM_NW && lda % 8 == 0 && lda >= (size_t)K &&
           ((uintptr_t)A | (uintptr_t)W) % 16 == 0;
}
static bool wide_takes(const void* A, const void* W, int M, int K, size_t lda) {
    return M > 16 && M <= 64 && K % 128 == 0 && K >= 256 && lda % 8 == 0 && lda >= (size_t)K &&
           ((uintptr_t)A | (uintptr_t)W) % 16 == 0;
}

// C += A W^T through the streaming products, which then also prepare the RMS norm that reads C
// next: xg[M, ldx] = bf16(C * gain) and sums of squares in ssq[tiles, SSQ_LD] (see the kernels);
// *ssq_tiles says how many.  Up to 16 rows: gemm_stream (N in steps of 16).  17 to 64 rows:
// gemm_stream_wide cut along k, the preparation in the sum kernel (N in steps of 256, scratch
// needed).  Refuses (BR_BAD_ARG) anything else: the caller then runs the norm itself.
extern "C" int br_gemm_bf16_norm_prepare(const void* A, const void* W, float* C, int M, int N, int K, size_t lda,
                                         size_t ldc, const float* gain, void* xg, size_t ldx, float* ssq,
                                         int* ssq_tiles, void* scratch, size_t scratch_bytes, int wl, int whole, hipStream_t s) {
    if (M <= 0 || N <= 0 || (wl != WL_ROWS && wl != WL_BLOCKED)) return BR_BAD_ARG;
    if (ldc < (size_t)N || ldx < (size_t)N || !gain || !xg || !ssq || !ssq_tiles) return BR_BAD_ARG;
    StreamNorm nrm{gain, (bf16*)xg, ldx, ssq, 0, 0.f, 0.f};
    if (N % 16 == 0 && M <= 64 && (stream_takes(A, W, M, K, lda) || (whole && wide_takes(A, W, M, K, lda)))) {
        const int rt = tile_norms(M, N, K, br_device_cus()) ? tile_rows(M, N, K, OUT_F32_ACC, br_device_cus(), true) : 0;
        if (rt) {
            *ssq_tiles = N / 16;
            return launch_stream_tile(rt, 1, (const bf16*)A, (const bf16*)W, C, M, N, K, lda, ldc, OUT_F32_ACC, s, nrm, wl);
        }
    }
    if (stream_takes(A, W, M, K, lda) && N % 16 == 0) {
        *ssq_tiles = N / 16;
        return M <= 8 ? launch_stream<8, 1>((const bf16*)A, (const bf16*)W, C, M, N, K, lda, ldc, OUT_F32_ACC, s, nrm, wl)
                      : launch_stream<16, 1>((const bf16*)A, (const bf16*)W, C, M, N, K, lda, ldc, OUT_F32_ACC, s, nrm, wl);
    }
    if (wide_takes(A, W, M, K, lda) && N % 256 == 0 && scratch && (uintptr_t)scratch % 16 == 0) {
        *ssq_tiles = N / 256;
        return M <= 32 ? launch_stream_wide<2>((const bf16*)A, (const bf16*)W, C, M, N, K, lda, ldc, OUT_F32_ACC,
                                               (float*)scratch, scratch_bytes, s, 1, nrm, 0, 0, wl)
                       : launch_stream_wide<4>((const bf16*)A, (const bf16*)W, C, M, N, K, lda, ldc, OUT_F32_ACC,
                                               (float*)scratch, scratch_bytes, s, 1, nrm, 0, 0, wl);
    }
    return BR_BAD_ARG;
}

// C = rsqrt(sum of the ssq tiles / norm_width + eps) * (XG W^T), XG and ssq from br_gemm_bf16_norm_prepare:
// the product of the normed rows.  mode: 0 bf16, 1 float, 3 SwiGLU.
extern "C" int br_gemm_bf16_norm_scaled(const void* XG, const void* W, void* C, int M, int N, int K, size_t lda,
                                        size_t ldc, int mode, const float* ssq, int ssq_tiles, int norm_width,
                                        float eps, void* scratch, size_t scratch_bytes, int wl, int whole, hipStream_t s) {
    if (M <= 0 || N <= 0) return BR_OK;
    if (wl != WL_ROWS && wl != WL_BLOCKED) return BR_BAD_ARG;
    if (!ssq || ssq_tiles <= 0 || norm_width <= 0 || (mode != OUT_BF16 && mode != OUT_F32 && mode != OUT_SWIGLU))
        return BR_BAD_ARG;
    if (mode == OUT_SWIGLU ? (N % 16 != 0 || ldc < (size_t)N / 2) : ldc < (size_t)N) return BR_BAD_ARG;
    StreamNorm nrm{nullptr, nullptr, 0, (float*)ssq, ssq_tiles, 1.f / (float)norm_width, eps};
    if (M <= 64 && (stream_takes(XG, W, M, K, lda) || (whole && wide_takes(XG, W, M, K, lda)))) {
        const int rt = tile_norms(M, N, K, br_device_cus()) ? tile_rows(M, N, K, mode, br_device_cus()) : 0;
        if (rt) return launch_stream_tile(rt, 2, (const bf16*)XG, (const bf16*)W, C, M, N, K, lda, ldc, mode, s, nrm, wl);
    }
    if (stream_takes(XG, W, M, K, lda))
        return M <= 8 ? launch_stream<8, 2>((const bf16*)XG, (const bf16*)W, C, M, N, K, lda, ldc, mode, s, nrm, wl)
                      : launch_stream<16, 2>((const bf16*)XG, (const bf16*)W, C, M, N, K, lda, ldc, mode, s, nrm, wl);
    if (wide_takes(XG, W, M, K, lda)) {
        float* sc = (scratch && (uintptr_t)scratch % 16 == 0) ? (float*)scratch : nullptr;
        return M <= 32 ? launch_stream_wide<2>((const bf16*)XG, (const bf16*)W, C, M, N, K, lda, ldc, mode, sc,
                                               scratch_bytes, s, 2, nrm, 0, 0, wl)
                       : launch_stream_wide<4>((const bf16*)XG, (const bf16*)W, C, M, N, K, lda, ldc, mode, sc,
                                               scratch_bytes, s, 2, nrm, 0, 0, wl);
    }
    return BR_BAD_ARG;
}

// Several products in one launch: C[m, col(n)] = sum_k A[b][m, k] W[n, k] with b = n / per the branch of weight row n, A[b] the
// branch's rows b a_step elements behind the first's, and col(n) = n, or n + gap from n = gap_at on; float results, up to 64
// rows.  A mixer's projections of inputs that differ are four launches otherwise, each with its own ramp and, from 17 rows on, a
// second launch for the sums of its runs along k: four of 4,096 by 4,096, weights in no cache,
// 6 rows 34.4 -> 21.4 us, 24 rows 58.6 -> 23.5, 64 rows 60.0 -> 27.9; four of 2,048 by 2,048 20.4 -> 7.7, 39.0 -> 8.3, 46.0 -> 10.9.
template <int MB, int HB>
static int launch_branches_wide(const bf16* A, const bf16* W, float* C, int M, int N, int K, size_t lda, size_t ldc, const StreamBranches& br, int cus,
                                hipStream_t s) {
    auto kern = gemm_stream_wide_kernel<MB, HB, true>;
    constexpr size_t lds = (size_t)WIDE_S * (16 * HB + 16 * MB) * 256 + 64 * 4;
    static bool set = false;
    if (!set) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) return BR_LAUNCH_FAILED;
        set = true;
    }
    const int ntiles = N / (16 * HB);
    kern<<<ntiles < cus ? ntiles : cus, 512, lds, s>>>(A, W, C, M, N, K, lda, ldc, OUT_F32, 0, 0, ntiles, 1, K / 128, 0, br, WL_ROWS);
    return br_check_launch();
}

extern "C" int br_gemm_bf16_branches_takes(int M, int per, int K) {
    return M > 0 && M <= 64 && per > 0 && per % 128 == 0 && K % STREAM_KC == 0 && K / STREAM_KC >= STREAM_NW;
}

// Beyond 128 rows the branches make one product of whole 256-wide columns of tiles (256x256, 128x256).  `room`: the bytes of scratch that a product
// for each would be given.  Where that would be cut into runs along k, the tiles of 128 rows add up the same runs (`run` k-tiles each;
// one chain over all of K rounds more: 4,096 by 4,096, 300 rows: error against 64 bits 4.0e-7 of the result, four runs 1.9e-7), so that the
// bits are those of the products one by one.  Taken where it is counted faster, which it was at every size timed: few tiles need no sum kernels, many
// fill their rounds.  Four of 4,096 by 4,096, us by 129 / 300 / 512 / 640 / 1,024 / 1,801 / 3,000 / 7,000 rows one by one 94 / 114 / 140 / 166 / 184 / 234 / 369 /
// 786, at once 68 / 65 / 72 / 118 / 131 / 206 / 319 / 740 (as one chain 55 / 60 / 67 / 84 / 109 up to 1,024); of 2,048 by 2,048 66 / 72 / 82 / 88 / 122 / 115 / 126 / 224 and
// 43 / 37 / 40 / 40 / 38 / 56 / 104 / 228.  A run costs about 2 us besides its k-tiles: the ring starts anew.
static int branches_tile(int M, int branches, int per, int K, size_t room, int cus, int* run) {       // 12, 13, or 0: a product for each
    if (M <= 128 || branches < 2 || branches > 64 || per <= 0 || per % 256 || K <= 0 || K % DMA_BK || (long long)branches * per > 0x3fffffff || cus <= 0) return 0;
    const int nk = K / DMA_BK, N = branches * per;
    if (!quad_takes(nullptr, M, N, K, (size_t)K, 4)) return 0;
    int k, p, rest_k, rest_p;
    const double one = choose_quad(M, per, K, OUT_F32, cus, room, &k, &p);
    if (quad_whole_rounds(M, per, K, OUT_F32, cus, room, one, &rest_k, &rest_p)) {
        if (rest_p > 1) return 0;                                    // columns with runs and columns without
        p = 1;
    }
    int kpp = (nk + p - 1) / p;
    kpp += kpp & 1;
    *run = p > 1 ? kpp : nk;
    const double tall = p > 1 ? 1e30 : quad_count(M, N, K, OUT_F32, cus, 0, 1);
    const double flat = quad_count(M, N, K, OUT_F32, cus, 1, 1) + (p > 1 ? 2.0 * p : 0.0);
    if (min(tall, flat) >= branches * one) return 0;
    return tall <= flat ? 12 : 13;
}
extern "C" int br_gemm_bf16_branches_pay(int M, int branches, int per, int K, size_t room) {
    int run;
    return branches_tile(M, branches, per, K, room, br_device_cus(), &run) != 0;
}

template <int BM, int NSA, int NSB>
static int launch_branches_tiles(const bf16* A, const bf16* W, float* C, int M, int N, int K, size_t lda, size_t ldc, QuadBranches br, int run, hipStream_t s) {
    const int tm = (M + BM - 1) / BM, tn = N / 256;
    if ((long long)tm * tn > 0x7fffffffLL) return BR_BAD_ARG;
    br.whole = (long long)tm * tn <= br_device_cus();
    gemm_tile_quad_kernel<BM, 256, NSA, NSB, 2, OUT_F32, QUAD_BRANCHES><<<(unsigned)(tm * tn), 256, 0, s>>>(A, W, C, M, N, K, lda, ldc, tm, tn, run, 0, WL_ROWS, br);
    return br_check_launch();
}

// tail_rows > 0 (up to 16 rows, in steps of 16, at most per): further weight rows, multiplying one more branch's activations, the
// tanh of whose sums goes to tail [M, tail_ld]: instead of two launches of their own, 8.4 us of a single-token step a layer.
extern "C" int br_gemm_bf16_branches(const void* A_, const void* W_, float* C, int M, int branches, int per, int K, size_t a_step, size_t lda,
                                     size_t ldc, int gap_at, int gap, int tail_rows, void* tail, size_t tail_ld, size_t room, hipStream_t s) {
    const bf16 *A = (const bf16*)A_, *W = (const bf16*)W_;
    int run;
    if (const int kind = branches_tile(M, branches, per, K, room, br_device_cus(), &run)) {
        if (tail_rows || lda < (size_t)K || lda % 8 || a_step % 8 || gap < 0 || gap % 4 || gap_at < 0 || gap_at % per || ldc < (size_t)branches * per + gap ||
            ((uintptr_t)A | (uintptr_t)W) % 16 || !quad_takes(C, M, branches * per, K, lda, ldc))
            return BR_BAD_ARG;
        const QuadBranches br = {per, a_step, gap_at, gap, 0};
        return kind == 12 ? launch_branches_tiles<256, QUAD12>(A, W, C, M, branches * per, K, lda, ldc, br, run, s)
                          : launch_branches_tiles<128, QUAD13>(A, W, C, M, branches * per, K, lda, ldc, br, run, s);
    }
    if (branches < 1 || branches > 64 || !br_gemm_bf16_branches_takes(M, per, K) || lda < (size_t)K || lda % 8 || a_step % 8 || gap < 0 ||
        gap_at % per || ((uintptr_t)A | (uintptr_t)W) % 16 || ldc < (size_t)branches * per || (long long)branches * per > 0x3fffffff)
        return BR_BAD_ARG;
    if (tail_rows && (M > 16 || tail_rows < 0 || tail_rows > per || tail_rows % 16 || !tail || tail_ld < (size_t)tail_rows)) return BR_BAD_ARG;
    const int N = branches * per, cus = br_device_cus();
    if (!cus) return BR_LAUNCH_FAILED;
    const StreamBranches br = {per, a_step, gap_at, gap, tail_rows ? N : 0x7fffffff, (bf16*)tail, tail_ld};
    // Tiles of one round also beyond 16 rows (four of 2,048 by 2,048: 24 rows 11.6 -> 8.3 us, 64 rows 15.0 -> 10.9); four of 4,096 by 4,096 by 24 and 64
    // rows stay with the shared activations (23.6 and 27.8, by tiles 25 and 34).
    if (M <= 16 || N <= 32 * cus) {
        const int rt = tile_rows(M <= 16 ? M : 1, N, K, OUT_F32, cus, true);
#define BR_BRANCH_TILE(MB_)                                                                                                              \
    return rt == 16 || tail_rows ? launch_tile_form<16, MB_, 3>(A, W, C, M, N + tail_rows, K, lda, ldc, OUT_F32, s, br, WL_ROWS)          \
                                 : launch_tile_form<32, MB_, 3>(A, W, C, M, N, K, lda, ldc, OUT_F32, s, br, WL_ROWS)
        if (M <= 16) BR_BRANCH_TILE(1);
        if (M <= 32) BR_BRANCH_TILE(2);
        if (M <= 48) BR_BRANCH_TILE(3);
        BR_BRANCH_TILE(4);
#undef BR_BRANCH_TILE
    }
    // units of 64 rows, or of 128 where these fill the chip's rounds better (a unit's chunk costs its rows and 16 more, as in wide_shape)
    const long long r64 = (N / 64 + cus - 1) / cus, r128 = (N / 128 + cus - 1) / cus;
    if (r128 * 144 < r64 * 80)
        return M <= 32 ? launch_branches_wide<2, 8>(A, W, C, M, N, K, lda, ldc, br, cus, s)
                       : launch_branches_wide<4, 8>(A, W, C, M, N, K, lda, ldc, br, cus, s);
    return M <= 32 ? launch_branches_wide<2, 4>(A, W, C, M, N, K, lda, ldc, br, cus, s)
                   : launch_branches_wide<4, 4>(A, W, C, M, N, K, lda, ldc, br, cus, s);
}

// The runs along k of A W^T (65 to 1,024 rows, a product meant to be added into float rows), left in `scratch` as [*runs][M][N] floats for
// br_gemm_bf16_add_runs_norm, where br_gemm_bf16_ex would cut the product.  Refuses (BR_BAD_ARG, nothing launched) where it would not,
// and more than 8,192 columns.  whole: a product that gemm_stream_tile takes is left, too, as one run.
extern "C" int br_gemm_bf16_leave_runs(const void* A_, const void* W_, int M, int N, int K, size_t lda, void* scratch_, size_t scratch_bytes, int wl,
                                       int whole, int* runs, hipStream_t s) {
    const bf16 *A = (const bf16*)A_, *W = (const bf16*)W_;
    float* scratch = (float*)scratch_;
    if (M <= 64 || M > 1024 || N <= 64 || N > 8192 || N % 4 || K <= 0 || K % DMA_BK || lda < (size_t)K || lda % 8 || !scratch || !runs ||
        ((uintptr_t)A | (uintptr_t)W | (uintptr_t)scratch) % 16 || (wl != WL_ROWS && (wl != WL_BLOCKED || K % 128)))
        return BR_BAD_ARG;
    const int cus = br_device_cus(), mode = OUT_F32_ACC;
    if (!cus) return BR_LAUNCH_FAILED;
    const int rt = tile_takes(M, K, lda) ? tile_rows(M, N, K, mode, cus) : 0;
    if (rt) {
        if (!whole || (size_t)M * N * sizeof(float) > scratch_bytes) return BR_BAD_ARG;
        *runs = 1;
        return launch_stream_tile(rt, 0, A, W, scratch, M, N, K, lda, N, OUT_F32, s, StreamNorm{}, wl);
    }
    int kernel = 0, parts = 1, k2, p2;
    if (M > 128 && quad_takes(scratch, M, N, K, lda, N)) {
        const double single = choose_quad(M, N, K, mode, cus, scratch_bytes, &kernel, &parts);
        if (quad_whole_rounds(M, N, K, mode, cus, scratch_bytes, single, &k2, &p2) > 0) return BR_BAD_ARG;
    } else choose_tile(M, N, K, mode, cus, scratch_bytes, &kernel, &parts);
    if (parts < 2) return BR_BAD_ARG;
    if (kernel == 12) return launch_tile_quad<256, 256, QUAD12>(A, W, scratch, M, N, K, lda, N, mode, s, wl, parts, scratch, runs);
    if (kernel == 13) return launch_tile_quad<128, 256, QUAD13>(A, W, scratch, M, N, K, lda, N, mode, s, wl, parts, scratch, runs);
    if (kernel == 14) return launch_tile_quad<256, 192, QUAD14>(A, W, scratch, M, N, K, lda, N, mode, s, wl, parts, scratch, runs);
    if (kernel == 15) return launch_tile_quad<256, 224, 2, 3, 4>(A, W, scratch, M, N, K, lda, N, mode, s, wl, parts, scratch, runs);
    if (kernel == 5) return launch_tile_dma<128, 256, 2, 4, 3>(A, W, scratch, M, N, K, lda, N, mode, s, parts, scratch, wl, runs);
    if (kernel == 6) return launch_tile_dma<128, 128, 2, 2, 2>(A, W, scratch, M, N, K, lda, N, mode, s, parts, scratch, wl, runs);
    return BR_BAD_ARG;
}

// C += the runs [runs][M][N] in run order, and h[M, ldh] = bf16(C gain / rms(C)).
extern "C" int br_gemm_bf16_add_runs_norm(const float* sums, int runs, float* C, int M, int N, size_t ldc, const float* gain, float eps, void* h,
                                          size_t ldh, hipStream_t s) {
    if (M <= 0) return BR_OK;
    if (N <= 0 || N > 8192 || N % 4 || runs < 1 || ldc < (size_t)N || ldc % 4 || ldh < (size_t)N || ldh % 4 ||
        ((uintptr_t)sums | (uintptr_t)C | (uintptr_t)gain | (uintptr_t)h) % 16)
        return BR_BAD_ARG;
    const size_t stride = (size_t)M * N;
    const int threads = N >= 4096 ? 1024 : (N / 4 + 63) / 64 * 64;
    if (N <= 4096) gemm_split_sum_norm_kernel<1><<<M, threads, 0, s>>>(sums, runs, stride, C, N, ldc, gain, eps, (bf16*)h, ldh);
    else gemm_split_sum_norm_kernel<2><<<M, threads, 0, s>>>(sums, runs, stride, C, N, ldc, gain, eps, (bf16*)h, ldh);
    return br_check_launch();
}

// The float sums of the runs of A W^T (17 to 64 rows, bf16 result meant), left in `scratch` as
// [*parts][M][N] for a consumer that adds them in run order and rounds, which gives the bits of
// br_gemm_bf16 (or, with ssq, of br_gemm_bf16_norm_scaled) without the sum kernel's launch.
// Refuses (BR_BAD_ARG, nothing launched) where those would not cut the product.
extern "C" int br_gemm_bf16_wide_partial(const void* A, const void* W, int M, int N, int K, size_t lda,
                                         const float* ssq, int ssq_tiles, int norm_width, float eps, void* scratch,
                                         size_t scratch_bytes, int wl, int* parts, hipStream_t s) {
    if (M <= 16 || M > 64 || N <= 0 || !parts || (wl != WL_ROWS && wl != WL_BLOCKED)) return BR_BAD_ARG;
    if (!scratch || (uintptr_t)scratch % 16 || !wide_takes(A, W, M, K, lda)) return BR_BAD_ARG;
    if (ssq && (ssq_tiles <= 0 || norm_width <= 0)) return BR_BAD_ARG;
    if (!ssq && wl == WL_ROWS && narrow_blocks(M, N, K, OUT_BF16, br_device_cus(), scratch_bytes)) return BR_BAD_ARG;
    StreamNorm nrm{};
    if (ssq) nrm = StreamNorm{nullptr, nullptr, 0, (float*)ssq, ssq_tiles, 1.f / (float)norm_width, eps};
    const int norm = ssq ? 2 : 0;
    return M <= 32 ? launch_stream_wide<2>((const bf16*)A, (const bf16*)W, nullptr, M, N, K, lda, (size_t)N, OUT_BF16,
                                           (float*)scratch, scratch_bytes, s, norm, nrm, 0, 0, wl, parts)
                   : launch_stream_wide<4>((const bf16*)A, (const bf16*)W, nullptr, M, N, K, lda, (size_t)N, OUT_BF16,
                                           (float*)scratch, scratch_bytes, s, norm, nrm, 0, 0, wl, parts);
}

// into how many runs along k br_gemm_bf16_ex and br_gemm_bf16_norm_prepare cut a product of 17 to 64 rows
extern "C" int br_gemm_bf16_wide_parts(int M, int N, int K, int mode, size_t scratch_bytes) {
    const int cus = br_device_cus();
    if (!cus || M <= 16 || M > 64 || K % 128 || K < 256) return 0;
    if (narrow_blocks(M, N, K, mode, cus, scratch_bytes)) return 1;
    int hb, parts;
    wide_shape(M, N, K, mode, cus, scratch_bytes, &hb, &parts);
    return parts;
}

// ------------------------------------------- routed experts by the quad tiles -----
// Steps whose (token, slot) pairs are grouped by expert: C[p, :] = W[e] A[p, :] for every expert's pairs, all
// experts in one launch of gemm_tile_quad_kernel (GROUPED).  `gated`: W is [E][2 F][K], C bfloat16 [pairs, F] (N = 2 F), the
// rows of A taken through `order` (A below 4 GB); else W is [E][N][K] and C float32 or bfloat16 [pairs, N].
extern "C" int br_experts_tiles_takes(int N, int K) { return N > 0 && K > 0 && N % 16 == 0 && K % DMA_BK == 0; }

template <int BM, int BN, int NSA, int NSB, int WVM>
static int launch_experts_tiles(const bf16* A, const bf16* W, void* C, int mode, int pairs, int N, int K, size_t ldc, const QuadGroups& gr,
                                hipStream_t s) {
    // no more tiles than the pairs make when every expert's last one is nearly empty
    const int tn = (N + BN - 1) / BN, nk = K / DMA_BK;
    const long long tm = (long long)pairs / BM + (gr.experts < pairs ? gr.experts : pairs);
    if (tm * tn > 0x7fffffc0LL) return BR_BAD_ARG;
    const unsigned grid = (unsigned)((tm * tn + 7) / 8 * 8);
#define BR_EXPERTS(MODE_) \
    gemm_tile_quad_kernel<BM, BN, NSA, NSB, WVM, MODE_, QUAD_EXPERTS><<<grid, 256, 0, s>>>(A, W, C, 0, N, K, (size_t)K, ldc, 0, tn, nk, 0, WL_ROWS, gr)
    if (mode == OUT_SWIGLU) BR_EXPERTS(OUT_SWIGLU);
    else if (mode == OUT_F32) BR_EXPERTS(OUT_F32);
    else BR_EXPERTS(OUT_BF16);
#undef BR_EXPERTS
    return br_check_launch();
}

// 128x256 or 256x256 tiles, for rows an expert of which the host knows the mean only.
// Gated product: the fewer rounds of workgroups by the times a k-tile of `choose_quad`, with every expert's pairs taken as the mean and half a
// standard deviation of evenly drawn ones, rounded up to tiles; from eight rounds of 128-row tiles on the taller one may be counted a fifth
// longer, since a tile multiplies only the blocks of 64 rows that it has and there is no round of few tiles to wait for.  us with 128 rows a tile
// and 256, equal rows an expert / rows that random weights draw (half to twice the mean; two draws):
//   32 experts of 1,792 by 4,096: 64 pairs an expert 171, 174 / 185, 177; 179, 182.  112: 188, 191 / 219, 204; 215, 215.  160: 249, 222 / 261, 285; 254,
//     264.  225: 274, 256 / 274, 325; 311, 324.  256 (128 rows taken): 281, 263 / 318, 335; 326, 331.  300: 356, 417 / 360, 395; 337, 333.  350: 392, 437 / 393,
//     394; 384, 412.  400: 419, 441 / 441, 429; 447, 426.  450: 460, 448 / 489, 439; 479, 504.  512: 469, 453 / 525, 513; 517, 510.  603: 584, 558 / 602,
//     572; 598, 582.  900: 823, 772 / 852, 835; 856, 768.  1,800: 1,629, 1,474 / 1,638, 1,504; 1,633, 1,476
//   16 experts of 1,408 by 2,048: 64: 33, 34 / 38, 47; 39, 45.  136: 67, 47 / 61, 60; 65, 60.  225: 67, 64 / 66, 63; 66, 64.  300: 83, 121 / 72, 115; 72, 118.  450:
//     105, 124 / 103, 121; 102, 124.  512 (128 rows taken): 106, 129 / 130, 125; 132, 124.  768: 171, 189 / 170, 188; 172, 186.  900: 203, 193 / 199, 194; 203,
//     198.  1,800: 371, 380 / 374, 383; 373, 384
// Over 24 means from 64 to 1,800, these two shapes and equal, mildly and clearly uneven rows the choice takes 1.3 % longer than the faster height each
// time; a line at 448 pairs takes 2.9, always 128 rows 3.5.
// Down product (short k, float rows), where an expert has more rows than the lower tile: the taller one from four rounds of 128-row tiles on, and with
// fewer where its rounds are the fewer both so counted and for rows spread evenly over 0.7 to 1.3 times the mean.  Same shapes: 32 experts 128 pairs
// 115, 115 / 132, 137; 127, 140, 160: 146, 124 / 149, 144; 147, 141, 300: 202, 205 / 208, 200; 206, 202, 603: 339, 311 / 362, 315; 362, 314, 1,800: 943, 841 / 1,024, 857;
// 1,004, 860.  16 experts 160: 28, 32 / 30, 38; 30, 37, 225 (128 rows taken): 33, 40 / 46, 40; 46, 41, 300: 45, 43 / 45, 42; 46, 42, 400 (128): 52, 46 / 50, 73; 52, 73, 450
// (128): 54, 47 / 68, 76; 55, 76, 603: 73, 78 / 74, 78; 73, 81, 768: 80, 83 / 94, 84; 95, 84, 1,200: 137, 126 / 142, 130; 143, 127.  1.2 % longer than the faster; four
// rounds alone 1.8.
static bool experts_tall_tiles(int pairs, int E, int N, bool gated, int cus) {
    const double mean = (double)pairs / E, high = mean + 0.5 * sqrt(mean);
    // rounds of tiles of 128 (i = 0) or 256 rows for experts' rows spread evenly over `from` to `to`, and the time they take
    auto rounds = [&](double from, double to, int i) {
        double tiles = 0.0;
        for (int q = 0; q < 16; ++q) tiles += ceil((from + (to - from) * (q + 0.5) / 16) / (128 << i));
        return E * tiles / 16 * ((N + 255) / 256) / cus;
    };
    auto time = [&](double from, double to, int i) {
        const double r = rounds(from, to, i), whole = floor(r), share = r - whole;
        return (whole + (share > 0 ? (whole ? 0.9 + 0.1 * share : 0.6 + 0.4 * share * share * share) : 0.0)) * QUAD_FULL[i ? 0 : 1];
    };
    const double low = time(high, high, 0), tall = time(high, high, 1);
    if (gated) return tall <= (rounds(high, high, 0) >= 8.0 ? 1.2 : 1.03) * low;
    return mean > 128 && (rounds(mean, mean, 0) >= 4.0 || (tall <= 1.03 * low && time(0.7 * mean, 1.3 * mean, 1) <= time(0.7 * mean, 1.3 * mean, 0)));
}

// rows of the tiles that br_experts_tiles takes
extern "C" int br_experts_tiles_rows(int pairs, int E, int N, int gated) {
    return pairs > 0 && E > 0 && N > 0 && experts_tall_tiles(pairs, E, N, gated != 0, br_device_cus()) ? 256 : 128;
}

// rows: 128 or 256 a tile (tests and measurements), 0 by the rule
extern "C" int br_experts_tiles(const void* A, const void* W, const int* first, const int* order, void* C, int gated, int out_is_bf16,
                                int a_rows, int pairs, int E, int N, int K, int top, float limit, float alpha, int rows, hipStream_t s) {
    if (pairs <= 0) return BR_OK;
    if (rows != 0 && rows != 128 && rows != 256) return BR_BAD_ARG;
    const size_t ldc = gated ? (size_t)N / 2 : (size_t)N;
    if (!br_experts_tiles_takes(N, K) || E <= 0 || top <= 0 || (gated && !out_is_bf16) || ((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) % 16 != 0 ||
        !quad_takes(C, order ? a_rows : min(a_rows, 256), N, K, K, ldc))
        return BR_BAD_ARG;
    const bool exact = top > 1 && (unsigned long long)pairs * top < (1ull << 32);
    const QuadGroups gr = {first, order, E, top, exact ? (unsigned)(((1ull << 32) + top - 1) / top) : 0u, limit, alpha};
    const int mode = gated ? OUT_SWIGLU : out_is_bf16 ? OUT_BF16 : OUT_F32;
    const int cus = br_device_cus();
    if (!cus) return BR_LAUNCH_FAILED;
    if (rows ? rows == 256 : experts_tall_tiles(pairs, E, N, gated != 0, cus))
        return launch_experts_tiles<256, 256, 2, 3, 2>((const bf16*)A, (const bf16*)W, C, mode, pairs, N, K, ldc, gr, s);
    return launch_experts_tiles<128, 256, 3, 3, 2>((const bf16*)A, (const bf16*)W, C, mode, pairs, N, K, ldc, gr, s);
}

// rows of a block of the blocked weight layout (the host lays weights out by it)
extern "C" int br_gemm_bf16_block_rows() { return WL_BLOCK_ROWS; }
