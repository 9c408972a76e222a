// True 32-bit matrix product: C[M,N] (+)= A[M,K] * W[N,K]^T in float, every product and sum in 32 bits (on the vector units, or
// on the matrix cores' float instruction, which rounds nothing to fewer bits).
//
// The order of an output element's sum depends on K alone, never on M, on the tile it falls in, on which kernel computed it
// or on the other rows of the batch, so that whole prompts and token-by-token runs agree bit for bit:
//  * K in steps of 64 (aligned weights): k is cut into 8 segments of whole 64s (segment s: 64s number s n / 8 .. (s + 1) n / 8
//    of the n there are).  Within a segment, 16 k at a time, four v_mfma_f32_16x16x4_f32 of which number i takes k + i, k + 4 +
//    i, k + 8 + i and k + 12 + i (a lane's 16 bytes are four instructions' operands); the segments are added in order.  The
//    streaming kernel gives each of its 8 waves a segment; the tiles sum segment by segment, or every segment in a workgroup
//    of its own with the segments added by a second launch.
//  * any other K: ascending k by one thread, the 64x64x16 LDS-tiled form below.
//
// reference: op_linear_proj, kernels/megakernel_ops.hip:166-276 (one block per output row, f32 accumulate).
#include "common.h"
#include <algorithm>
#include <type_traits>

#define F32_BM 64
#define F32_BN 64
#define F32_BK 16

// mode 0: C = AW^T ; mode 1: C += AW^T (C holds the residual stream)
template <int MODE>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                       float* __restrict__ C, int M, int N, int K,
                                                       size_t lda, size_t ldc) {
    __shared__ float As[F32_BK][F32_BM + 4];
    __shared__ float Ws[F32_BK][F32_BN + 4];
    const int tid = threadIdx.x;
    const int tx = tid & 15, ty = tid >> 4;
    const int m0 = blockIdx.y * F32_BM, n0 = blockIdx.x * F32_BN;
    const int lr = tid >> 2, lk = (tid & 3) * 4;  // loader: row lr, k offset lk..lk+3
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

    for (int k0 = 0; k0 < K; k0 += F32_BK) {
        {
            const int m = m0 + lr, n = n0 + lr;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int k = k0 + lk + e;
                As[lk + e][lr] = (m < M && k < K) ? A[(size_t)m * lda + k] : 0.f;
                Ws[lk + e][lr] = (n < N && k < K) ? W[(size_t)n * K + k] : 0.f;
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < F32_BK; ++k) {
            float a[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[k][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = Ws[k][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= N) continue;
            float* c = C + (size_t)m * ldc + n;
            if (MODE == 1) *c = *c + acc[i][j]; else *c = acc[i][j];
        }
    }
}

// ------------------------------------------------------------ K in steps of 64 -----
#define F32_SEGS 8
#define F32_KC 64            // k that segments are whole multiples of

__device__ __forceinline__ void f32_dma16(unsigned lds, const void* p) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(p) : "m0", "memory");
}
__device__ __forceinline__ void f32_dma16_nt(unsigned lds, const void* p) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds), "v"(p) : "m0", "memory");
}
__device__ __forceinline__ void f32_dma4(unsigned lds, const void* p) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds), "v"(p) : "m0", "memory");
}
// 1 KB of LDS from rows of `ROWB` bytes, 16 bytes a lane, the 16-byte columns of a row exchanged by `SW(row)`: `src(row, col)`
// gives the address of the row's 16-byte column.  Rows that do not lie at multiples of 16 bytes come 4 bytes a lane.
template <int ROWB, class Src, class Sw>
__device__ __forceinline__ void f32_bring(unsigned lds, int row0, int lane, bool aligned, bool nt, Src src, Sw sw) {
    constexpr int CPL = ROWB / 16;
    if (aligned) {
        const int row = row0 + lane / CPL, col = (lane % CPL) ^ sw(row);
        if (nt) f32_dma16_nt(lds, src(row, col));
        else f32_dma16(lds, src(row, col));
        return;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int at = q * 16 + (lane >> 2), row = row0 + at / CPL, col = (at % CPL) ^ sw(row);
        f32_dma4(lds + q * 256, (const float*)src(row, col) + (lane & 3));
    }
}

// M <= 16, K from 512: bound by reading the weights.  One workgroup a compute unit walks over tiles of 16 weight rows, tile t
// of workgroup b being b + t * grid; each wave walks its segment of k in chunks of 64 through an LDS ring of its own (direct
// loads of 256-byte row pieces, the weights non-temporal, the next chunk on its way across tile ends), the waves' sums meet
// in LDS at a tile's end.  28,672 x 4,096 (470 MB) at 1 / 4 / 16 rows: 69 / 76 / 104 us (6.9 / 6.2 / 4.5 TB/s), 4,096 x 14,336:
// 37 / 37 / 43, where the 64x64 tiles of one thread a sum took 549 / 552 / 580 and 1,435 / 1,479 / 1,534.
template <int XR, int MODE>
__global__ __launch_bounds__(512) void gemm_f32_stream_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                              float* __restrict__ C, int M, int N, int K, size_t lda, size_t ldc,
                                                              int ntiles, int a_aligned) {
    constexpr int NW = F32_SEGS, ROWB = F32_KC * 4, STAGE = (16 + XR) * ROWB, S = 2;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    float* red = (float*)(smem + NW * S * STAGE);             // [2][NW][16][17]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    unsigned char* ring = smem + wave * (S * STAGE);
    const unsigned ring_lds = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)ring);
    const int nch = K / F32_KC, c0 = wave * nch / NW, ncw = (wave + 1) * nch / NW - c0;
    const int my_tiles = (ntiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x, nitems = my_tiles * ncw;
    int is_t = 0, is_c = 0, cp_t = 0, cp_c = 0, buf = 0;
    auto issue = [&](int slot) {
        const int n0 = ((int)blockIdx.x + is_t * (int)gridDim.x) * 16, k0 = (c0 + is_c) * F32_KC;
        const unsigned lds = __builtin_amdgcn_readfirstlane(ring_lds + slot * STAGE);
        auto sw = [](int row) { return row & 7; };
#pragma unroll
        for (int q = 0; q < 4; ++q)
            f32_bring<ROWB>(lds + q * 1024, 4 * q, lane, true, true, [&](int row, int col) { return W + (size_t)min(n0 + row, N - 1) * K + k0 + col * 4; }, sw);
#pragma unroll
        for (int q = 0; q < XR / 4; ++q)
            f32_bring<ROWB>(lds + (4 + q) * 1024, 4 * q, lane, a_aligned, false, [&](int row, int col) { return A + (size_t)min(row, M - 1) * lda + k0 + col * 4; }, sw);
        if (++is_c == ncw) { is_c = 0; ++is_t; }
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (nitems > 0) issue(0);
    for (int it = 0; it < nitems; ++it) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        if (it + 1 < nitems) issue((it + 1) & 1);
        const unsigned char* st = ring + (it & 1) * STAGE;
        const int xr = XR == 8 ? (r16 & 7) : r16;
        f32x4 wf[4], xv[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            wf[b] = *(const f32x4*)(st + r16 * ROWB + (((4 * b + g) ^ (r16 & 7)) * 16));
            xv[b] = *(const f32x4*)(st + (16 + xr) * ROWB + (((4 * b + g) ^ (xr & 7)) * 16));
        }
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[b][i], xv[b][i], acc, 0, 0, 0);
        if (++cp_c < ncw) continue;
        cp_c = 0;
        const int n0 = ((int)blockIdx.x + cp_t * (int)gridDim.x) * 16;
        ++cp_t;
        float* rb = red + buf * (NW * 16 * 17);
#pragma unroll
        for (int r = 0; r < 4; ++r) rb[(wave * 16 + 4 * g + r) * 17 + r16] = acc[r];
        acc = {0.f, 0.f, 0.f, 0.f};
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int m = tid >> 4, nl = tid & 15, n = n0 + nl;
        if (m < M && n < N) {
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) v += rb[(w * 16 + nl) * 17 + m];
            float* c = C + (size_t)m * ldc + n;
            *c = MODE == 1 ? *c + v : v;
        }
        buf ^= 1;
    }
}

// Any M: 16 TJ rows x 64 columns by four waves along the columns (16 TJ x 16 each), two workgroups to a compute unit, a ring of two or three
// LDS stages of 32 k by direct loads, bound by the matrix cores.  A wave has the operands of 16 k in registers twice: while one set is
// multiplied, the other is read from LDS and the direct loads of the stage that is two or three on are asked for one at a time (the
// path into LDS takes one of them per 16 cycles: bunched behind the barrier they held up the products).  28,672 x 4,096 at 20 / 128 / 279 / 450
// rows 105 -> 92, 274 -> 257, 602 -> 553, 1,022 -> 912 us, 4,096 x 14,336 at 279 rows 279 -> 266 (123 TFLOP/s; a loop of the instruction alone
// makes 155, at a clock of 2.4 GHz where this kernel is given 2.1 to 2.2).  Before: 128 columns by waves of 32, operands read before their products.
// More stages, at one workgroup to a compute unit or two: nothing.  Error against 64 bits at 64 rows of 4,096: 4.1e-7 of the norm, 1.1e-6 with
// one ascending sum.  TJ is chosen so that the rows fill their tiles (279 rows: three of 96).  SPLIT: segment blockIdx.y alone, into a
// matrix of its own.  The accumulators hold the product transposed: four columns of a row a lane.
#define F32_TN 64
template <int N_, class F>
__device__ __forceinline__ void f32_for(F&& f) {
    if constexpr (N_ > 0) {
        f32_for<N_ - 1>(f);
        f(std::integral_constant<int, N_ - 1>{});
    }
}
template <int LEFT>
__device__ __forceinline__ void f32_wait() {                  // all but the last LEFT loads, and all reads of LDS
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LEFT) : "memory");
}
template <int TJ, int MODE, bool SPLIT>
__global__ __launch_bounds__(256, 2) void gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                            float* __restrict__ C, int M, int N, int K, size_t lda, size_t ldc,
                                                            int tiles_m, int a_aligned, int c_aligned) {
    constexpr int BM = 16 * TJ, BN = F32_TN, ROWB = 128, STAGE = (BM + BN) * ROWB, S = TJ <= 3 || TJ == 5 ? 3 : 2;
    __shared__ __attribute__((aligned(1024))) unsigned char st[S * STAGE];
    int pid = blockIdx.x;
    {
        const int total = gridDim.x, per = total / 8, xcd = pid % 8, idx = pid / 8;
        if (pid < per * 8) pid = xcd * per + idx;
    }
    const int m0 = pid % tiles_m * BM, n0 = pid / tiles_m * BN;      // the row tiles of the same weights in turn
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)st);
    const int nch = K / F32_KC;
    const int s0 = SPLIT ? (int)blockIdx.y : 0, s1 = SPLIT ? s0 + 1 : F32_SEGS;
    const int kt0 = s0 * nch / F32_SEGS * 2, kt1 = s1 * nch / F32_SEGS * 2;      // stages of 32 k
    auto sw = [](int row) { return (row >> 1) & 7; };
    constexpr int NA = (BM / 8 + 3) / 4, NB = BN / 32;         // a wave's loads of a stage (four times NA where rows lie anywhere)
    // load q of stage kt: of activation rows, then of weight rows
    auto bring = [&](auto aligned_, int q, unsigned base, int k0) {
        constexpr bool ALIGNED = decltype(aligned_)::value;
        if (q < NA) {
            const int r8 = min(4 * q + wave, BM / 8 - 1);     // (every wave has the same number of loads on its way; the last rows twice)
            f32_bring<ROWB>(base + r8 * 1024, r8 * 8, lane, ALIGNED, false,
                            [&](int row, int col) { return A + (size_t)min(m0 + row, M - 1) * lda + k0 + col * 4; }, sw);
        } else {
            const int r8 = 4 * (q - NA) + wave;
            f32_bring<ROWB>(base + BM * ROWB + r8 * 1024, r8 * 8, lane, true, false,
                            [&](int row, int col) { return W + (size_t)min(n0 + row, N - 1) * K + k0 + col * 4; }, sw);
        }
    };
    auto stage_at = [&](int kt) { return __builtin_amdgcn_readfirstlane(lds0 + (unsigned)(kt - kt0) % S * STAGE); };
    auto issue = [&](int kt) {
#pragma unroll
        for (int q = 0; q < NA + NB; ++q) {
            if (a_aligned) bring(std::true_type{}, q, stage_at(kt), kt * 32);
            else bring(std::false_type{}, q, stage_at(kt), kt * 32);
        }
    };
    f32x4 acc[TJ], sum[TJ];
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) { acc[j][r] = 0.f; sum[j][r] = 0.f; }
    // Two sets of operands, of 16 k each: one is multiplied while the other is read from LDS.
    struct Set { f32x4 wf, af[TJ]; };
    auto read = [&](Set& o, int kt, int b, auto r_) {         // operand r of k-step b of stage kt
        constexpr int r = decltype(r_)::value;
        const unsigned char* ap = st + (unsigned)(kt - kt0) % S * STAGE;
        const unsigned char* wp = ap + (BM + wave * 16) * ROWB;
        const int col = ((4 * b + g) ^ sw(r16)) * 16;
        if constexpr (r == 0) o.wf = *(const f32x4*)(wp + r16 * ROWB + col);
        else o.af[r - 1] = *(const f32x4*)(ap + (16 * (r - 1) + r16) * ROWB + col);
    };
    // the products of a set, `then(n)` behind the n-th; what `then` does stays there
    constexpr int NM = 4 * TJ;
    auto multiply = [&](const Set& o, auto then) {
        f32_for<NM>([&](auto n_) {
            constexpr int e = decltype(n_)::value / TJ, j = decltype(n_)::value % TJ;
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.wf[e], o.af[j][e], acc[j], 0, 0, 0);
            then(n_);
        });
        __builtin_amdgcn_sched_barrier(0);
    };
    // operand reads behind every second product (TJ = 1 has fewer products than that takes: behind each)
    auto reading = [&](Set& o, int kt, int b, auto n_) {
        constexpr int n = decltype(n_)::value, each = NM >= 2 * (TJ + 1) ? 2 : 1;
        if constexpr (n % each == 0 && n / each <= TJ) {
            read(o, kt, b, std::integral_constant<int, n / each>{});
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // all but the loads of the last `LEFT` stages asked for have come
    auto arrived = [&](auto left_) {
        constexpr int LEFT = decltype(left_)::value;
        constexpr int FOURS = LEFT * (4 * NA + NB) < 63 ? LEFT * (4 * NA + NB) : 63;
        static_assert(LEFT * (NA + NB) < 64, "vmcnt");
        if (a_aligned) f32_wait<LEFT * (NA + NB)>();
        else f32_wait<FOURS>();
    };
    Set x0, x1;
    if (kt0 < kt1) {
#pragma unroll
        for (int i = 0; i < S; ++i)
            if (kt0 + i < kt1) issue(kt0 + i);
        if (kt0 + S <= kt1) arrived(std::integral_constant<int, S - 1>{});
        else arrived(std::integral_constant<int, 0>{});
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        f32_for<TJ + 1>([&](auto r_) { read(x0, kt0, 0, r_); });
    }
    int seg = s0, seg_end = (s0 + 1) * nch / F32_SEGS * 2;
    for (int kt = kt0; kt < kt1; ++kt) {
        while (kt == seg_end) {                               // a segment is whole: onto the sum, in order
#pragma unroll
            for (int j = 0; j < TJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) { sum[j][r] += acc[j][r]; acc[j][r] = 0.f; }
            ++seg;
            seg_end = (seg + 1) * nch / F32_SEGS * 2;
        }
        multiply(x0, [&](auto n_) { reading(x1, kt, 1, n_); });
        // the next stage has come, and this one has been read by all waves: it is asked for again behind the barrier
        if (kt + S <= kt1) arrived(std::integral_constant<int, S - 2>{});
        else arrived(std::integral_constant<int, 0>{});
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const bool more = kt + S < kt1;
        if (more && !a_aligned) issue(kt + S);
        if (more && a_aligned) {
            const unsigned base = stage_at(kt + S);
            const int k0 = (kt + S) * 32;
            multiply(x1, [&](auto n_) {
                reading(x0, kt + 1, 0, n_);
                f32_for<NA + NB>([&](auto q_) {
                    constexpr int q = decltype(q_)::value;
                    if constexpr (decltype(n_)::value == (2 * q + 1) * NM / (2 * (NA + NB))) {
                        bring(std::true_type{}, q, base, k0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                });
            });
        } else if (kt + 1 < kt1) {
            multiply(x1, [&](auto n_) { reading(x0, kt + 1, 0, n_); });
        } else {
            multiply(x1, [](auto) {});
        }
    }
    if (SPLIT) C += (size_t)blockIdx.y * M * N;
    const int n = n0 + wave * 16 + 4 * g;
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
        const int m = m0 + 16 * j + r16;
        if (m >= M) continue;
        float* c = C + (size_t)m * ldc + n;
        f32x4 v = sum[j];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] += acc[j][r];
        if (c_aligned && n + 3 < N) {
            if (MODE == 1) {
                const f32x4 o = *(const f32x4*)c;
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = o[r] + v[r];
            }
            *(f32x4*)c = v;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) c[r] = MODE == 1 ? c[r] + v[r] : v[r];
        }
    }
}

// C (+)= the segments' matrices [F32_SEGS][M][N], added in order; a thread VEC neighbours of a row.
template <int MODE, int VEC>
__global__ __launch_bounds__(256) void gemm_f32_segments_kernel(const float* __restrict__ part, float* __restrict__ C, int M, int N,
                                                                size_t ldc) {
    typedef float vec __attribute__((ext_vector_type(VEC)));
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * VEC, all = (size_t)M * N;
    if (i >= all) return;
    vec p[F32_SEGS];
#pragma unroll
    for (int s = 0; s < F32_SEGS; ++s) p[s] = *(const vec*)(part + s * all + i);
    const int row = (int)(i / (unsigned)N), col = (int)(i - (size_t)row * N);
    float* c = C + (size_t)row * ldc + col;
    vec v;
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
        v[e] = 0.f;
#pragma unroll
        for (int s = 0; s < F32_SEGS; ++s) v[e] += p[s][e];
    }
    if (MODE == 1) {
        const vec o = *(const vec*)c;
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] = o[e] + v[e];
    }
    *(vec*)c = v;
}

template <int XR>
static int launch_f32_stream(const float* A, const float* W, float* C, int M, int N, int K, size_t lda, size_t ldc, int acc, int aligned,
                             int cus, hipStream_t s) {
    constexpr size_t lds = (size_t)F32_SEGS * 2 * (16 + XR) * F32_KC * 4 + 2 * F32_SEGS * 16 * 17 * 4;
    const int ntiles = (N + 15) / 16, grid = ntiles < cus ? ntiles : cus;
#define BR_F32_STREAM(MODE_)                                                                                                     \
    do {                                                                                                                         \
        auto kern = gemm_f32_stream_kernel<XR, MODE_>;                                                                           \
        static bool set = false;                                                                                                 \
        if (!set) {                                                                                                              \
            if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)      \
                return BR_LAUNCH_FAILED;                                                                                         \
            set = true;                                                                                                          \
        }                                                                                                                        \
        kern<<<grid, 512, lds, s>>>(A, W, C, M, N, K, lda, ldc, ntiles, aligned);                                                \
    } while (0)
    if (acc) BR_F32_STREAM(1); else BR_F32_STREAM(0);
#undef BR_F32_STREAM
    return br_check_launch();
}

template <int TJ, bool SPLIT>
static int launch_f32_tiles(const float* A, const float* W, float* C, int M, int N, int K, size_t lda, size_t ldc, int acc, int aligned,
                            float* scratch, hipStream_t s) {
    const int tm = (M + 16 * TJ - 1) / (16 * TJ), tn = (N + F32_TN - 1) / F32_TN;
    if (SPLIT) {
        const dim3 grid((unsigned)(tm * tn), F32_SEGS);
        gemm_f32_tile_kernel<TJ, 0, SPLIT><<<grid, 256, 0, s>>>(A, W, scratch, M, N, K, lda, (size_t)N, tm, aligned, N % 4 == 0 && (uintptr_t)scratch % 16 == 0);
        const size_t all = (size_t)M * N;
        const bool fours = N % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)C | (uintptr_t)scratch) % 16 == 0;
        const unsigned blocks = (unsigned)(((fours ? all / 4 : all) + 255) / 256);
        if (fours && acc) gemm_f32_segments_kernel<1, 4><<<blocks, 256, 0, s>>>(scratch, C, M, N, ldc);
        else if (fours) gemm_f32_segments_kernel<0, 4><<<blocks, 256, 0, s>>>(scratch, C, M, N, ldc);
        else if (acc) gemm_f32_segments_kernel<1, 1><<<blocks, 256, 0, s>>>(scratch, C, M, N, ldc);
        else gemm_f32_segments_kernel<0, 1><<<blocks, 256, 0, s>>>(scratch, C, M, N, ldc);
    } else {
        const int c_aligned = ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
        if (acc) gemm_f32_tile_kernel<TJ, 1, SPLIT><<<(unsigned)(tm * tn), 256, 0, s>>>(A, W, C, M, N, K, lda, ldc, tm, aligned, c_aligned);
        else gemm_f32_tile_kernel<TJ, 0, SPLIT><<<(unsigned)(tm * tn), 256, 0, s>>>(A, W, C, M, N, K, lda, ldc, tm, aligned, c_aligned);
    }
    return br_check_launch();
}

// Whole rounds of tiles (two workgroups to a compute unit) go as they are; the weight rows behind them, or all where there is no whole
// round, segment by segment, every segment in a workgroup of its own, where that is counted the faster: in runs of columns whose
// segments' sums fit the scratch.  In us, fitted to 550 products of 17 to 450 rows (as they are within 5 % on average, in segments 8): a workgroup alone on
// its compute unit takes 0.0062 + 0.0036 TJ a k, two beside each other 0.0108 + 0.0062 TJ; a launch 4; in segments 8 for the launches, 0.9 of
// those times, and the segments' sums written and read at 4.8 TB/s.  Over those products the choice is 0.9 % slower than the faster form each time.  279 rows
// by 28,672 x 4,096: 512 tiles of 1,344 twice, 320 in segments: 553 us, 602 at once; 640 rows by 4,096 x 14,336, whose segments do not fit at once: 593 us,
// 864 with no segments; 350 rows by 6,144 x 4,096 193, 254.  As they are / in segments: 17 rows by 4,096 x 1,024 17.1 / 10.7, by 11,264 x 2,048 30.6 / 22.5, by
// 28,672 x 2,048 42 / 45; 65 rows by 4,096 x 512 17 / 13.
template <int TJ>
static int launch_f32_tile(const float* A, const float* W, float* C, int M, int N, int K, size_t lda, size_t ldc, int acc, int aligned,
                           int cus, float* scratch, size_t scratch_floats, hipStream_t s) {
    const int tm = (M + 16 * TJ - 1) / (16 * TJ), tn = (N + F32_TN - 1) / F32_TN, round = 2 * cus;
    if ((long long)tm * tn > 0x7fffffffLL) return BR_BAD_ARG;
    // the time of `tiles` workgroups of `k` each
    auto rounds = [&](long long tiles, double k) {
        const long long tail = tiles % round;
        const double alone = k * (0.0062 + 0.0036 * TJ), beside = k * (0.0108 + 0.0062 * TJ);
        return (double)(tiles / round) * beside + (tail == 0 ? 0.0 : tail <= cus ? alone : beside);
    };
    int whole = tn, run = 0;                                           // columns of tiles: as they are, of a run in segments
    const int fit = (int)std::min<size_t>(scratch_floats / ((size_t)F32_SEGS * M * F32_TN), (size_t)tn);
    if (K >= F32_KC * F32_SEGS && fit > 0) {
        const int first = (int)((long long)tm * tn / round * round / tm), left = tn - first;
        const long long rest = (long long)tm * left;
        const double as_is = rounds(rest, K) + (first ? 0.0 : 4.0);
        const int runs = left > 0 ? (left + fit - 1) / fit : 0, each = runs ? (left + runs - 1) / runs : 0;
        double in_segments = 0.0;
        for (int c = 0; c < left; c += each) {
            const long long u = (long long)tm * std::min(each, left - c) * F32_SEGS;
            in_segments += 8.0 + 0.9 * rounds(u, (double)K / F32_SEGS) + (double)u * 16 * TJ * F32_TN * 8 / 4.8e6;
        }
        if (left > 0 && in_segments < as_is) whole = first, run = each;
    }
    if (whole > 0) {
        const int rc = launch_f32_tiles<TJ, false>(A, W, C, M, std::min(N, whole * F32_TN), K, lda, ldc, acc, aligned, nullptr, s);
        if (rc != BR_OK) return rc;
    }
    for (int c = whole; c < tn; c += run) {
        const int n = c * F32_TN;
        const int rc = launch_f32_tiles<TJ, true>(A, W + (size_t)n * K, C + n, M, std::min(N - n, run * F32_TN), K, lda, ldc, acc, aligned, scratch, s);
        if (rc != BR_OK) return rc;
    }
    return BR_OK;
}

// `scratch`: room for the segments' sums of products with few tiles (null: none).
extern "C" int br_gemm_f32(const float* A, const float* W, float* C, int M, int N, int K, size_t lda, size_t ldc, int accumulate,
                           float* scratch, size_t scratch_floats, hipStream_t s) {
    if (M <= 0 || N <= 0) return BR_OK;
    if (K <= 0 || lda < (size_t)K || ldc < (size_t)N) return BR_BAD_ARG;
    if (K % F32_KC == 0 && (uintptr_t)W % 16 == 0) {
        const int cus = br_device_cus();
        if (!cus) return BR_LAUNCH_FAILED;
        const int aligned = lda % 4 == 0 && (uintptr_t)A % 16 == 0;
        if (M <= 8 && K >= F32_KC * F32_SEGS) return launch_f32_stream<8>(A, W, C, M, N, K, lda, ldc, accumulate, aligned, cus, s);
        if (M <= 16 && K >= F32_KC * F32_SEGS) return launch_f32_stream<16>(A, W, C, M, N, K, lda, ldc, accumulate, aligned, cus, s);
        const int rows = (M + (M + 127) / 128 - 1) / ((M + 127) / 128);         // of a tile, before rounding up to 16
#define BR_F32_TILE(TJ_) launch_f32_tile<TJ_>(A, W, C, M, N, K, lda, ldc, accumulate, aligned, cus, scratch, scratch ? scratch_floats : 0, s)
        switch ((rows + 15) / 16) {
            case 1: return BR_F32_TILE(1);
            case 2: return BR_F32_TILE(2);
            case 3: return BR_F32_TILE(3);
            case 4: return BR_F32_TILE(4);
            case 5: return BR_F32_TILE(5);
            case 6: return BR_F32_TILE(6);
            case 7: return BR_F32_TILE(7);
            default: return BR_F32_TILE(8);
        }
#undef BR_F32_TILE
    }
    dim3 grid((N + F32_BN - 1) / F32_BN, (M + F32_BM - 1) / F32_BM);
    if (grid.y > 65535) return BR_BAD_ARG;
    if (accumulate) gemm_f32_kernel<1><<<grid, 256, 0, s>>>(A, W, C, M, N, K, lda, ldc);
    else gemm_f32_kernel<0><<<grid, 256, 0, s>>>(A, W, C, M, N, K, lda, ldc);
    return br_check_launch();
}
