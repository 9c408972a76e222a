// Routed experts for steps of some ten pairs an expert, the weights streamed by all waves together.
//
// Between the streams of routed_experts.hip (a wave's ring holds 16 pairs; an expert with more has its rows read again) and the prompt
// products' tiles (128 pairs a tile, most of them padding, and a fresh start for every tile) the experts' matrices are
// still what a step reads.  Here a unit is 16 HB weight rows of one expert against up to 16 MB of its pairs over all of
// k, and one workgroup a compute unit walks an equal run of units.  A stage of the workgroup's ring of three holds one
// 128-wide chunk of the unit's weights and activations, brought by all eight waves with direct loads two chunks ahead
// across unit ends, one barrier a chunk: 32 KB of weights more on their way than a stream's waves have, and every byte of
// activations serves 16 HB rows.  Wave w multiplies the weight rows 16 (w % 4) .. + 16 (and 64 + 16 (w % 4) .. + 16 where
// the unit has them) with k-steps 2 (w / 4), 2 (w / 4) + 1 of the chunk; the two halves are added in LDS at the unit's
// end, in the stage that was multiplied last.  Where a unit starts in k depends on its rows only, and its height on the
// matrices only, so a pair's output does not depend on what else is in the step.
//   UP: a unit's rows are blocks of 8 gate rows and the up rows of the same channels, y[p, f] the gated unit, bfloat16;
//   else rows of W_d, out[p, n] float.
// 32 experts of 1,792 by 4,096, 8 of them chosen evenly, weights in no cache, both products in us, streams / these / the prompt products'
// tiles: 16 tokens 225 / 230 / 260, 24 tokens 246 / 231 / 263, 40 tokens 266 / 242 / 259 (6.1 and 5.5 TB/s), 64 tokens 362 / 237 / 259,
// 96 tokens 500 / 257 / 262.  16 experts of 1,408 by 2,048, 4 chosen: 16 tokens 59 / 59 / 70, 32 tokens 56 / 56 / 77, 64 tokens
// 84 / 57 / 76, 100 tokens 115 / 62 / 82.  In a step of 40 sequences among other work: 193 + 87 by the tiles, 152 + 83 by these.  Bound
// by the memory; the rest is each launch's start (routing tables, first chunks) and the barriers at a unit's end.
#include "expert_units.h"

#define RXW_S 3
#define RXW_NW 8
#define RXW_MAX_E 512
#define RXW_MAX_PAIRS 2048

template <int MB, int HB, bool UP>
__global__ __launch_bounds__(RXW_NW * 64) void experts_wide_kernel(const bf16* __restrict__ A, const bf16* __restrict__ Wt,
                                                                   const int* __restrict__ first, const int* __restrict__ order,
                                                                   void* __restrict__ C, int pairs, int E, int N, int K, int top,
                                                                   float limit, float alpha) {
    constexpr int S = RXW_S, D = S - 1, NW = RXW_NW, H = 16 * HB, XR = 16 * MB;
    constexpr int ROWS = H + XR, STAGE = ROWS * 256;          // stacked rows of a stage: weights, then activations
    constexpr int NLD = ROWS / 4, NDMA = (NLD + NW - 1) / NW; // wave-loads of 4 rows; of each wave (surplus ones repeat the last)
    constexpr int RLD = XR + 1, UROWS = UP ? H / 2 : H;       // output columns of a unit
    constexpr bool TWO = HB > 4;
    static_assert(HB >= 4 && HB <= 8 && NDMA <= 63 && H * RLD * 4 <= STAGE, "stage");
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    int* firstL = (int*)(smem + S * STAGE);                   // [E + 2]
    int* cum = firstL + E + 2;                                // [E + 1] units before expert e
    int* tok = cum + E + 1;                                   // UP: [pairs] the token of a pair
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int rb = wave & 3, khalf = wave >> 2;
    const bool has1 = TWO && rb + 4 < HB;
    const int tiles = (N + UROWS - 1) / UROWS;
    for (int e = tid; e <= E; e += NW * 64) {
        firstL[e] = first[e];
        if (e == E) firstL[E + 1] = first[E];
    }
    if (UP)
        for (int p = tid; p < pairs; p += NW * 64) tok[p] = order[p] / top;
    __syncthreads();
    if (tid < 64) {
        int run = 0;
        for (int e0 = 0; e0 < E; e0 += 64) {
            const int e = e0 + lane;
            const int mine = e < E ? (firstL[e + 1] - firstL[e] + XR - 1) / XR * tiles : 0;
            int sum = mine;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int v = __shfl_up(sum, o, 64);
                if (lane >= o) sum += v;
            }
            if (e < E) cum[e] = run + sum - mine;
            run += __shfl(sum, 63, 64);
        }
        if (lane == 0) cum[E] = run;
    }
    __syncthreads();
    const int total = __builtin_amdgcn_readfirstlane(cum[E]);
    const int u0 = (int)((long long)total * blockIdx.x / gridDim.x), u1 = (int)((long long)total * (blockIdx.x + 1) / gridDim.x);
    if (u0 >= u1) return;
    const int nch = K / 128, nitems = (u1 - u0) * nch;
    const unsigned ring_lds = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)smem);

    // the sums of two chunks, and of the pairs before them: the error against 64 bits is 8.4e-8 of the result at K = 1,792 (streams
    // 8.6e-8, tiles 2.5e-7), where one chain over all of k leaves 1.7e-7
    f32x4 acc[TWO ? 2 : 1][MB], sum[TWO ? 2 : 1][MB];
    auto clear = [](f32x4(&v)[TWO ? 2 : 1][MB]) {
#pragma unroll
        for (int t = 0; t < (TWO ? 2 : 1); ++t)
#pragma unroll
            for (int j = 0; j < MB; ++j) v[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    auto end_run = [&]() {
#pragma unroll
        for (int t = 0; t < (TWO ? 2 : 1); ++t)
#pragma unroll
            for (int j = 0; j < MB; ++j) sum[t][j] += acc[t][j];
        clear(acc);
    };
    clear(acc);
    clear(sum);

    RxUnit is = rx_unit_at<XR>(__builtin_amdgcn_readfirstlane(u0), cum, firstL, E, tiles), cp = is;
    int issued = 0, is_left = 0, is_wrap = 0;                 // chunks asked for; of unit `is` to go, and until its first in k
    unsigned is_off = 0, cp_off = 0;                          // the ring's stage to fill, to multiply (bytes)
    const bf16* src[NDMA];                                    // this lane's 16 bytes of each of its wave's loads
    auto load_index = [&](int q) { return wave * NDMA + q < NLD - 1 ? wave * NDMA + q : NLD - 1; };
    auto enter = [&]() {                                      // the issue cursor is at another unit
        const int rot = (int)((((unsigned)(is.e * tiles + is.t) * 2654435761u) >> 8) % (unsigned)nch);
        is_left = nch;
        is_wrap = nch - rot;
        const bf16* we = Wt + (size_t)is.e * (UP ? 2 * N : N) * K;
#pragma unroll
        for (int q = 0; q < NDMA; ++q) {
            const int row = load_index(q) * 4 + (lane >> 4);
            const bf16* gp;
            if (row < H) {
                int n;
                if (UP) {
                    n = min(is.t * UROWS + (row >> 4) * 8 + (row & 7), N - 1) + ((row & 8) ? N : 0);
                } else n = min(is.t * UROWS + row, N - 1);
                gp = we + (size_t)n * K;
            } else {
                const int p = is.p0 + min(row - H, is.np - 1);
                gp = A + (size_t)(UP ? tok[p] : p) * K;
            }
            src[q] = gp + (size_t)rot * 128 + (((lane & 15) ^ (row & 7)) * 8);
        }
    };
    auto issue = [&]() {
#pragma unroll
        for (int q = 0; q < NDMA; ++q) {
            const unsigned lds = __builtin_amdgcn_readfirstlane(ring_lds + is_off + load_index(q) * 1024);
            if (load_index(q) * 4 < H)                        // weights pass once: non-temporal
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds), "v"(src[q]) : "m0", "memory");
            else
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src[q]) : "m0", "memory");
            src[q] += 128;
        }
        if (--is_wrap == 0) {                                 // on to the unit's first chunk
#pragma unroll
            for (int q = 0; q < NDMA; ++q) src[q] -= (size_t)nch * 128;
        }
        ++issued;
        is_off = is_off + STAGE == S * STAGE ? 0 : is_off + STAGE;
        if (--is_left == 0 && issued < nitems) {
            rx_next_unit<XR>(is, firstL, E, tiles);
            enter();
        }
    };
    enter();
#pragma unroll
    for (int j = 0; j < D; ++j)
        if (issued < nitems) issue();
    int cp_left = nch;
    for (int it = 0; it < nitems; ++it) {
        // the chunk to multiply has landed when at most the loads of the chunk asked for after it are in flight; this wave's
        // reads of the stage that is asked for again next are done
        if (issued - it - 1 >= 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NDMA) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                         // every wave's part of it is there; the chunk before is done with
        asm volatile("" ::: "memory");
        if (issued < nitems) issue();
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
        if (--cp_left > 0) {
            if (((nch - cp_left) & 1) == 0) end_run();
            continue;
        }
        end_run();
        // The unit's end: sum[t][j][r] is weight row 64 t + 16 rb + 4 g + r of the unit, pair 16 j + r16.  The sums meet in
        // the stage that was multiplied last: it is asked for again behind the next chunk's barrier, which a wave reaches
        // after its part of the epilogue.
        cp_left = nch;
        float* red = (float*)st;                              // [H][RLD]
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                         // every wave has read its operands of the stage
        asm volatile("" ::: "memory");
        if (khalf == 1) {
#pragma unroll
            for (int t = 0; t < (TWO ? 2 : 1); ++t)
                if (t == 0 || has1)
#pragma unroll
                    for (int j = 0; j < MB; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r) red[(64 * t + 16 * rb + 4 * g + r) * RLD + 16 * j + r16] = sum[t][j][r];
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
                            *p = sum[t][j][r] + *p;
                        }
        }
        clear(sum);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        for (int e = tid; e < UROWS * cp.np; e += NW * 64) {
            const int m = e / UROWS, c = e % UROWS, n = cp.t * UROWS + c;
            if (n >= N) continue;
            if (UP) {
                const int gr = (c >> 3) * 16 + (c & 7);
                ((bf16*)C)[(size_t)(cp.p0 + m) * N + n] = (bf16)rx_glu(red[gr * RLD + m], red[(gr + 8) * RLD + m], limit, alpha);
            } else ((float*)C)[(size_t)(cp.p0 + m) * N + n] = red[c * RLD + m];
        }
        rx_next_unit<XR>(cp, firstL, E, tiles);
    }
}

// Blocks of 16 weight rows of a unit (4 to 8): the least of rounds of units over the compute units (every expert one group of
// pairs) times what a unit's chunk costs, its rows and a constant for the activations and the barrier.  By the matrices only.
// Measured (32 pairs a group, us): gate/up of 32 experts of 1,792 by 4,096 (112 rows make four whole rounds) 148 at 112 rows,
// 156 at 128, 152 at 96; their down matrices 79 at 128 rows, 82 at 112, 84 at 96.  Rings of four stages, units of 64 rows with two
// workgroups to a compute unit and groups of 16 pairs are within 3 % of that where they are not slower.
static int rx_wide_height(int E, int N, bool up, int cus) {
    int best = 8;
    double least = 1e30;
    for (int hb = 8; hb >= 4; --hb) {
        const int rows = up ? 8 * hb : 16 * hb;
        const long long units = (long long)E * ((N + rows - 1) / rows);
        const double t = (double)((units + cus - 1) / cus) * (16 * hb + 24);
        if (t < least) { least = t; best = hb; }
    }
    return best;
}

template <int MB, int HB, bool UP>
static int rx_launch_wide(const void* A, const void* Wt, const int* first, const int* order, void* C, int pairs, int E, int N, int K, int top,
                          float limit, float alpha, int cus, hipStream_t s) {
    constexpr size_t ring = (size_t)RXW_S * (16 * HB + 16 * MB) * 256, most = ring + (2 * RXW_MAX_E + 3) * 4 + RXW_MAX_PAIRS * 4;
    static_assert(most <= 160 * 1024, "LDS");
    auto kern = experts_wide_kernel<MB, HB, UP>;
    static bool set = false;
    if (!set) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most) != hipSuccess) return BR_LAUNCH_FAILED;
        set = true;
    }
    const size_t lds = ring + (size_t)(2 * E + 3) * 4 + (size_t)pairs * 4;
    kern<<<cus, RXW_NW * 64, lds, s>>>((const bf16*)A, (const bf16*)Wt, first, order, C, pairs, E, N, K, top, limit, alpha);
    return br_check_launch();
}

// Whether experts_wide_kernel takes `pairs` pairs of E experts' matrices of N rows over K: K in steps of 128 from 256.
extern "C" int br_experts_wide_takes(int E, int N, int K, int pairs) {
    return E > 0 && E <= RXW_MAX_E && N > 0 && K % 128 == 0 && K >= 256 && pairs > 0 && pairs <= RXW_MAX_PAIRS &&
           ((long long)E + pairs / 32) * ((N + 31) / 32) * (K / 128) < (1ll << 31);
}

// `up`: Wt [E][2 N][K], A the tokens' rows (through `order`), C bfloat16 [pairs, N]; else Wt [E][N][K], A the pairs' rows, C float
// [pairs, N].  Groups of 32 pairs up to 16 an expert on average, of 64 beyond: few experts then have more than a group, whose rows
// would be read again.  32 experts of 1,792 by 4,096, both products in us at groups of 32 / 64 (tiles), scores drawn evenly; with as
// much spread between the experts as between the tokens: 32 tokens 236 / 244 (257); 180 / 188 (225).  64 tokens 237 / 250 (259);
// 291 / 265 (259).  80 tokens 247 / 253 (259); 343 / 263 (251).  128 tokens 363 / 267 (268); 409 / 328 (257).  (A recorded
// step's tokens count with its padding, 64 for 33 to 64 that go to experts: 16 an expert are about 12 there.)
extern "C" int br_experts_wide(const void* A, const void* Wt, const int* first, const int* order, void* C, int up, int pairs, int E,
                               int N, int K, int top, float limit, float alpha, hipStream_t s) {
    if (pairs <= 0) return BR_OK;
    if (!br_experts_wide_takes(E, N, K, pairs) || top <= 0 || (up && !order) || (((uintptr_t)A | (uintptr_t)Wt) & 15) != 0) return BR_BAD_ARG;
    const int cus = br_device_cus();
    if (!cus) return BR_LAUNCH_FAILED;
    const bool tall = pairs > 16 * E;
#define RX_WIDE(HB_)                                                                                                           \
    case HB_:                                                                                                                  \
        if (up) return tall ? rx_launch_wide<4, HB_, true>(A, Wt, first, order, C, pairs, E, N, K, top, limit, alpha, cus, s)  \
                            : rx_launch_wide<2, HB_, true>(A, Wt, first, order, C, pairs, E, N, K, top, limit, alpha, cus, s); \
        return tall ? rx_launch_wide<4, HB_, false>(A, Wt, first, order, C, pairs, E, N, K, top, limit, alpha, cus, s)         \
                    : rx_launch_wide<2, HB_, false>(A, Wt, first, order, C, pairs, E, N, K, top, limit, alpha, cus, s);
    switch (rx_wide_height(E, N, up != 0, cus)) {
        RX_WIDE(4)
        RX_WIDE(5)
        RX_WIDE(6)
        RX_WIDE(7)
        RX_WIDE(8)
    }
#undef RX_WIDE
    return BR_BAD_ARG;
}
