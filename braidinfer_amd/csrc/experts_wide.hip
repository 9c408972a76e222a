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
// Groups of 32 pairs or of 64, by what the experts' real pairs cost: an expert with more than a group has its rows read again, and a chunk of
// the larger group brings 32 activation rows more.  32 experts of 1,792 by 4,096, 8 chosen, weights in no cache, both products in us, by
// groups of 32 / of 64 / as chosen (the prompt products' tiles), scores drawn evenly; with as much spread between the experts as between the
// tokens: 23 tokens 228 / 239 / 229 (251); 219 / 233 / 218 (231).  40 tokens 232 / 239 / 232 (251); 226 / 242 / 228 (230).  64 tokens 238 / 248 / 239
// (251); 285 / 261 / 264 (250).  16 experts of 1,408 by 2,048, 4 chosen, 64 tokens 58 / 64 / 59 (77); 80 / 66 / 67 (80).  Among a
// step's other work the tiles take longer, 193 + 87 at 40 sequences, and these 152 + 83.  Bound by the memory (6.1 and 5.5 TB/s at 40 tokens); the
// rest is each launch's start (routing tables, first chunks) and the barriers at a unit's end.
// (Both groups in one launch, every expert by its own, was tried: the workgroup whose run of units crosses from one to the other
// fills its ring twice, and all wait for it: 278 us at 64 uneven tokens, where one group for all takes 264.)
#include "expert_units.h"

#define RXW_S 3
#define RXW_NW 8
#define RXW_MAX_E 512
#define RXW_MAX_PAIRS 2048
#define RXW_MAX_XR 64              // pairs of the larger group

// Units u0 .. u1, groups of 16 MB pairs.
template <int MB, int HB, bool UP>
__device__ __forceinline__ void experts_wide_walk(const bf16* __restrict__ A, const bf16* __restrict__ Wt, void* __restrict__ C, unsigned char* smem,
                                                  const int* cum, const int* firstL, const int* tok, int u0, int u1, int E, int N, int K,
                                                  int tiles, float limit, float alpha) {
    constexpr int S = RXW_S, D = S - 1, NW = RXW_NW, H = 16 * HB, XR = 16 * MB;
    constexpr int ROWS = H + XR, STAGE = ROWS * 256;          // stacked rows of a stage: weights, then activations
    constexpr int NLD = ROWS / 4, NDMA = (NLD + NW - 1) / NW; // wave-loads of 4 rows; of each wave (surplus ones repeat the last)
    constexpr int RLD = XR + 1, UROWS = UP ? H / 2 : H;       // output columns of a unit
    constexpr bool TWO = HB > 4;
    static_assert(HB >= 4 && HB <= 8 && XR <= RXW_MAX_XR && NDMA <= 63 && H * RLD * 4 <= STAGE, "stage");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int rb = wave & 3, khalf = wave >> 2;
    const bool has1 = TWO && rb + 4 < HB;
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

template <int HB, bool UP>
__global__ __launch_bounds__(RXW_NW * 64) void experts_wide_kernel(const bf16* __restrict__ A, const bf16* __restrict__ Wt,
                                                                   const int* __restrict__ first, const int* __restrict__ order,
                                                                   void* __restrict__ C, int pairs, int E, int N, int K, int top,
                                                                   float limit, float alpha, int group) {
    constexpr int NW = RXW_NW, H = 16 * HB, UROWS = UP ? H / 2 : H;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    int* firstL = (int*)(smem + RXW_S * (H + RXW_MAX_XR) * 256);      // [E + 2]
    int* cum = firstL + E + 2;                                // [E + 1] units before expert e, then whether groups are of 64 pairs
    int* tok = cum + E + 2;                                   // UP: [pairs] the token of a pair
    const int tid = threadIdx.x, lane = tid & 63;
    const int tiles = (N + UROWS - 1) / UROWS;
    for (int e = tid; e <= E; e += NW * 64) {
        firstL[e] = first[e];
        if (e == E) firstL[E + 1] = first[E];
    }
    if (UP)
        for (int p = tid; p < pairs; p += NW * 64) tok[p] = order[p] / top;
    __syncthreads();
    if (tid < 64) {
        // groups of 32 pairs before each expert, and groups of 64 in the upper half
        const int groups = rx_sums_before(E, lane, [&](int e) {
            const int n = firstL[e + 1] - firstL[e];
            return ((n + 31) >> 5) + (((n + 63) >> 6) << 16);
        }, [&](int e, int before) { cum[e] = before; });
        // rounds of units over the workgroups times what a unit's chunk costs, its rows and 24 more for the activations and the barrier, 48
        // with groups of 64 (seven sets of 8 to 128 experts, 6 to 16 pairs each, even and uneven: 0.1 % behind the better of the two on
        // average, 9 % at most; by the number of units without rounds 2.5 and 33 %)
        const int u32 = (groups & 0xffff) * tiles, u64 = (groups >> 16) * tiles;
        const float per = __builtin_amdgcn_rcpf((float)gridDim.x);
        const bool larger = group ? group == 64
                                  : ceilf((float)u64 * per - 1e-3f) * (float)(H + 48) < ceilf((float)u32 * per - 1e-3f) * (float)(H + 24);
        for (int e = lane; e < E; e += 64) cum[e] = (larger ? cum[e] >> 16 : cum[e] & 0xffff) * tiles;
        if (lane == 0) {
            cum[E] = larger ? u64 : u32;
            cum[E + 1] = larger;
        }
    }
    __syncthreads();
    const int total = __builtin_amdgcn_readfirstlane(cum[E]);
    const bool tall = __builtin_amdgcn_readfirstlane(cum[E + 1]) != 0;
    // total b / grid, in 32 bits (at most a few hundred workgroups)
    const unsigned G = gridDim.x, each = (unsigned)total / G, over = (unsigned)total - each * G;
    const int u0 = (int)(blockIdx.x * each + blockIdx.x * over / G), u1 = (int)((blockIdx.x + 1) * each + (blockIdx.x + 1) * over / G);
    if (u0 >= u1) return;
    if (tall) experts_wide_walk<4, HB, UP>(A, Wt, C, smem, cum, firstL, tok, u0, u1, E, N, K, tiles, limit, alpha);
    else experts_wide_walk<2, HB, UP>(A, Wt, C, smem, cum, firstL, tok, u0, u1, E, N, K, tiles, limit, alpha);
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

template <int HB, bool UP>
static int rx_launch_wide(const void* A, const void* Wt, const int* first, const int* order, void* C, int pairs, int E, int N, int K, int top,
                          float limit, float alpha, int group, int cus, hipStream_t s) {
    constexpr size_t ring = (size_t)RXW_S * (16 * HB + RXW_MAX_XR) * 256, most = ring + (2 * RXW_MAX_E + 4) * 4 + RXW_MAX_PAIRS * 4;
    static_assert(most <= 160 * 1024, "LDS");
    auto kern = experts_wide_kernel<HB, UP>;
    static bool set = false;
    if (!set) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most) != hipSuccess) return BR_LAUNCH_FAILED;
        set = true;
    }
    const size_t lds = ring + (size_t)(2 * E + 4) * 4 + (size_t)pairs * 4;
    kern<<<cus, RXW_NW * 64, lds, s>>>((const bf16*)A, (const bf16*)Wt, first, order, C, pairs, E, N, K, top, limit, alpha, group);
    return br_check_launch();
}

// Whether experts_wide_kernel takes `pairs` pairs of E experts' matrices of N rows over K: K in steps of 128 from 256.
extern "C" int br_experts_wide_takes(int E, int N, int K, int pairs) {
    return E > 0 && E <= RXW_MAX_E && N > 0 && K % 128 == 0 && K >= 256 && pairs > 0 && pairs <= RXW_MAX_PAIRS &&
           ((long long)E + pairs / 32) * ((N + 31) / 32) * (K / 128) < (1ll << 31);
}

// The weight rows of a unit for these matrices on this device, 0 without one (tests ask).
extern "C" int br_experts_wide_rows(int E, int N, int up) {
    const int cus = br_device_cus();
    return cus ? 16 * rx_wide_height(E, N, up != 0, cus) : 0;
}

// `up`: Wt [E][2 N][K], A the tokens' rows (through `order`), C bfloat16 [pairs, N]; else Wt [E][N][K], A the pairs' rows, C float
// [pairs, N].  `group`: 0 (the kernel finds by the experts' pairs what is faster), or groups of 32 or 64 pairs.
extern "C" int br_experts_wide(const void* A, const void* Wt, const int* first, const int* order, void* C, int up, int pairs, int E,
                               int N, int K, int top, float limit, float alpha, int group, hipStream_t s) {
    if (pairs <= 0) return BR_OK;
    if (!br_experts_wide_takes(E, N, K, pairs) || top <= 0 || (up && !order) || (((uintptr_t)A | (uintptr_t)Wt) & 15) != 0 ||
        (group != 0 && group != 32 && group != 64))
        return BR_BAD_ARG;
    const int cus = br_device_cus();
    if (!cus) return BR_LAUNCH_FAILED;
#define RX_WIDE(HB_)                                                                                                                        case HB_:                                                                                                                                   return up ? rx_launch_wide<HB_, true>(A, Wt, first, order, C, pairs, E, N, K, top, limit, alpha, group, cus, s)                                   : rx_launch_wide<HB_, false>(A, Wt, first, order, C, pairs, E, N, K, top, limit, alpha, group, cus, s);
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
