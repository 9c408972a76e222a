// Long prompts through the recurrences over an outer-product state, 16 tokens at a time on the matrix cores' float
// instruction.  For a head with d key channels and e value channels the recurrences of this library with a decay per channel
// are, with S the d x e state (from a slot), w_t the decay of token t per channel, k_t what it writes, q_t what reads,
//
//     S_t = diag(w_t) S_(t-1) + k_t v_t^T,      o_t = S_t^T q_t                                 (INCLUDING the token's own write)
//     S_t = diag(w_t) S_(t-1) + k_t v_t^T,      o_t = (S_(t-1) + diag(u) k_t v_t^T)^T q_t       (a bonus u instead of it)
//
// Over a chunk of 16 tokens that starts from S, with products of decays over the chunk only (never a quotient of two):
//     o_t = (q_t . prod_{r <= t} w_r)^T S + sum_{s <= t} A[t, s] v_s,     A[t, s] = sum_c q_t[c] k_s[c] prod_{s < r <= t} w_r[c]
//     S' = diag(prod_r w_r) S + sum_s (k_s . prod_{r > s} w_r) v_s^T
// (with the bonus the products stop before t, and A[t, t] = sum_c q_t u k_t).  Everything but the two products with S is the
// same for all columns of the state and for all chunks at once, so `chunk_prepare` makes it for every (chunk, head) in
// parallel, in the order in which a lane of the second kernel wants its operands; `chunk_walk` then walks the chunks of a
// sequence in order, with S in the matrix cores' accumulators, which are at once the second operand of the read-out.  All
// products and sums are float; against a walk token by token only their order differs.  Chunks are counted from the
// sequence's first token of the step; a chunk's tokens beyond the sequence have decay 1, write nothing and read nothing.
//
// What bounds it: the walk is a serial chain of (17 + 17) / 2 float matrix instructions a wave and chunk (32 cycles each); a
// walk token by token is bound by the 49,000 lane operations a head of 128 x 128 takes a token, the matrix cores take a
// quarter of that time, and only 16 columns' workgroups times 4 waves are needed to have two waves a SIMD.
#include "common.h"

#define CW_C 16            // tokens of a chunk

__device__ __forceinline__ float cw_row16_sum(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, true));
    return v;
}

// Where a sequence's chunks lie in the scratch: sequence s has room for ceil(tokens / 16) chunks from cu[s] / 16 + s on.
__device__ __forceinline__ int cw_first(const int* cu, int s) { return cu[s] / CW_C + s; }
// Floats of a (chunk, head) in the scratch: read factors 16 D | write factors 16 D | A 256 | decay D.
template <int D> constexpr int cw_block() { return 33 * D + 256; }

// rows [T, width] float; FORM 0 (`glr`): q | f at columns 0, H d, `b1` the gate's bias, `b2` its lower bound (null: 0);
// FORM 1 (`wkv`): r | k at 0, H d and z at 2 H d + H e, `b1` the decay's bias, `b2` the bonus.
// grid (chunks of the longest sequence, H, sequences), D threads, a thread a channel.
template <int FORM, int D>
__global__ __launch_bounds__(D) void chunk_prepare_kernel(const float* __restrict__ rows, int width, const float* __restrict__ b1,
                                                          const float* __restrict__ b2, const int* __restrict__ cu_seqlens,
                                                          const int* __restrict__ slots, float* __restrict__ scratch, int H, int e) {
    constexpr int KB = D / 16;
    __shared__ __attribute__((aligned(16))) float stage[KB * 272];        // read factors: [channel / 16][channel % 16 / 4][token][4], padded
    __shared__ float part[136 * (D / 16)];
    const int s = blockIdx.z, h = blockIdx.y, c = threadIdx.x, lane = c & 63;
    if (slots[s] < 0) return;
    const int t0 = cu_seqlens[s] + (int)blockIdx.x * CW_C, n = min(CW_C, cu_seqlens[s + 1] - t0);
    if (n <= 0) return;
    const int hd = H * D;
    float q[CW_C], k[CW_C], w[CW_C];
    const float bias = b1 ? b1[h * D + c] : 0.f, low = b2 ? b2[h * D + c] : 0.f;
#pragma unroll
    for (int t = 0; t < CW_C; ++t) {
        const float* r = rows + (size_t)(t0 + min(t, n - 1)) * width + h * D + c;
        q[t] = r[0];
        k[t] = r[hd];
        w[t] = FORM == 1 ? r[2 * hd + H * e] : 0.f;
    }
#pragma unroll
    for (int t = 0; t < CW_C; ++t) {
        if (FORM == 0) {
            // as glr_scan_kernel applies them: exp and reciprocal by the hardware's own instructions (about an ulp each)
            const float gt = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * (k[t] + bias)));
            q[t] = q[t] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * q[t]));
            w[t] = low + (1.0f - low) * gt;
            k[t] = 1.0f - w[t];
        } else {
            w[t] = expf(-expf(w[t] + bias));
        }
        if (t >= n) { q[t] = 0.f; k[t] = 0.f; w[t] = 1.f; }
    }
    float* out = scratch + ((size_t)(cw_first(cu_seqlens, s) + blockIdx.x) * H + h) * cw_block<D>();
    // A: 136 sums over the channels, 16 lanes at a time here
    int pair = 0;
#pragma unroll
    for (int j = 0; j < CW_C; ++j) {
        float g = k[j];
#pragma unroll
        for (int t = j; t < CW_C; ++t) {
            float term;
            if (FORM == 0) {
                if (t > j) g *= w[t];
                term = q[t] * g;
            } else {
                if (t > j + 1) g *= w[t - 1];
                term = t == j ? q[t] * (low * g) : q[t] * g;
            }
            term = cw_row16_sum(term);
            if ((lane & 15) == 0) part[pair * (D / 16) + (c >> 4)] = term;
            ++pair;
        }
    }
    // the factors: prefix products for what reads, suffix products for what writes
    float p = 1.f;
#pragma unroll
    for (int t = 0; t < CW_C; ++t) {
        if (FORM == 0) p *= w[t];
        stage[(c >> 4) * 272 + ((c >> 2) & 3) * 68 + t * 4 + (c & 3)] = q[t] * p;
        if (FORM == 1) p *= w[t];
    }
    out[32 * D + 256 + c] = p;
    p = 1.f;
#pragma unroll
    for (int t = CW_C - 1; t >= 0; --t) {
        const float x = w[t];
        w[t] = k[t] * p;
        p *= x;
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const f32x4 v = {w[4 * g], w[4 * g + 1], w[4 * g + 2], w[4 * g + 3]};
        *(f32x4*)(out + 16 * D + (c >> 4) * 256 + (16 * g + (c & 15)) * 4) = v;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int f = c + i * D, l = f & 63;
        *(f32x4*)(out + f * 4) = *(const f32x4*)(stage + (f >> 6) * 272 + (l >> 4) * 68 + (l & 15) * 4);
    }
    for (int i = c; i < 256; i += D) {
        const int t = i >> 4, j = i & 15;
        float sum = 0.f;
        if (j <= t) {
            const float* pp = part + (j * CW_C - j * (j - 1) / 2 + t - j) * (D / 16);
#pragma unroll
            for (int x = 0; x < D / 16; ++x) sum += pp[x];
        }
        out[32 * D + i] = sum;
    }
}

// A workgroup walks a sequence's chunks for 16 columns of one head; wave w holds the state's rows w D / 4 .. + D / 4 and adds a
// quarter of every output element (its rows' share and, of the sum over A, the tokens 4 g + w), the quarters are added in
// wave order through LDS a chunk later.  S chunks of everything a chunk needs lie in an LDS ring filled by direct loads; one
// barrier a chunk.  v: the values' columns of the rows, `ldv` apart.  grid (sequences * H, e / 16): the workgroups of a head
// on one XCD where sequences * H is a multiple of 8.
template <int D, int S>
__global__ __launch_bounds__(256) void chunk_walk_kernel(const float* __restrict__ scratch, const float* __restrict__ v, int ldv,
                                                         float* __restrict__ o, float* __restrict__ state, size_t slot_stride,
                                                         const int* __restrict__ cu_seqlens, const int* __restrict__ slots, int H, int e,
                                                         int zero_padding) {
    constexpr int NKB = D / 64, RPL = D / 16, STAGE = (32 * D + 768) * 4, L = 2 * NKB + 1, BLOCK = cw_block<D>();
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    float* part = (float*)(smem + S * STAGE);                 // [2][4][16][17]
    const int s = blockIdx.x / H, h = blockIdx.x - s * H, cb = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int slot = slots[s], t0 = cu_seqlens[s], t1 = cu_seqlens[s + 1], he = H * e;
    if (slot < 0) {
        if (zero_padding)
            for (int i = tid; i < (t1 - t0) * 16; i += 256) o[(size_t)(t0 + (i >> 4)) * he + h * e + cb * 16 + (i & 15)] = 0.f;
        return;
    }
    const int nch = (t1 - t0 + CW_C - 1) / CW_C;
    if (nch <= 0) return;
    const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)smem);
    const float* blocks = scratch + ((size_t)cw_first(cu_seqlens, s) * H + h) * BLOCK;
    auto bring = [&](unsigned lds, const float* p) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(p) : "m0", "memory");
    };
    // a stage: read factors | write factors | A | decay | values (256 floats each of the last three)
    auto issue = [&](int ch) {
        const float* b = blocks + (size_t)ch * H * BLOCK;
        const unsigned st = __builtin_amdgcn_readfirstlane(lds0 + (ch % S) * STAGE);
#pragma unroll
        for (int j = 0; j < NKB; ++j) {
            const int kb = wave * NKB + j;
            bring(__builtin_amdgcn_readfirstlane(st + kb * 1024), b + kb * 256 + lane * 4);
            bring(__builtin_amdgcn_readfirstlane(st + D * 64 + kb * 1024), b + 16 * D + kb * 256 + lane * 4);
        }
        // the decay's D floats: lanes beyond them bring what the first ones bring
        const float* p = wave == 0   ? b + 32 * D + lane * 4
                         : wave == 1 ? b + 32 * D + 256 + (lane * 4) % D
                                     : v + (size_t)min(t0 + ch * CW_C + (lane >> 2), t1 - 1) * ldv + h * e + cb * 16 + ((lane & 3) ^ (lane >> 4)) * 4;
        const int at = wave < 2 ? wave : 2;                   // waves 2 and 3 both bring the values: every wave L loads
        bring(__builtin_amdgcn_readfirstlane(st + D * 128 + at * 1024), p);
    };
    f32x4 st[NKB];
    const int c = cb * 16 + r16;
    float* S0 = state + (size_t)slot * slot_stride + ((size_t)h * ((e + 3) >> 2) + (c >> 2)) * RPL * 64 + 16 * (c & 3);
#pragma unroll
    for (int j = 0; j < NKB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = 16 * (wave * NKB + j) + 4 * g + r;
            st[j][r] = S0[(size_t)(k % RPL) * 64 + k / RPL];
        }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // from here on only the ring's loads are counted
#pragma unroll
    for (int j = 0; j < S - 1; ++j)
        if (j < nch) issue(j);
    const int ot = tid >> 4;
    auto flush = [&](int ch) {                                // the quarters of chunk ch's outputs
        const float* pp = part + (ch & 1) * 4 * 272 + ot * 17 + (tid & 15);
        const int t = t0 + ch * CW_C + ot;
        if (t < t1) o[(size_t)t * he + h * e + cb * 16 + (tid & 15)] = ((pp[0] + pp[272]) + pp[544]) + pp[816];
    };
    for (int ch = 0; ch < nch; ++ch) {
        if (ch + S - 2 < nch) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * L) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (ch > 0) flush(ch - 1);
        if (ch + S - 1 < nch) issue(ch + S - 1);
        const float* sf = (const float*)(smem + (ch % S) * STAGE);
        f32x4 qf[NKB], kf[NKB], dec[NKB];
        float vv[4];
#pragma unroll
        for (int j = 0; j < NKB; ++j) {
            const int kb = wave * NKB + j;
            qf[j] = *(const f32x4*)(sf + kb * 256 + lane * 4);
            kf[j] = *(const f32x4*)(sf + 16 * D + kb * 256 + lane * 4);
            dec[j] = *(const f32x4*)(sf + 32 * D + 256 + 16 * kb + 4 * g);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) vv[i] = sf[32 * D + 512 + (4 * g + i) * 16 + (((r16 >> 2) ^ g) << 2) + (r16 & 3)];
        const float a = sf[32 * D + r16 * 16 + 4 * g + wave];
        const float va = sf[32 * D + 512 + (4 * g + wave) * 16 + (((r16 >> 2) ^ g) << 2) + (r16 & 3)];
        f32x4 oa = {0.f, 0.f, 0.f, 0.f};
        oa = __builtin_amdgcn_mfma_f32_16x16x4f32(a, va, oa, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NKB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) oa = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[j][r], st[j][r], oa, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NKB; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) st[j][r] *= dec[j][r];
#pragma unroll
            for (int i = 0; i < 4; ++i) st[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][i], vv[i], st[j], 0, 0, 0);
        }
        float* pw = part + (ch & 1) * 4 * 272 + wave * 272;
#pragma unroll
        for (int r = 0; r < 4; ++r) pw[(4 * g + r) * 17 + r16] = oa[r];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    flush(nch - 1);
#pragma unroll
    for (int j = 0; j < NKB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = 16 * (wave * NKB + j) + 4 * g + r;
            S0[(size_t)(k % RPL) * 64 + k / RPL] = st[j][r];
        }
}

// Whether a head of d x e goes this way.
extern "C" int br_chunk_takes(int d, int e) { return (d == 64 || d == 128) && e > 0 && e % 16 == 0; }
// Floats of scratch for T tokens of B sequences.
extern "C" size_t br_chunk_scratch(int T, int B, int H, int d) { return (size_t)(T / CW_C + B + 1) * H * (33 * (size_t)d + 256); }

template <int FORM, int D, int S>
static int chunk_run(const float* rows, int width, const float* b1, const float* b2, float* o, float* state, size_t slot_stride,
                     const int* cu, const int* slots, float* scratch, int B, int H, int e, int max_new, hipStream_t s) {
    constexpr size_t lds = (size_t)S * (32 * D + 768) * 4 + 2 * 4 * 272 * 4;
    static_assert(lds <= 80 * 1024, "two workgroups a compute unit");
    auto walk = chunk_walk_kernel<D, S>;
    static bool set = false;
    if (!set) {
        if (hipFuncSetAttribute((const void*)walk, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) return BR_LAUNCH_FAILED;
        set = true;
    }
    chunk_prepare_kernel<FORM, D><<<dim3((max_new + CW_C - 1) / CW_C, H, B), D, 0, s>>>(rows, width, b1, b2, cu, slots, scratch, H, e);
    walk<<<dim3(B * H, e / 16), 256, lds, s>>>(scratch, rows + 2 * H * D, width, o, state, slot_stride, cu, slots, H, e, FORM == 1);
    return br_check_launch();
}

// One step's tokens of B sequences (`max_new` the most a sequence brings) through the recurrence `form` (0: `glr`, 1: `wkv`,
// see chunk_prepare_kernel), from and into the slots' states; `scratch`: br_chunk_scratch floats.
extern "C" int br_chunk_scan(int form, const float* rows, int width, const float* b1, const float* b2, float* o, float* state,
                             size_t slot_stride, const int* cu_seqlens, const int* slots, float* scratch, size_t scratch_floats, int T,
                             int B, int H, int d, int e, int max_new, hipStream_t s) {
    if (B <= 0 || T <= 0) return BR_OK;
    if (!br_chunk_takes(d, e) || H <= 0 || H > 65535 || B > 65535 || (long long)B * H > 0x7fffffffLL || e / 16 > 65535 || max_new <= 0 ||
        max_new > T || (form != 0 && form != 1) || width < (form ? 3 : 2) * H * d + H * e || width % 4 || (uintptr_t)rows % 16 ||
        (uintptr_t)scratch % 16 || slot_stride < (size_t)H * ((e + 3) / 4) * d * 4 || scratch_floats < br_chunk_scratch(T, B, H, d))
        return BR_BAD_ARG;
#define CW_RUN(F, D_, S_) chunk_run<F, D_, S_>(rows, width, b1, b2, o, state, slot_stride, cu_seqlens, slots, scratch, B, H, e, max_new, s)
    if (form == 0) return d == 64 ? CW_RUN(0, 64, 4) : CW_RUN(0, 128, 3);
    return d == 64 ? CW_RUN(1, 64, 4) : CW_RUN(1, 128, 3);
#undef CW_RUN
}
