// Long prompts through the recurrences over an outer-product state, 16 tokens at a time on the matrix cores' float
// instruction.  For a head with d key channels and e value channels the recurrences of this library with a decay per channel
// are, with S the d x e state (from a slot), w_t the decay of token t per channel, k_t what it writes, q_t what reads,
//
//     S_t = diag(w_t) S_(t-1) + k_t v_t^T,      o_t = S_t^T q_t                                 (INCLUDING the token's own write)
//     S_t = diag(w_t) S_(t-1) + k_t v_t^T,      o_t = (S_(t-1) + diag(u) k_t v_t^T)^T q_t       (a bonus u instead of it)
//     S_t = diag(w_t) S_(t-1) + k_t u_t^T,      u_t = beta_t (v_t - (diag(w_t) S_(t-1))^T k_t)  (the delta rule; o_t as first)
//
// Over a chunk of 16 tokens that starts from S, with products of decays over the chunk only (never a quotient of two):
//     o_t = (q_t . prod_{r <= t} w_r)^T S + sum_{s <= t} A[t, s] v_s,     A[t, s] = sum_c q_t[c] k_s[c] prod_{s < r <= t} w_r[c]
//     S' = diag(prod_r w_r) S + sum_s (k_s . prod_{r > s} w_r) v_s^T
// (with the bonus the products stop before t, and A[t, t] = sum_c q_t u k_t).  The delta rule's u take the place of v there:
// with L[t, s] = beta_t sum_c k_t[c] k_s[c] prod_{s < r <= t} w_r[c] for s < t they are u = U - W S, where the rows of U and W
// follow by U_t = beta_t v_t - sum_s L[t, s] U_s and W_t = beta_t k_t . prod_{r <= t} w_r - sum_s L[t, s] W_s.  Everything but the products with S is the
// same for all columns of the state and for all chunks at once, so `chunk_prepare` makes it for every (chunk, head) in
// parallel, in the order in which a lane of the second kernel wants its operands; `chunk_walk` then walks the chunks of a
// sequence in order, with S in the matrix cores' accumulators, which are at once the second operand of the read-out.  All
// products and sums are float; against a walk token by token only their order differs, and an infinite value or one that is
// not a number shows from its token on, not before.  Chunks are counted from the
// sequence's first token of the step; a chunk's tokens beyond the sequence have decay 1, write nothing and read nothing.
//
// What bounds it: the walk is a serial chain, a chunk of a head of 128 x 128 costing a wave 17 float matrix instructions (32
// cycles each) and twice as much again in operand reads, the exchange of the quarters and the barrier (0.7 us a chunk with a
// workgroup to a compute unit; a deeper ring changes nothing).  A walk token by token is bound by the 49,000 lane operations a
// token of such a head takes.  32 heads of 128 x 128: 2,048 tokens 123 us (30 of them `chunk_prepare`, which is bound by its
// reads and writes), 8,192 tokens 465; token by token, twice in pieces, 307 and 1,153.  64 heads of 64 x 64: 106 and 411,
// token by token 235 and 938.
#include "common.h"

#define CW_C 16            // tokens of a chunk
#define CW_FINITE 3.402823466e38f

__device__ __forceinline__ float cw_row16_sum(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, true));
    return v;
}

template <int N>
__device__ __forceinline__ double cw_sum(const float* x) {
    if constexpr (N == 1) return x[0];
    else return cw_sum<N / 2>(x) + cw_sum<N / 2>(x + N / 2);
}

// Which chunks a launch is over, and where a sequence's lie in the scratch.  All at once (`run` 0): sequence s has room for
// ceil(tokens / 16) chunks from cu[s] / 16 + s on.  Where the scratch is smaller: chunks `from` .. from + run of every sequence,
// those of the i-th of the `longs` sequences of at least `least` tokens from i run on; the states wait in their slots
// between the launches, so the bits are the same.
struct CwPart {
    int least, longs, from, run;
};
__device__ __forceinline__ int cw_first(const int* cu, int s, const CwPart& part) {
    if (!part.run) return cu[s] / CW_C + s;
    int rank = 0;
    for (int i = 0; i < s; ++i) rank += cu[i + 1] - cu[i] >= part.least;
    return rank < part.longs ? rank * part.run : -1;
}
// Floats of a (chunk, head) in the scratch: read factors 16 D | write factors 16 D | A 256 | the chunk's decay D | what its
// rounding left D, and for the delta rule -W 16 D | U 16 e.
__host__ __device__ constexpr int cw_block(int D, int e, bool delta) { return 34 * D + 256 + (delta ? 16 * (D + e) : 0); }

#define CW_GLR 0
#define CW_WKV 1
#define CW_FIXED 2
#define CW_DELTA 3
// q, k: rows `qk_stride` apart, query/key head h / (H / G) at columns D apart; v: rows `v_stride` apart, head h at columns e apart.
//  GLR: k holds the gates' sums, `b1` their bias, `b2` their lower bounds (null: 0): w = b2 + (1 - b2) sigmoid(k + b1), the key
//       1 - w, the query silu(q), as glr_scan_kernel.
//  WKV: `z` (rows `qk_stride` apart) the decays' sums, `b1` their bias, `b2` the bonus: w = exp(-exp(z + b1)), as wkv_scan_kernel.
//  FIXED: w = b1[h], one number a head; `silu`: silu of q, k and v, the latter written back over v for the walk.
//  DELTA: `gb` [T, 2 H] decay and beta a head, or with `gc` [T, H D] a decay a key channel and beta in gb's second half.
struct CwIn {
    const float *q, *k, *z, *b1, *b2, *gb, *gc;
    float* v;
    size_t qk_stride, v_stride;
    const int *cu, *slots;
    int H, G, e, silu;
};

// grid (chunks of the longest sequence in the launch, H, sequences), D threads, a thread a channel.
template <int FORM, int D>
__global__ __launch_bounds__(D) void chunk_prepare_kernel(const CwIn in, const CwPart run, float* __restrict__ scratch) {
    constexpr bool DELTA = FORM == CW_DELTA, WKV = FORM == CW_WKV;
    constexpr int KB = D / 16;
    __shared__ __attribute__((aligned(16))) float stage[KB * 272];        // read factors: [channel / 16][channel % 16 / 4][token][4], padded
    __shared__ float part[(DELTA ? 256 : 136) * (D / 16)];
    __shared__ __attribute__((aligned(16))) float Lm[DELTA ? 256 : 4];
    const int s = blockIdx.z, h = blockIdx.y, c = threadIdx.x, H = in.H, e = in.e;
    if (in.slots[s] < 0) return;
    const int t0 = in.cu[s] + (run.from + (int)blockIdx.x) * CW_C, n = min(CW_C, in.cu[s + 1] - t0);
    if (n <= 0 || in.cu[s + 1] - in.cu[s] < run.least) return;
    const int first = cw_first(in.cu, s, run);
    if (first < 0) return;
    const int kh = h / (H / in.G);
    float q[CW_C], k[CW_C], w[CW_C], beta[DELTA ? CW_C : 1];
    const float bias = (FORM == CW_GLR || WKV) && in.b1 ? in.b1[h * D + c] : 0.f, low = (FORM == CW_GLR || WKV) && in.b2 ? in.b2[h * D + c] : 0.f;
#pragma unroll
    for (int t = 0; t < CW_C; ++t) {
        const size_t row = (size_t)(t0 + min(t, n - 1));
        q[t] = in.q[row * in.qk_stride + kh * D + c];
        k[t] = in.k[row * in.qk_stride + kh * D + c];
        w[t] = WKV ? in.z[row * in.qk_stride + h * D + c] : FORM == CW_FIXED ? in.b1[h] : 0.f;
        if (DELTA) {
            w[t] = in.gc ? in.gc[row * H * D + h * D + c] : in.gb[row * 2 * H + h];
            beta[DELTA ? t : 0] = t < n ? in.gb[row * 2 * H + H + h] : 0.f;
        }
    }
#pragma unroll
    for (int t = 0; t < CW_C; ++t) {
        if (FORM == CW_GLR) {
            // as glr_scan_kernel applies them: exp and reciprocal by the hardware's own instructions (about an ulp each)
            const float gt = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * (k[t] + bias)));
            q[t] = q[t] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * q[t]));
            w[t] = low + (1.0f - low) * gt;
            k[t] = 1.0f - w[t];
        } else if (WKV) {
            w[t] = expf(-expf(w[t] + bias));
        } else if (FORM == CW_FIXED && in.silu) {
            q[t] = q[t] / (1.0f + expf(-q[t]));
            k[t] = k[t] / (1.0f + expf(-k[t]));
        }
        if (t >= n) { q[t] = 0.f; k[t] = 0.f; w[t] = 1.f; }
    }
    if (FORM == CW_FIXED && in.silu) {
        for (int i = c; i < n * e; i += D) {
            float* x = in.v + (size_t)(t0 + i / e) * in.v_stride + h * e + i % e;
            const float y = *x;
            *x = y / (1.0f + expf(-y));
        }
    }
    float* out = scratch + ((size_t)(first + (int)blockIdx.x) * H + h) * cw_block(D, e, DELTA);
    // A (and L): 136 (120) sums over the channels, 16 lanes at a time here
    int pair = 0;
#pragma unroll
    for (int j = 0; j < CW_C; ++j) {
        float g = k[j];
#pragma unroll
        for (int t = j; t < CW_C; ++t) {
            float term;
            if (!WKV) {
                if (t > j) g *= w[t];
                term = q[t] * g;
            } else {
                if (t > j + 1) g *= w[t - 1];
                term = t == j ? q[t] * (low * g) : q[t] * g;
            }
            term = cw_row16_sum(term);
            if ((c & 15) == 0) part[pair * (D / 16) + (c >> 4)] = term;
            if (DELTA && t > j) {
                term = cw_row16_sum(k[t] * g);
                if ((c & 15) == 0) part[(136 + pair - j - 1) * (D / 16) + (c >> 4)] = term;      // 120 pairs s < t: j + 1 diagonals before
            }
            ++pair;
        }
    }
    // the factors: prefix products for what reads, suffix products for what writes, rounded to float once at their end
    double p = 1.0;
    float W[DELTA ? CW_C : 1];
#pragma unroll
    for (int t = 0; t < CW_C; ++t) {
        if (!WKV) p *= w[t];
        stage[(c >> 4) * 272 + ((c >> 2) & 3) * 68 + t * 4 + (c & 3)] = (float)(q[t] * p);
        if (DELTA) W[DELTA ? t : 0] = (float)(beta[DELTA ? t : 0] * (k[t] * p));
        if (WKV) p *= w[t];
    }
    // a decay that is the same in every chunk must not carry the same rounding error through all of them
    out[32 * D + 256 + c] = (float)p;
    out[33 * D + 256 + c] = (float)(p - (float)p);
    p = 1.0;
#pragma unroll
    for (int t = CW_C - 1; t >= 0; --t) {
        const float x = w[t];
        w[t] = (float)(k[t] * p);
        p *= x;
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const f32x4 v = {w[g], w[4 + g], w[8 + g], w[12 + g]};
        *(f32x4*)(out + 16 * D + (c >> 4) * 256 + (16 * g + (c & 15)) * 4) = v;
    }
    __syncthreads();
    auto unstage = [&](float* to) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int f = c + i * D, l = f & 63;
            *(f32x4*)(to + f * 4) = *(const f32x4*)(stage + (f >> 6) * 272 + (l >> 4) * 68 + (l & 15) * 4);
        }
    };
    unstage(out);
    for (int i = c; i < 256; i += D) {
        const int t = i >> 4, j = i & 15;
        float sum = 0.f;
        if (j <= t) {
            const float* pp = part + (j * CW_C - j * (j - 1) / 2 + t - j) * (D / 16);
            sum = (float)cw_sum<D / 16>(pp);
        }
        out[32 * D + i] = sum;
        if (DELTA) {
            sum = 0.f;
            if (j < t) {
                const float* pp = part + (136 + j * CW_C - j * (j - 1) / 2 + t - j - j - 1) * (D / 16);
                sum = t < n ? (float)(cw_sum<D / 16>(pp) * in.gb[(size_t)(t0 + t) * 2 * H + H + h]) : 0.f;
            }
            Lm[DELTA ? i : 0] = sum;
        }
    }
    if constexpr (DELTA) {
        __syncthreads();
        auto solve = [&](float (&x)[CW_C]) {                  // x_t -= sum_{s < t} L[t, s] x_s
#pragma unroll
            for (int t = 1; t < CW_C; ++t) {
                float sum = 0.f;
#pragma unroll
                for (int j = 0; j < t; ++j) sum = fmaf(Lm[t * 16 + j], x[j], sum);
                x[t] -= sum;
            }
        };
        solve(W);
        // token t in row 4 (t % 4) + t / 4 of the product with S, so that its results lie as the state's update wants them
#pragma unroll
        for (int t = 0; t < CW_C; ++t) stage[(c >> 4) * 272 + ((c >> 2) & 3) * 68 + (4 * (t & 3) + (t >> 2)) * 4 + (c & 3)] = -W[t];
        float* uo = out + 50 * D + 256;
        for (int x = c; x < e; x += D) {
            float u[CW_C];
#pragma unroll
            for (int t = 0; t < CW_C; ++t) u[t] = beta[t] * in.v[(size_t)(t0 + min(t, n - 1)) * in.v_stride + h * e + x];
            solve(u);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 v = {u[g], u[4 + g], u[8 + g], u[12 + g]};
                *(f32x4*)(uo + (x >> 4) * 256 + (16 * g + (x & 15)) * 4) = v;
            }
        }
        __syncthreads();
        unstage(out + 34 * D + 256);
    }
}

// The sequence that `rank` others of a step are longer than (of equal ones: that come before it).  Steps of more than 64 sequences: as they come.
// Where they come longest first, nothing is looked for; else bit by bit the largest key that more than `rank` are not below (counted one after
// another, 64 sequences of 50 tokens took 336 us where the walk alone takes 286).
__device__ __forceinline__ int cw_by_length(const int* cu, int B, int rank) {
    if (B > 64) return rank;
    const int lane = threadIdx.x & 63, at = lane < B ? lane : B - 1;
    const int len = cu[at + 1] - cu[at], next = lane + 1 < B ? cu[at + 2] - cu[at + 1] : 0;
    if (!__any(next > len)) return rank;
    // above any other length the index alone counts, as for lengths that are equal
    const int key = lane < B ? (len < (1 << 24) ? len : (1 << 24)) * 64 + 63 - lane : -1;
    const int most = __builtin_amdgcn_readfirstlane(cu[B] - cu[0]);
    int found = 0;
    for (int bit = 31 - __clz((most < (1 << 24) ? most : (1 << 24)) | 1) + 6; bit >= 0; --bit) {
        const int higher = found | 1 << bit;
        if (__popcll(__ballot(key >= higher)) > rank) found = higher;
    }
    return __ffsll((unsigned long long)__ballot(key == found)) - 1;
}

// A workgroup walks a sequence's chunks for 16 CB columns of one head; wave w holds the state's rows w D / 4 .. + D / 4 and adds a
// quarter of every output element (its rows' share and, of the sum over A, the tokens 4 w .. + 4), the quarters are added
// in a fixed order through LDS a chunk later.  Sums are kept short and their largest terms late, so that they round about as
// often as a walk token by token: the products with S in chains of 8 terms that are added in pairs, A's on top of them, the
// state's update in the order of the tokens.  Error against 64 bits over 96 to 1,801 tokens with gates from nearly 0 to nearly 1, as a
// share of the walk's: outputs 0.47 to 0.97, gated 0.86 to 1.09 (5.6e-8 of the norm against 5.3e-8); states 0.39 to 1.06, gated to 1.27
// where both are about one rounding (3.9e-8 against 3.1e-8).  With one chain a sum, float products of decays and the rounded decay
// alone the outputs were at 1.0 to 3.0 and the states at up to 2.6.  S chunks of everything a chunk needs lie in an LDS ring filled
// by direct loads; one barrier a chunk.  Registers for two workgroups to a compute unit, all of them ordinary ones: with room for twice
// as many the compiler keeps the sums in accumulation registers and moves the state back and forth.  That, with the chunk before left
// and A's product formed behind the update, took 142 us for 2,048 tokens of 32 heads where this takes 123 (a fixed decay 148 and 125,
// delta rule 213 and 190; 64 heads of 64 x 64 113 and 106).  v: the values' columns of the rows, `ldv` apart.  grid (sequences * H,
// e / (16 CB)), or where H is a multiple of 8 (H, e / (16 CB), sequences), the longest first: the workgroups of a head on one XCD where sequences * H
// is a multiple of 8, and what a step's longest sequences need is not behind the others (with the sequences side by side two workgroups of the longest
// shared a compute unit while others lay idle: 32 heads of 128 x 128, gated, 3,517 and 1,501 tokens 296 -> 247 us, 1,307, 804 and 301 142 -> 117, three times
// 1,200, 300, 150 and 96 291 -> 224; equal ones as before).
template <int D, int CB, int S, int FORM>
__global__ __launch_bounds__(256, 2) void chunk_walk_kernel(const float* __restrict__ scratch, const float* __restrict__ v, int ldv,
                                                            float* __restrict__ o, float* __restrict__ state, size_t slot_stride,
                                                            const int* __restrict__ cu_seqlens, const int* __restrict__ slots, int H, int e,
                                                            int zero_padding, const CwPart run) {
    constexpr bool DELTA = FORM == CW_DELTA, FIXED = FORM == CW_FIXED;
    constexpr int NKB = D / 64, RPL = D / 16, STAGE = ((DELTA ? 48 : 32) * D + 512 + 256 * CB) * 4, L = (DELTA ? 3 : 2) * NKB + 1;
    constexpr int PB = DELTA ? 1 : 2;                         // buffers of output quarters
    const int BLOCK = cw_block(D, e, DELTA);
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    float* part = (float*)(smem + S * STAGE);                 // [PB][4][CB][16][17]
    float* pu = part + PB * 4 * CB * 272;                     // DELTA: [4][CB][64][4] the waves' shares of -W S
    const int s = gridDim.z > 1 ? cw_by_length(cu_seqlens, gridDim.z, blockIdx.z) : blockIdx.x / H, h = blockIdx.x % H, cb = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int slot = slots[s], he = H * e;
    int t0 = cu_seqlens[s], t1 = cu_seqlens[s + 1];
    const int first = cw_first(cu_seqlens, s, run);
    if (t1 - t0 < run.least || first < 0) return;
    if (run.run) {
        t0 += run.from * CW_C;
        t1 = min(t1, t0 + run.run * CW_C);
    }
    if (slot < 0) {
        if (zero_padding)
            for (int i = tid; i < (t1 - t0) * 16; i += 256) for (int x = 0; x < CB; ++x) o[(size_t)(t0 + (i >> 4)) * he + h * e + (cb * CB + x) * 16 + (i & 15)] = 0.f;
        return;
    }
    const int nch = (t1 - t0 + CW_C - 1) / CW_C;
    if (nch <= 0) return;
    const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)smem);
    const float* blocks = scratch + ((size_t)first * H + h) * BLOCK;
    // a stage: read factors | write factors | A | both parts of the decay | values (256 floats each of the last three); a lane's byte offsets
    // within a chunk's block, the block itself is a scalar address that goes on by a chunk's blocks
    unsigned qoff[NKB], koff[NKB];
#pragma unroll
    for (int j = 0; j < NKB; ++j) {
        qoff[j] = (unsigned)((wave * NKB + j) * 1024 + lane * 16);
        koff[j] = qoff[j] + D * 64;
    }
    // waves 0 and 1 bring A and the decay's 2 D floats, waves 2 and 3 the values (both the same 16 columns, or 16 each): L loads a wave
    const unsigned moff = wave == 0 ? 128 * D + lane * 16 : 128 * D + 1024 + (lane * 16) % (8 * D);
    const unsigned values = wave < 2 ? 0u : ~0u;
    const unsigned long long values64 = wave < 2 ? 0ull : ~0ull;
    unsigned long long block = (unsigned long long)blocks;
    const int vx = cb * CB + (CB == 2 ? wave & 1 : 0);        // the 16 columns this wave brings values of
    unsigned long long vbase = (unsigned long long)(v + (size_t)t0 * ldv + h * e + vx * 16);      // the chunk's first row: rows of a prompt reach beyond 4 GB
    const unsigned vcol = ((lane & 3) ^ (lane >> 4)) * 16, uoff = (50 * D + 256) * 4 + vx * 1024 + lane * 16;
    const int vrow = lane >> 2;
    int vlast = t1 - 1 - t0, left = nch - 1, slot_i = 0;      // the sequence's last row, counted from the chunk's first
    auto bring = [&](unsigned lds, unsigned off, unsigned long long base) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "m0", "memory");
    };
    // The next chunk, or behind the last one that again, into a stage nobody reads: no branch stands between a matrix
    // instruction and the reads of its result, where the compiler has been seen to leave out the idle states they need.
    auto issue = [&]() {
        const unsigned base = __builtin_amdgcn_readfirstlane(lds0 + slot_i * STAGE);
#pragma unroll
        for (int j = 0; j < NKB; ++j) {
            bring(base + (wave * NKB + j) * 1024, qoff[j], block);
            bring(base + D * 64 + (wave * NKB + j) * 1024, koff[j], block);
            if (DELTA) bring(base + (32 * D + 512 + 256 * CB) * 4 + (wave * NKB + j) * 1024, qoff[j] + (34 * D + 256) * 4, block);
        }
        const unsigned voff = DELTA ? uoff : (unsigned)min(vrow, vlast) * (unsigned)ldv * 4 + vcol;
        bring(base + D * 128 + min(wave, 1 + CB) * 1024, (moff & ~values) | (voff & values),
              DELTA ? block : (block & ~values64) | (vbase & values64));
        const int go = left > 0;
        block += (unsigned long long)(go * H) * (unsigned)(BLOCK * 4);
        vbase += (unsigned long long)(go * CW_C * 4) * (unsigned)ldv;
        vlast -= go * CW_C;
        left -= go;
        slot_i = slot_i == S - 1 ? 0 : slot_i + 1;
    };
    f32x4 st[CB][NKB];
    float* S0[CB];
#pragma unroll
    for (int x = 0; x < CB; ++x) {
        const int c = (cb * CB + x) * 16 + r16;
        S0[x] = state + (size_t)slot * slot_stride + ((size_t)h * ((e + 3) >> 2) + (c >> 2)) * RPL * 64 + 16 * (c & 3);
#pragma unroll
        for (int j = 0; j < NKB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int k = 16 * (wave * NKB + j) + 4 * g + r;
                st[x][j][r] = S0[x][(size_t)(k % RPL) * 64 + k / RPL];
            }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // from here on only the ring's loads are counted
#pragma unroll
    for (int j = 0; j < S - 1; ++j) issue();
    const int ot = tid >> 4;
    float* op = o + (size_t)(t0 + ot) * he + h * e + cb * CB * 16 + (tid & 15);       // this thread's element of the chunk before
    float quarter[CB][4];                                     // of chunk ch's output elements, chunks in order
    auto collect = [&](int ch) {
#pragma unroll
        for (int x = 0; x < CB; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) quarter[x][y] = part[((ch & (PB - 1)) * 4 * CB + y * CB + x) * 272 + ot * 17 + (tid & 15)];
    };
    auto leave = [&](int ch) {
#pragma unroll
        for (int x = 0; x < CB; ++x) {
            const double v = ((double)quarter[x][0] + quarter[x][1]) + ((double)quarter[x][2] + quarter[x][3]);
            if (t0 + ch * CW_C + ot < t1) op[x * 16] = (float)v;
        }
        op += (size_t)CW_C * he;
    };
    const float* sf = (const float*)smem;                     // the stage in use
    int cur = 0;
    for (int ch = 0; ch < nch; ++ch) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * L) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        // the operands first: the matrix instructions start as soon as they are there, the rest runs beside them
        f32x4 qf[NKB], kf[NKB], dec[NKB], rest[FIXED ? NKB : 1];
        float vv[CB][4], va[CB], vz[CB];
        const float a = sf[32 * D + r16 * 16 + 4 * wave + g];
#pragma unroll
        for (int j = 0; j < NKB; ++j) qf[j] = *(const f32x4*)(sf + (wave * NKB + j) * 256 + lane * 4);
#pragma unroll
        for (int j = 0; j < NKB; ++j) {
            const int kb = wave * NKB + j;
            dec[j] = *(const f32x4*)(sf + 32 * D + 256 + 16 * kb + 4 * g);
            if constexpr (FIXED) rest[j] = *(const f32x4*)(sf + 33 * D + 256 + 16 * kb + 4 * g);
            kf[j] = *(const f32x4*)(sf + 16 * D + kb * 256 + lane * 4);
        }
        // factors of this wave's rows times the state, in chains of 8 rows
        auto times_state = [&](const f32x4 (&f)[NKB], f32x4 (&to)[CB][2 * NKB]) {
#pragma unroll
            for (int j = 0; j < NKB; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int x = 0; x < CB; ++x) {
                        f32x4 from = {0.f, 0.f, 0.f, 0.f};
                        if (r & 1) from = to[x][2 * j + r / 2];
                        to[x][2 * j + r / 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[j][r], st[x][j][r], from, 0, 0, 0);
                    }
        };
        auto pairs = [&](const f32x4 (&p)[2 * NKB]) {
            if constexpr (NKB == 1) return p[0] + p[1];
            else return (p[0] + p[1]) + (p[2] + p[3]);
        };
        // The decayed state, on which the chunk's writes are summed.  A decay that never changes (FIXED) rounds it once: what it and the
        // decay's own rounding leave goes ahead of the chunk's writes, and their sum onto the state.
        f32x4 kept[CB][NKB], add[CB][NKB];
        auto decay = [&]() {
#pragma unroll
            for (int j = 0; j < NKB; ++j)
#pragma unroll
                for (int x = 0; x < CB; ++x)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float old = st[x][j][r], k = old * dec[j][r];
                        kept[x][j][r] = k;
                        add[x][j][r] = FIXED ? fmaf(old, rest[FIXED ? j : 0][r], fmaf(old, dec[j][r], -k)) : k;
                    }
        };
        f32x4 ro[CB][2 * NKB];
        if constexpr (DELTA) {
            f32x4 uf[CB], wf[NKB], pa[CB][2 * NKB];
#pragma unroll
            for (int j = 0; j < NKB; ++j) wf[j] = *(const f32x4*)(sf + 32 * D + 512 + 256 * CB + (wave * NKB + j) * 256 + lane * 4);
#pragma unroll
            for (int x = 0; x < CB; ++x) uf[x] = *(const f32x4*)(sf + 32 * D + 512 + x * 256 + lane * 4);
            times_state(wf, pa);
            times_state(qf, ro);
            decay();
#pragma unroll
            for (int x = 0; x < CB; ++x) *(f32x4*)(pu + ((wave * CB + x) * 64 + lane) * 4) = pairs(pa[x]);
            if (ch > 0) {
                collect(ch - 1);
                leave(ch - 1);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int x = 0; x < CB; ++x) {                    // u = U - W S
                f32x4 share[4];
#pragma unroll
                for (int y = 0; y < 4; ++y) share[y] = *(const f32x4*)(pu + ((y * CB + x) * 64 + lane) * 4);
                const f32x4 u = uf[x] + ((share[0] + share[1]) + (share[2] + share[3]));
#pragma unroll
                for (int r = 0; r < 4; ++r) vv[x][r] = u[r];
                va[x] = wave < 2 ? (wave == 0 ? u[0] : u[1]) : (wave == 2 ? u[2] : u[3]);
            }
        } else {
#pragma unroll
            for (int x = 0; x < CB; ++x) {
                va[x] = sf[32 * D + 512 + x * 256 + (4 * wave + g) * 16 + (((r16 >> 2) ^ wave) << 2) + (r16 & 3)];
#pragma unroll
                for (int i = 0; i < 4; ++i) vv[x][i] = sf[32 * D + 512 + x * 256 + (4 * i + g) * 16 + (((r16 >> 2) ^ i) << 2) + (r16 & 3)];
            }
        }
        // A's zeros above the diagonal keep a token's value from the tokens before it only while it is finite: others pass here as
        // zero and are added to their own and later tokens' sums below
        unsigned long long odd = 0;
#pragma unroll
        for (int x = 0; x < CB; ++x) {
            const bool fine = fabsf(va[x]) <= CW_FINITE;
            odd |= __ballot(!fine);
            vz[x] = fine ? va[x] : 0.f;
        }
        // Everything that is not on the chain from one chunk's state to the next stands between matrix instructions: the chunk before
        // leaves while the products with S run, A's product half way through the update, so that its results are there at the end
        if constexpr (!DELTA) {
            if (ch > 0) collect(ch - 1);
            times_state(qf, ro);
            decay();
            if (ch > 0) leave(ch - 1);
        }
        issue();
        auto update = [&](int i0, int i1) {
#pragma unroll
            for (int i = i0; i < i1; ++i)
#pragma unroll
                for (int j = 0; j < NKB; ++j)
#pragma unroll
                    for (int x = 0; x < CB; ++x) add[x][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][i], vv[x][i], add[x][j], 0, 0, 0);
        };
        f32x4 outs[CB];
        update(0, 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < CB; ++x) outs[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, vz[x], pairs(ro[x]), 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        update(2, 4);
#pragma unroll
        for (int j = 0; j < NKB; ++j)
#pragma unroll
            for (int x = 0; x < CB; ++x) st[x][j] = FIXED ? kept[x][j] + add[x][j] : add[x][j];
#pragma unroll
        for (int x = 0; x < CB; ++x) {
            float* pw = part + (((ch & (PB - 1)) * 4 + wave) * CB + x) * 272;
#pragma unroll
            for (int r = 0; r < 4; ++r) pw[(4 * g + r) * 17 + r16] = outs[x][r];
        }
        if (odd) {                                            // infinite or not a number: this wave's tokens 4 wave + i of A
            for (int x = 0; x < CB; ++x) {
                float* pw = part + (((ch & (PB - 1)) * 4 + wave) * CB + x) * 272;
                for (int i = 0; i < 4; ++i) {
                    const float u = __shfl(va[x], 16 * i + r16, 64);
                    for (int r = 0; r < 4; ++r)
                        if (!(fabsf(u) <= CW_FINITE) && 4 * wave + i <= 4 * g + r) pw[(4 * g + r) * 17 + r16] += sf[32 * D + (4 * g + r) * 16 + 4 * wave + i] * u;
                }
            }
        }
        cur = cur == S - 1 ? 0 : cur + 1;
        sf = (const float*)(smem + cur * STAGE);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");          // no load into LDS outlives the workgroup
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    collect(nch - 1);
    leave(nch - 1);
#pragma unroll
    for (int x = 0; x < CB; ++x)
#pragma unroll
        for (int j = 0; j < NKB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int k = 16 * (wave * NKB + j) + 4 * g + r;
                S0[x][(size_t)(k % RPL) * 64 + k / RPL] = st[x][j][r];
            }
}

// Whether a head of d x e goes this way.
extern "C" int br_chunk_takes(int d, int e) { return (d == 64 || d == 128) && e > 0 && e % 16 == 0; }
// Floats of scratch for a chunk of all heads, and for all of T tokens of B sequences at once.
extern "C" size_t br_chunk_block(int H, int d, int e, int delta) { return (size_t)H * (size_t)cw_block(d, e, delta != 0); }
extern "C" size_t br_chunk_scratch(int T, int B, int H, int d, int e, int delta) {
    return (size_t)(T / CW_C + B + 1) * br_chunk_block(H, d, e, delta);
}

template <int D, int CB, int S, int FORM>
static int chunk_walk(const CwIn& in, const CwPart& part, const float* scratch, float* o, float* state, size_t slot_stride, int B,
                      int zero_padding, hipStream_t s) {
    constexpr bool DELTA = FORM == CW_DELTA;
    constexpr size_t lds = (size_t)S * ((DELTA ? 48 : 32) * D + 512 + 256 * CB) * 4 + (DELTA ? 1 : 2) * 4 * CB * 272 * 4 + (DELTA ? 4096 * CB : 0);
    static_assert(lds <= 160 * 1024, "LDS");
    auto walk = chunk_walk_kernel<D, CB, S, FORM>;
    static bool set = false;
    if (!set) {
        if (hipFuncSetAttribute((const void*)walk, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) return BR_LAUNCH_FAILED;
        set = true;
    }
    const dim3 grid = in.H % 8 == 0 && B <= 65535 ? dim3(in.H, in.e / (16 * CB), B) : dim3(B * in.H, in.e / (16 * CB));
    walk<<<grid, 256, lds, s>>>(scratch, in.v, (int)in.v_stride, o, state, slot_stride, in.cu, in.slots, in.H, in.e, zero_padding, part);
    return br_check_launch();
}

template <int FORM, int D>
static int chunk_run(const CwIn& in, const CwPart& part, float* o, float* state, size_t slot_stride, float* scratch, int B, int chunks,
                     int T, int max_new, hipStream_t s) {
    constexpr bool DELTA = FORM == CW_DELTA;
    chunk_prepare_kernel<FORM, D><<<dim3(chunks, in.H, B), D, 0, s>>>(in, part, scratch);
    const int rc = br_check_launch();
    if (rc != BR_OK) return rc;
    // 16 columns a workgroup as long as the tokens are those of few sequences as long as the longest: 2.5 workgroups of 16 columns to a compute unit
    // (delta rule with heads of 128, which holds the most in LDS: 1.9), or 3 (1) of about equal ones, whose last round is as long as the others.
    // Beyond, 32 columns, which share a chunk's loads.  us with 16 / 32: 32 heads of 128 x 128, gated, 2,048 tokens 127 / 168, 3,517 and 1,501 tokens
    // 264 / 308, 1,307, 804 and 301 121 / 136, 1,500, 700, 400 and 200 145 / 156, 1,300, 900, 700, 500 and 300 186 / 161, three times 1,000 155 / 152, four
    // times 900 175 / 152, 16 times 300 256 / 220, 64 times 50 339 / 290; fixed, 1,307, 804 and 301 127 / 142; delta rule, 2,048 tokens 189 / 275, 3,517 and 1,501
    // 455 / 579, 1,307, 804 and 301 231 / 236, 1,500, 700, 400 and 200 270 / 284, twice 1,000 186 / 173, 700, 650 and 600 185 / 169; 16 heads, twice 1,000
    // 104 / 146, three times 171 / 158, 1,300 .. 300 184 / 212; 64 heads of 64 x 64, WKV, 3,517 and 1,501 219 / 249, 1,300 .. 300 159 / 141; 12 heads, delta rule, 16
    // times 300 75 / 86.
    const int cus = br_device_cus();
    if (!cus) return BR_LAUNCH_FAILED;
    const bool equal = (double)T >= 0.9 * max_new * part.longs, held = D == 128 && DELTA;
    const double units = (equal ? (double)part.longs : (double)T / max_new) * in.H * (in.e / 16);
#define CW_WALK(CB, S) return chunk_walk<D, CB, S, FORM == CW_WKV ? CW_GLR : FORM>(in, part, scratch, o, state, slot_stride, B, FORM != CW_GLR, s)
    if (in.e % 32 || units <= (equal ? (held ? 1.0 : 3.0) : (held ? 1.9 : 2.5)) * cus) CW_WALK(1, (D == 64 ? 4 : 3));
    if constexpr (DELTA) CW_WALK(2, (D == 64 ? 4 : 2));
    else CW_WALK(2, (D == 64 ? 5 : 3));
#undef CW_WALK
}

// One step's tokens of B sequences (`max_new` the most a sequence brings) through a recurrence (see CwIn for the forms' inputs),
// from and into the slots' states.  Sequences of fewer than `least` tokens are left alone: their outputs and states are another
// kernel's.  `scratch`: br_chunk_scratch floats, or fewer, then the chunks are taken in several launches; at least a chunk of each of
// the `longs` sequences that are not left alone.
extern "C" int br_chunk_scan(int form, const float* q, const float* k, float* v, size_t qk_stride, size_t v_stride, const float* z,
                             const float* b1, const float* b2, const float* gb, const float* gc, int silu, float* o, float* state,
                             size_t slot_stride, const int* cu_seqlens, const int* slots, float* scratch, size_t scratch_floats, int T,
                             int B, int H, int G, int d, int e, int max_new, int least, int longs, hipStream_t s) {
    if (B <= 0 || T <= 0) return BR_OK;
    if (!br_chunk_takes(d, e) || H <= 0 || H > 65535 || B > 65535 || (long long)B * H > 0x7fffffffLL || e / 16 > 65535 || max_new <= 0 ||
        max_new > T || G <= 0 || H % G || form < CW_GLR || form > CW_DELTA || v_stride % 4 || ((uintptr_t)v | (uintptr_t)scratch) % 16 ||
        v_stride >= (1ull << 26) || slot_stride < (size_t)H * ((e + 3) / 4) * d * 4 ||
        longs <= 0 || longs > B || scratch_floats < longs * br_chunk_block(H, d, e, form == CW_DELTA) || (form == CW_WKV && (!z || !b1 || !b2)) ||
        (form == CW_FIXED && !b1) || (form == CW_DELTA && !gb) || ((form == CW_GLR || form == CW_WKV) && G != H))
        return BR_BAD_ARG;
    const CwIn in = {q, k, z, b1, b2, gb, gc, v, qk_stride, v_stride, cu_seqlens, slots, H, G, e, silu};
    const int all = (max_new + CW_C - 1) / CW_C;
    const bool once = scratch_floats >= br_chunk_scratch(T, B, H, d, e, form == CW_DELTA);
    int run = all;
    if (!once) {
        const size_t room = scratch_floats / br_chunk_block(H, d, e, form == CW_DELTA) / longs;
        run = room < (size_t)all ? (int)room : all;
    }
    for (int from = 0; from < all; from += run) {
        const CwPart part = {least, longs, from, once ? 0 : run};
        const int chunks = all - from < run ? all - from : run;
#define CW_RUN(F) d == 64 ? chunk_run<F, 64>(in, part, o, state, slot_stride, scratch, B, chunks, T, max_new, s) : chunk_run<F, 128>(in, part, o, state, slot_stride, scratch, B, chunks, T, max_new, s)
        const int rc = form == CW_GLR ? CW_RUN(CW_GLR) : form == CW_WKV ? CW_RUN(CW_WKV) : form == CW_FIXED ? CW_RUN(CW_FIXED) : CW_RUN(CW_DELTA);
#undef CW_RUN
        if (rc != BR_OK) return rc;
    }
    return BR_OK;
}
