// Attention over the paged cache, one wave or four per (query token, query head), in float
// arithmetic for both storage types.  It serves prompts and single tokens alike: a
// query at position p of its sequence sees keys lo..p, lo = max(0, p - window + 1),
// all of which are in the cache when it runs (the step stores its own keys first).
//
// The sum runs over keys in chunks of 64 in ascending position, with the online-softmax
// recurrence of the reference (m' = max(m, s), c = exp(m - m'), d = d c + w,
// acc = acc c + w v; kernels/megakernel_ops.hip:2310-2342), scores scaled by `scale`
// (rsqrt(head_dim) there, :2192-2194), kv head = q head / (nq / nkv) (:2192).  Chunk i belongs
// to class i % 4; a class is one such recurrence, and the classes are joined by it in their order.  The
// chunking depends only on (p, window), never on how tokens were cut into steps or on
// what else is in the batch, so whole prompts and token-by-token runs agree bit for bit, also
// between the two forms: one wave a (token, head) for all classes in turn, and where there are
// few (single tokens) a wave a class, so that the classes' reads wait for memory side by side.
//
// This is the whole attention of the 32-bit path and the reference the matrix-core
// kernels are tested against.
#include "common.h"

#define MAX_DPL 8   // head_dim <= 64 * MAX_DPL

// VEC: the rows of keys and the rows of a value channel are read 16 bytes at a time, in the same order of sums (head sizes in
// steps of a 16-byte load, pages of whole 64s, aligned cache).  WIN: behind a window's edge chunks seldom start with a page; their
// values are read one by one up to the first such piece and then so, page by page, in the same order (32 tokens through windows
// of 100, 32 heads of 128 in bfloat16: 30 us; all of them one by one 88, by one wave 64).  A kernel of its own: in the other it takes
// registers (contexts of 2,000 keys without a window, 8 heads of 64, 500 tokens: 520 us, 690 with it).  Bound by the latency of those reads.  Short requests (3 sequences of
// 29 to 163 tokens, 32 heads of 128 in float): a step of single tokens takes 12.8 us with a wave a class, the prompt 94 with one
// wave for all; both forms with one wave and no classes averaged 35 over a prompt and six steps, one element a read 106.
template <typename T> struct as_vec;
template <> struct as_vec<float> { static constexpr int N = 4; typedef f32x4 type; };
template <> struct as_vec<bf16> { static constexpr int N = 8; typedef bf16x8 type; };

struct AsPart { float m, l, acc[MAX_DPL]; };            // a lane's channels lane, lane + 64, ..

// What weights are taken relative to: the largest score so far, and while all of them are minus infinity (weight 0) or not a number
// (which is to show in the sums) a finite one.
__device__ __forceinline__ float as_base(float m) { return m == -INFINITY ? 0.f : m; }

// onto `a` the keys that `b` summed: the recurrence's own step for more than one key
__device__ __forceinline__ void as_join(AsPart& a, const AsPart& b) {
    if (b.m == -INFINITY && b.l == 0.f) return;
    const float m = fmaxf(a.m, b.m), ca = expf(a.m - as_base(m)), cb = expf(b.m - as_base(m));          // exp(-inf) = 0 on the first
    a.l = fmaf(b.l, cb, a.l * ca);
#pragma unroll
    for (int i = 0; i < MAX_DPL; ++i) a.acc[i] = fmaf(b.acc[i], cb, a.acc[i] * ca);
    a.m = m;
}

template <typename T, bool VEC, int WAVES, bool WIN>
__global__ __launch_bounds__(64 * WAVES) void attn_simple_kernel(
    const T* __restrict__ q, size_t q_stride, T* __restrict__ out, const int* __restrict__ pos,
    const int* __restrict__ seq_of_token, const int* __restrict__ slots,
    const int* __restrict__ block_table, int table_stride, const T* __restrict__ cache,
    int nq, int nkv, int hd, int page, int window, float scale) {
    constexpr int VN = as_vec<T>::N;
    typedef typename as_vec<T>::type vec_t;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float* qs = lds;                                     // [hd]
    float* pall = lds + ((hd + 3) & ~3);                 // [WAVES][64]
    float* joinL = pall + WAVES * 64;                    // WAVES 4: [4][2 + hd]
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float* ps = pall + wave * 64;
    const int kvh = h / (nq / nkv);
    T* o = out + ((size_t)t * nq + h) * hd;
    const int slot = slots[seq_of_token[t]];
    if (slot < 0) {
        for (int d = threadIdx.x; d < hd; d += 64 * WAVES) o[d] = from_f32<T>(0.f);
        return;
    }
    const T* qr = q + (size_t)t * q_stride + (size_t)h * hd;
    for (int d = threadIdx.x; d < hd; d += 64 * WAVES) qs[d] = to_f32<T>(qr[d]);
    __syncthreads();
    const int p = pos[t];
    const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    const int* bt = block_table + (size_t)slot * table_stride;
    // one page: [K|V][kvh], keys [tok][hd], values transposed [hd][tok]
    const size_t page_elems = (size_t)2 * nkv * page * hd;
    const size_t k_off = (size_t)kvh * page * hd, v_off = ((size_t)nkv + kvh) * page * hd;

    auto nothing = []() {
        AsPart a;
        a.m = -INFINITY;
        a.l = 0.f;
#pragma unroll
        for (int i = 0; i < MAX_DPL; ++i) a.acc[i] = 0.f;
        return a;
    };
    auto walk = [&](int cls) {
        AsPart a = nothing();
        for (int j0 = lo + 64 * cls; j0 <= p; j0 += 256) {
            const int j = j0 + lane;
            float s = -INFINITY;
            if (j <= p) {
                const T* kr = cache + (size_t)bt[j / page] * page_elems + k_off + (size_t)(j % page) * hd;
                float dot = 0.f;
                if (VEC) {
#pragma unroll 8
                    for (int d = 0; d < hd; d += VN) {
                        const vec_t kv = *(const vec_t*)(kr + d);
#pragma unroll
                        for (int e = 0; e < VN; ++e) dot = fmaf(qs[d + e], to_f32<T>(kv[e]), dot);
                    }
                } else
                    for (int d = 0; d < hd; ++d) dot = fmaf(qs[d], to_f32<T>(kr[d]), dot);
                s = dot * scale;
            }
            const float m_new = fmaxf(a.m, wave_max(s)), base = as_base(m_new);
            const float corr = expf(a.m - base);         // exp(-inf) = 0 on the first chunk
            const float w = (j <= p) ? expf(s - base) : 0.f;
            a.l = fmaf(a.l, corr, wave_sum(w));
            // `ps` is this wave's own: its reads of the chunk before are done, its writes wait here
            __builtin_amdgcn_wave_barrier();
            ps[lane] = w;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            const int nk = (p - j0 + 1) < 64 ? (p - j0 + 1) : 64;
#pragma unroll
            for (int i = 0; i < MAX_DPL; ++i) a.acc[i] *= corr;
            auto one = [&](int jj, const T* vc) {        // key jj of the chunk, its value's channels a page's row apart
                const float pw = ps[jj];
#pragma unroll
                for (int i = 0; i < MAX_DPL; ++i) {
                    const int d = lane + 64 * i;
                    if (d < hd) a.acc[i] = fmaf(pw, to_f32<T>(vc[(size_t)d * page]), a.acc[i]);
                }
            };
            if constexpr (WIN && VEC) {
                for (int jj = 0; jj < nk;) {
                    const int off = (j0 + jj) % page, end = min(nk, jj + page - off);
                    const T* vc = cache + (size_t)bt[(j0 + jj) / page] * page_elems + v_off + off - jj;
                    for (; jj < end && (j0 + jj) % VN; ++jj) one(jj, vc + jj);
#pragma unroll 4
                    for (; jj + VN <= end; jj += VN) {
                        vec_t vv[MAX_DPL];
#pragma unroll
                        for (int i = 0; i < MAX_DPL; ++i)
                            if (64 * i < hd) vv[i] = *(const vec_t*)(vc + (size_t)min(lane + 64 * i, hd - 1) * page + jj);
#pragma unroll
                        for (int i = 0; i < MAX_DPL; ++i)
                            if (64 * i < hd)
#pragma unroll
                                for (int e = 0; e < VN; ++e) a.acc[i] = fmaf(ps[jj + e], to_f32<T>(vv[i][e]), a.acc[i]);
                    }
                    for (; jj < end; ++jj) one(jj, vc + jj);
                }
                a.m = m_new;
                continue;
            }
            int jj = 0;
            if (VEC) {                                   // the chunk lies in one page
                const T* vc = cache + (size_t)bt[j0 / page] * page_elems + v_off + (j0 % page);
#pragma unroll 4
                for (; jj + VN <= nk; jj += VN) {
                    vec_t vv[MAX_DPL];
#pragma unroll
                    for (int i = 0; i < MAX_DPL; ++i)
                        if (64 * i < hd) vv[i] = *(const vec_t*)(vc + (size_t)min(lane + 64 * i, hd - 1) * page + jj);
#pragma unroll
                    for (int i = 0; i < MAX_DPL; ++i)
                        if (64 * i < hd)
#pragma unroll
                            for (int e = 0; e < VN; ++e) a.acc[i] = fmaf(ps[jj + e], to_f32<T>(vv[i][e]), a.acc[i]);
                }
            }
            for (; jj < nk; ++jj) {
                const int jk = j0 + jj;
                one(jj, cache + (size_t)bt[jk / page] * page_elems + v_off + (jk % page));
            }
            a.m = m_new;
        }
        return a;
    };
    AsPart a;
    if (WAVES == 1) {
        // with windows the walk stands here once, in the loop: twice it takes registers that a third of the waves are missing
        constexpr bool ONCE = WIN && VEC;
        a = ONCE ? nothing() : walk(0);
        for (int cls = ONCE ? 0 : 1; cls < 4 && lo + 64 * cls <= p; ++cls) as_join(a, walk(cls));
    } else {
        a = walk(wave);
        float* part = joinL + wave * (2 + hd);
        if (wave > 0) {
            if (lane == 0) { part[0] = a.m; part[1] = a.l; }
#pragma unroll
            for (int i = 0; i < MAX_DPL; ++i)
                if (lane + 64 * i < hd) part[2 + lane + 64 * i] = a.acc[i];
        }
        __syncthreads();
        if (wave > 0) return;
        for (int w = 1; w < WAVES; ++w) {
            const float* other = joinL + w * (2 + hd);
            AsPart b;
            b.m = other[0];
            b.l = other[1];
#pragma unroll
            for (int i = 0; i < MAX_DPL; ++i) b.acc[i] = lane + 64 * i < hd ? other[2 + lane + 64 * i] : 0.f;
            as_join(a, b);
        }
    }
#pragma unroll
    for (int i = 0; i < MAX_DPL; ++i) {
        const int d = lane + 64 * i;
        if (d < hd) o[d] = from_f32<T>(a.acc[i] / a.l);
    }
}

extern "C" int br_attn_simple(const void* q, size_t q_stride, void* out, int is_bf16, const int* pos,
                              const int* seq_of_token, const int* slots, const int* block_table,
                              int table_stride, const void* cache, int T, int nq, int nkv, int hd,
                              int page, int window, float scale, hipStream_t s) {
    if (T <= 0) return BR_OK;
    if (nq <= 0 || nkv <= 0 || nq % nkv || hd <= 0 || hd > 64 * MAX_DPL || page <= 0 || window < 0 ||
        nq > 65535)
        return BR_BAD_ARG;
    dim3 grid(T, nq);
    // a wave a class while that gives no more waves than the chip holds at four to a SIMD (16 a compute unit)
    const bool four = (long long)T * nq * 4 <= 16ll * br_device_cus();
    const size_t lds = (size_t)(((hd + 3) & ~3) + (four ? 4 * 64 + 4 * (2 + hd) : 64)) * sizeof(float);
    const bool vec = hd % (is_bf16 ? 8 : 4) == 0 && page % 64 == 0 && (uintptr_t)cache % 16 == 0;
#define AS_LAUNCH(TT, V, W, N) \
    attn_simple_kernel<TT, V, W, N><<<grid, 64 * W, lds, s>>>((const TT*)q, q_stride, (TT*)out, pos, seq_of_token, slots, block_table, \
                                                           table_stride, (const TT*)cache, nq, nkv, hd, page, window, scale)
#define AS_FORM(TT, V) do { \
        if (V && window > 0) { if (four) AS_LAUNCH(TT, V, 4, V); else AS_LAUNCH(TT, V, 1, V); } \
        else { if (four) AS_LAUNCH(TT, V, 4, false); else AS_LAUNCH(TT, V, 1, false); } \
    } while (0)
    if (is_bf16) { if (vec) AS_FORM(bf16, true); else AS_FORM(bf16, false); }
    else { if (vec) AS_FORM(float, true); else AS_FORM(float, false); }
#undef AS_FORM
#undef AS_LAUNCH
    return br_check_launch();
}
