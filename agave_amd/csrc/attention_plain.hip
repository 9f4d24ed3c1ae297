// Plain attention over the paged cache for gfx950, for any head size up to 512 and either
// element type: scores, probabilities and sums in 32-bit, exact expf, no skipping of small
// probabilities.  It is the true 32-bit path and the fallback for head sizes the bfloat16 kernels
// refuse.
//
// Reference: src/backend/kernels/cpu/sdpa.zig:34-88 (scores * scale, softmax, weighted sum
// of V), window bounds as src/ops/attention.zig:92-93 with the callers' convention of
// src/models/gpt_oss.zig:518-519: a query at position p sees keys max(0, p-W+1) .. p.
//
// Cache pages: K [page][kv head][64 rows][hd]; V transposed [page][kv head][hd][64 rows].
// Position j of sequence b lies in page table[b][j/64 - base[b]], row j % 64.
#include "common_impl.h"
#include "fours.h"
#include <math.h>

#define ROWS 16              // query rows a workgroup: tokens next to each other times the heads of a key head
#define COMPUTE_UNITS 256
#define MOST_SPLITS 16

// The largest / the sum over a row of 16 lanes, in each of them.
__device__ __forceinline__ float lanes16_max(float v) {
    v = fmaxf(v, dpp_get<0xB1, 0xF>(v, v));
    v = fmaxf(v, dpp_get<0x4E, 0xF>(v, v));
    v = fmaxf(v, dpp_get<0x141, 0xF>(v, v));
    return fmaxf(v, dpp_get<0x140, 0xF>(v, v));
}
__device__ __forceinline__ float lanes16_sum(float v) {
    v += dpp_get<0xB1, 0xF>(0.f, v);
    v += dpp_get<0x4E, 0xF>(0.f, v);
    v += dpp_get<0x141, 0xF>(0.f, v);
    return v + dpp_get<0x140, 0xF>(0.f, v);
}

// A workgroup of 4 waves takes 16 query rows (`run` neighbouring tokens of one key head's query heads) through the pages they
// see, a page of 64 keys at a time: every wave the scores of 16 keys, then, with the page's probabilities in LDS, the sums over
// the page for a quarter of the value elements.  Both are products for v_mfma_f32_16x16x4_f32, whose operands K and V come
// straight from memory in 16-byte pieces (it takes the summed index in any order as long as both operands agree).  Tokens of
// several sequences in one workgroup (any tok_seq is taken) go one sequence after another, or, with gridDim.z turns, the
// z-th of them in a workgroup of its own.
// gridDim.y workgroups share a row's pages and leave (sum, maximum, unnormalised result) for attn_plain_merge_kernel: with a
// token per sequence there are few rows and the pages one after another bound the time.
// NT: tiles of 64 value elements (16 a wave).  FULL: the head is as long as they are, and a page's keys are asked for at once.  VEC, VEC_V: q and keys, and values, are aligned to four elements.  A probability of
// 0 must not meet a value that is not finite (a key behind a token's position may hold anything): such pages are summed element
// by element.
// Bound by the 32-bit products (half of them for a token of 4 rows' padding) and, with few tokens, by the loads' way from memory.
// Measured, 16 heads on 4 key heads of 128 in 32 bits: prompts of 97, 259 and 421 tokens 63 us (a workgroup per token and head, a
// key a thread: 943 us), 2,000 tokens 0.45 ms (16.8 ms); a token each behind as many keys 15 us (59 us), behind 4,000 keys
// 33 us (562 us).  Errors against 64 bits are half as large (2.0 to 2.8e-7 after 4.2 to 5.5e-7).
// A token each is a chain: the position, the page's id, its keys, products, sums, values, the store; 10.2 us inside, of which the queries'
// way to LDS took 1.8, the id 1.0 and the keys behind it 4.0.  Now the first page travels while the queries are staged, all of its
// keys at once, and rows' tokens come from a table and not from divisions: a decode step of three sequences through eight layers
// 634 -> 610 us, prompts of 97 and 421 tokens 1.31 -> 1.26 and 2.94 -> 2.79 ms.
template <typename T, int NT, bool VEC, bool VEC_V, bool FULL>
__global__ __launch_bounds__(256) void attn_plain_kernel(
    const T* __restrict__ q, long ldq, T* __restrict__ out, long ldo, const T* __restrict__ k_pages,
    const T* __restrict__ v_pages, const int* __restrict__ table, int width, const int* __restrict__ base,
    int n_pages, const int* __restrict__ tok_seq, const int* __restrict__ tok_pos, int N, int nh, int nkv, int hd,
    float scale, int window, int run, float* __restrict__ part_o, float* __restrict__ part_ml) {
    constexpr int HDP = NT * 64;
    if constexpr (FULL) hd = HDP;
    constexpr bool V_AHEAD = NT <= 4;                        // a page's values are asked for before its scores are made
    __shared__ __attribute__((aligned(16))) float Qs[ROWS][HDP + 4];
    __shared__ __attribute__((aligned(16))) float P[ROWS][AGAVE_PAGE + 4];
    __shared__ __attribute__((aligned(16))) float wmax[4][ROWS], wsum[4][ROWS];
    __shared__ __attribute__((aligned(16))) int row_pos[ROWS], row_lo[ROWS], row_seq[ROWS], row_tok[ROWS];

    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const int G = nh / nkv, chunks = (G + ROWS - 1) / ROWS;
    const int chunk = blockIdx.x % chunks, kvh = blockIdx.x / chunks % nkv;
    int t0 = blockIdx.x / chunks / nkv * run, tokens = min(run, N - t0);
    if (gridDim.z > 1) {                                     // this workgroup's turn of the sequences among its tokens
        const int t = t0 + (lane < tokens ? lane : 0);
        unsigned long long left = __ballot(lane < tokens && (lane == 0 || tok_seq[t] != tok_seq[t > 0 ? t - 1 : 0]));
        for (int i = blockIdx.z; i > 0; --i) left &= left - 1;
        if (left == 0) return;
        const int a = __builtin_ctzll(left);
        left &= left - 1;
        tokens = (left == 0 || blockIdx.z + 1 == gridDim.z ? tokens : __builtin_ctzll(left)) - a;       // (the last turn takes all that are left)
        t0 += a;
    }
    const int heads = min(G - chunk * ROWS, ROWS), head0 = kvh * G + chunk * ROWS;
    const int rows = min(tokens * heads, ROWS);
    const int split = blockIdx.y, splits = gridDim.y;

    // One token (a decode step): its page ids need none of the other rows', and its first page travels while the queries are staged.
    const bool one = tokens == 1;
    const int one_seq = tok_seq[t0], one_pos = tok_pos[t0];
    f32x4_t x[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {                           // four elements a thread and turn
        const int row = (tid + 256 * i) / (HDP / 4), d = (tid + 256 * i) % (HDP / 4) * 4, real = min(row, rows - 1);
        const int tok = one ? 0 : real / heads;
        x[i] = ld4<VEC>(q + (size_t)(t0 + tok) * ldq + (size_t)(head0 + real - tok * heads) * hd, d, hd);
    }
    auto page_of = [&](int seq, int pbase, int page) -> long {
        const int col = page - pbase;
        const long pg = col >= 0 && col < width ? table[(size_t)seq * width + col] : -1;
        return pg >= n_pages ? -1 : pg;
    };
    constexpr int KD = FULL && V_AHEAD ? HDP / 16 : 1;       // a page's keys all at once, before its values
    f32x4_t kk[KD], vv[V_AHEAD ? NT : 1][4];
    auto values = [&](const T* vr, f32x4_t (&v)[4], int nt) {
        const T* row = vr + (size_t)min((4 * nt + w) * 16 + r, hd - 1) * AGAVE_PAGE;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = ld4<VEC_V>(row, 16 * j + 4 * g, AGAVE_PAGE);
    };
    auto ask = [&](long pg) {
        if constexpr (KD > 1) {
            const T* kr = k_pages + ((size_t)(pg * nkv + kvh) * AGAVE_PAGE + 16 * w + r) * hd;
#pragma unroll
            for (int i = 0; i < KD; ++i) kk[i] = ld4<VEC>(kr, 16 * i + 4 * g, hd);
        }
        if constexpr (V_AHEAD)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) values(v_pages + (size_t)(pg * nkv + kvh) * hd * AGAVE_PAGE, vv[nt], nt);
    };
    int asked = -1;                                          // the page that has been asked for
    if (one) {
        const int lo = window > 0 && one_pos - window + 1 > 0 ? one_pos - window + 1 : 0;
        const int first = lo / AGAVE_PAGE, count = one_pos / AGAVE_PAGE - first + 1, share = (count + splits - 1) / splits;
        const int page = first + split * share;
        const long pg = page < first + count ? page_of(one_seq, base[one_seq], page) : -1;
        if (pg >= 0) {
            ask(pg);
            asked = page;
        }
    }
    if (tid < ROWS) {
        const int tok = one ? 0 : tid / heads, at = t0 + tok;
        const bool real = tid < rows;
        const int p = !real ? -1 : (one ? one_pos : tok_pos[at]);
        row_pos[tid] = p;
        row_lo[tid] = real && window > 0 && p - window + 1 > 0 ? p - window + 1 : 0;
        row_seq[tid] = !real ? -1 : (one ? one_seq : tok_seq[at]);
        row_tok[tid] = tok;
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int row = (tid + 256 * i) / (HDP / 4), d = (tid + 256 * i) % (HDP / 4) * 4;
        *reinterpret_cast<f32x4_t*>(&Qs[row][d]) = row < rows ? x[i] : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();

    // rows 4 g + e; value element (4 nt + w) 16 + r
    float m[4], l[4];
    f32x4_t o[NT];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        m[e] = -INFINITY;
        l[e] = 0.f;
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) o[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int4 pos4 = *reinterpret_cast<const int4*>(&row_pos[4 * g]), lo4 = *reinterpret_cast<const int4*>(&row_lo[4 * g]);
    const int pos[4] = {pos4.x, pos4.y, pos4.z, pos4.w}, low[4] = {lo4.x, lo4.y, lo4.z, lo4.w};

    bool fresh = true;                                       // no page has been used yet
    for (int s0 = 0, s1; s0 < rows; s0 = s1) {               // a run of rows of one sequence
        const int seq = one ? one_seq : row_seq[s0];
        int lo = row_lo[s0], hi = row_pos[s0];
        for (s1 = one ? rows : s0 + 1; s1 < rows && row_seq[s1] == seq; ++s1) {
            lo = min(lo, row_lo[s1]);
            hi = max(hi, row_pos[s1]);
        }
        if (hi < 0) continue;
        const int first = lo / AGAVE_PAGE, count = hi / AGAVE_PAGE - first + 1, share = (count + splits - 1) / splits;
        const int from = first + split * share, to = min(from + share, first + count), pbase = base[seq];
        for (int page = from; page < to; ++page) {
            const long pg = page_of(seq, pbase, page);
            if (pg < 0) continue;
            const T* kr = k_pages + ((size_t)(pg * nkv + kvh) * AGAVE_PAGE + 16 * w + r) * hd;
            const T* vr = v_pages + (size_t)(pg * nkv + kvh) * hd * AGAVE_PAGE;
            const int key0 = page * AGAVE_PAGE;
            if (page != asked) ask(pg);
            asked = -1;
            // scores of keys 16 w + r
            f32x4_t sum[4] = {};
            auto scores = [&](f32x4_t kv, int d) {
                const f32x4_t qv = *reinterpret_cast<const f32x4_t*>(&Qs[r][d + 4 * g]);
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[e], kv[e], sum[e], 0, 0, 0);
            };
            if constexpr (KD > 1) {
#pragma unroll
                for (int i = 0; i < KD; ++i) scores(kk[i], 16 * i);
            } else {
#pragma unroll 8
                for (int d = 0; d < hd; d += 16) scores(ld4<VEC>(kr, d + 4 * g, hd), d);
            }
            f32x4_t s = (sum[0] + sum[1]) + (sum[2] + sum[3]);
            const int key = key0 + 16 * w + r;
            bool seen[4];
            f32x4_t most;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                seen[e] = 4 * g + e >= s0 && 4 * g + e < s1 && key >= low[e] && key <= pos[e];
                s[e] = seen[e] ? s[e] * scale : -INFINITY;
                most[e] = lanes16_max(s[e]);
            }
            if (r == 0) *reinterpret_cast<f32x4_t*>(&wmax[w][4 * g]) = most;
            __syncthreads();
            f32x4_t total;
            float alpha[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = 4 * g + e;
                const float m_new = fmaxf(m[e], fmaxf(fmaxf(wmax[0][row], wmax[1][row]), fmaxf(wmax[2][row], wmax[3][row])));
                // m_new is finite whenever any key of this or an earlier page was seen
                alpha[e] = 0.f;
                if (!fresh) alpha[e] = m[e] == -INFINITY ? 0.f : expf(m[e] - m_new);
                const float pr = seen[e] ? expf(s[e] - m_new) : 0.f;
                m[e] = m_new;
                P[row][16 * w + r] = pr;
                total[e] = lanes16_sum(pr);
            }
            if (r == 0) *reinterpret_cast<f32x4_t*>(&wsum[w][4 * g]) = total;
            __syncthreads();
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = 4 * g + e;
                l[e] = l[e] * alpha[e] + ((wsum[0][row] + wsum[1][row]) + (wsum[2][row] + wsum[3][row]));
            }
            fresh = false;
            const bool inside = key0 >= lo && key0 + AGAVE_PAGE - 1 <= hi;
            f32x4_t pf[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) pf[j] = *reinterpret_cast<const f32x4_t*>(&P[r][16 * j + 4 * g]);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if ((4 * nt + w) * 16 >= hd) continue;
                f32x4_t late[4];
                if constexpr (!V_AHEAD) values(vr, late, nt);
                f32x4_t (&v)[4] = V_AHEAD ? vv[V_AHEAD ? nt : 0] : late;
                f32x4_t add = {};
                if (!inside) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int at = key0 + 16 * j + 4 * g + e;
                            if (at < lo || at > hi) v[j][e] = 0.f;     // (no row sees it: it may hold anything)
                        }
                }
                float nothing = 0.f;                         // (0 times what is not finite is not a number)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) nothing = fmaf(v[j][e], 0.f, nothing);
                const bool finite = nothing == 0.f;
                if (__all(finite)) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) add = __builtin_amdgcn_mfma_f32_16x16x4f32(pf[j][e], v[j][e], add, 0, 0, 0);
                } else {
                    const T* row = vr + (size_t)min((4 * nt + w) * 16 + r, hd - 1) * AGAVE_PAGE;
                    for (int k = 0; k < AGAVE_PAGE; ++k) {
                        const float x = ld(row + k);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float pr = P[4 * g + e][k];
                            if (pr != 0.f) add[e] = fmaf(pr, x, add[e]);
                        }
                    }
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) o[nt][e] = o[nt][e] * alpha[e] + add[e];
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int row = 4 * g + e;
        if (row >= rows) continue;
        const int tok = row_tok[row];
        const size_t t = t0 + tok;
        const int h = head0 + row - tok * heads;
        const float inv = l[e] > 0.f ? 1.0f / l[e] : 0.f;
        const size_t part = (t * nh + h) * splits + split;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int d = (4 * nt + w) * 16 + r;
            if (d >= hd) continue;
            if (splits > 1) part_o[part * hd + d] = o[nt][e];
            else st(out + t * ldo + (size_t)h * hd + d, o[nt][e] * inv);
        }
        if (splits > 1 && w == 0 && r == 0) {
            part_ml[2 * part] = m[e];
            part_ml[2 * part + 1] = l[e];
        }
    }
}

// The results that a row's workgroups left: a workgroup per (token, head).  A share without a key holds zeros and counts as
// such.  One whose scores are all not a number has no maximum either, but a sum and results that are not numbers: it goes into
// the row's as any other, so that a row comes out as it does from one workgroup.
// Bound by its ways to memory: the shares' maxima, sums and a thread's column of their results are asked for at once (one after the
// other, three sequences' tokens of 32-bit rows through eight layers 693 us a step, so 675).
template <typename T>
__global__ __launch_bounds__(128) void attn_plain_merge_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                               T* __restrict__ out, long ldo, int nh, int hd, int splits) {
    const size_t row = blockIdx.x;
    const float* ml = part_ml + 2 * row * splits;
    float ms[MOST_SPLITS], ls[MOST_SPLITS], x[MOST_SPLITS];
#pragma unroll
    for (int s = 0; s < MOST_SPLITS; ++s) {                  // (past the last share: the last one again, not counted)
        ms[s] = ml[2 * min(s, splits - 1)];
        ls[s] = ml[2 * min(s, splits - 1) + 1];
    }
    auto ask = [&](int d) {
#pragma unroll
        for (int s = 0; s < MOST_SPLITS; ++s) x[s] = part_o[(row * splits + min(s, splits - 1)) * hd + min(d, hd - 1)];
    };
    ask(threadIdx.x);
    __builtin_amdgcn_sched_barrier(0);
    float m = -INFINITY, l = 0.f, f[MOST_SPLITS];
#pragma unroll
    for (int s = 0; s < MOST_SPLITS; ++s) m = fmaxf(m, ms[s]);
#pragma unroll
    for (int s = 0; s < MOST_SPLITS; ++s) {
        f[s] = s < splits && ms[s] != -INFINITY ? expf(ms[s] - m) : 0.f;
        if (s < splits) l = fmaf(ls[s], f[s], l);
    }
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    for (int d = threadIdx.x; d < hd; d += 128) {
        if (d != (int)threadIdx.x) ask(d);
        float sum = 0.f;
#pragma unroll
        for (int s = 0; s < MOST_SPLITS; ++s)
            if (s < splits) sum = fmaf(x[s], f[s], sum);
        st(out + (row / nh) * ldo + (row % nh) * hd + d, sum * inv);
    }
}

// Few keys: a workgroup per token and head, four lanes a key, then a thread per value element (two from 257 elements on).  Bound by
// its chain of trips to memory; the kernel above brings whole pages and multiplies tiles that are mostly empty.  A key's product
// has sixteen running sums.  Takes any number of keys, a page at a time.
// Measured in 32 bits, us, tiles of rows and so: a prompt of 5 tokens, 8 heads of 256 over 4, 13.7 and 5.7 (an element at a time a key
// and a thread, the kernel before both, 9.9), of 512 over one 21.9 and 7.7 (16.2); of 33 tokens 13.7 and 7.8, 22.1 and 11.5; eight
// tokens behind 64 keys 13.8 and 7.8, 22.0 and 11.3.  Errors against 64 bits 0.6 to 1.3e-7 after 0.8 to 1.9e-7.
template <typename T, bool VEC, bool VEC_V>
__global__ __launch_bounds__(256) void attn_plain_few_keys_kernel(
    const T* __restrict__ q, long ldq, T* __restrict__ out, long ldo, const T* __restrict__ k_pages,
    const T* __restrict__ v_pages, const int* __restrict__ table, int width, const int* __restrict__ base,
    int n_pages, const int* __restrict__ tok_seq, const int* __restrict__ tok_pos, int nh, int nkv, int hd, float scale, int window) {
    __shared__ __attribute__((aligned(16))) float qs[512], P[AGAVE_PAGE];
    __shared__ float wmax[4], wsum[4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int t = blockIdx.x / nh, h = blockIdx.x % nh, kvh = h / (nh / nkv);
    const int seq = tok_seq[t], hi = tok_pos[t], lo = window > 0 && hi - window + 1 > 0 ? hi - window + 1 : 0;
    const int pbase = base[seq];
    for (int d = tid; d < (hd + 3) / 4 * 4; d += 256) qs[d] = d < hd ? ld(q + (size_t)t * ldq + (size_t)h * hd + d) : 0.f;
    __syncthreads();
    float m = -INFINITY, l = 0.f, o[2] = {0.f, 0.f};
    for (int page = lo / AGAVE_PAGE; page * AGAVE_PAGE <= hi; ++page) {
        const int col = page - pbase;
        const long pg = col >= 0 && col < width ? table[(size_t)seq * width + col] : -1;
        if (pg < 0 || pg >= n_pages) continue;               // (the same for the whole workgroup)
        const T* v[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) v[a] = v_pages + ((size_t)(pg * nkv + kvh) * hd + min(tid + 256 * a, hd - 1)) * AGAVE_PAGE;
        const int j0 = max(lo - page * AGAVE_PAGE, 0), j1 = min(hi - page * AGAVE_PAGE, AGAVE_PAGE - 1);      // the keys that are seen
        f32x4_t vv[2][4];
        auto values = [&](int j) {                           // of the sixteen keys from j on
#pragma unroll
            for (int a = 0; a < 2; ++a)
                if (256 * a < hd)
#pragma unroll
                    for (int i = 0; i < 4; ++i) vv[a][i] = ld4<VEC_V>(v[a], j + 4 * i, AGAVE_PAGE);
        };
        values(j0 & ~15);
        const int key = tid >> 2;
        const bool seen = key >= j0 && key <= j1;
        f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
        if (seen) {
            const T* kr = k_pages + ((size_t)(pg * nkv + kvh) * AGAVE_PAGE + key) * hd;
#pragma unroll 8
            for (int d = 4 * (tid & 3); d < hd; d += 16) {
                const f32x4_t kv = ld4<VEC>(kr, d, hd), qv = *reinterpret_cast<const f32x4_t*>(&qs[d]);
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] = fmaf(kv[e], qv[e], sum[e]);
            }
        }
        float s = (sum[0] + sum[1]) + (sum[2] + sum[3]);
        s += dpp_get<0xB1, 0xF>(0.f, s);
        s += dpp_get<0x4E, 0xF>(0.f, s);
        s = seen ? s * scale : -INFINITY;
        const float most = wave_max(s);
        if (lane == 0) wmax[w] = most;
        __syncthreads();
        const float m_new = fmaxf(m, fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3])));
        const float alpha = m == -INFINITY ? 0.f : expf(m - m_new), pr = seen ? expf(s - m_new) : 0.f;
        m = m_new;
        if ((tid & 3) == 0) P[key] = pr;
        const float total = wave_sum((tid & 3) == 0 ? pr : 0.f);
        if (lane == 0) wsum[w] = total;
        __syncthreads();
        l = l * alpha + ((wsum[0] + wsum[1]) + (wsum[2] + wsum[3]));
        o[0] *= alpha;
        o[1] *= alpha;
        float add[2] = {0.f, 0.f};
        for (int j = j0 & ~15; j <= j1; j += 16) {
            if (j != (j0 & ~15)) values(j);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4_t pv = *reinterpret_cast<const f32x4_t*>(&P[j + 4 * i]);
#pragma unroll
                for (int a = 0; a < 2; ++a)
                    if (256 * a < hd)
#pragma unroll
                        for (int e = 0; e < 4; ++e) add[a] = pv[e] != 0.f ? fmaf(pv[e], vv[a][i][e], add[a]) : add[a];    // (a key that is not seen may hold anything)
            }
        }
        o[0] += add[0];
        o[1] += add[1];
        __syncthreads();                                     // P, wmax and wsum are written again
    }
    const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
    for (int a = 0; a < 2; ++a)
        if (tid + 256 * a < hd) st(out + (size_t)t * ldo + (size_t)h * hd + tid + 256 * a, o[a] * inv);
}

template <typename T, int NT>
static void launch_rows(const T* q, long ldq, T* out, long ldo, const T* k_pages, const T* v_pages, const int* table, int width,
                        const int* base, int n_pages, const int* tok_seq, const int* tok_pos, int N, int nh, int nkv, int hd, float scale,
                        int window, bool few_keys, bool one_token_each, int run, int turns, int splits, float* part_o, float* part_ml, hipStream_t stream) {
    const int chunks = (nh / nkv + ROWS - 1) / ROWS;
    const dim3 grid((N + run - 1) / run * nkv * chunks, splits, turns);
    // four elements at a time where rows are aligned to as many (a value row is a page long, so its pages' start decides)
    const uintptr_t wide = 4 * sizeof(T);
    const bool vec_v = (uintptr_t)v_pages % wide == 0;
    const bool vec = vec_v && hd % 4 == 0 && ldq % 4 == 0 && (uintptr_t)k_pages % wide == 0 && (uintptr_t)q % wide == 0;
    if (few_keys) {
#define FEW_GO(VEC_, VEC_V_) attn_plain_few_keys_kernel<T, VEC_, VEC_V_><<<N * nh, 256, 0, stream>>>(q, ldq, out, ldo, k_pages, v_pages, table, \
        width, base, n_pages, tok_seq, tok_pos, nh, nkv, hd, scale, window)
        if (vec) FEW_GO(true, true); else if (vec_v) FEW_GO(false, true); else FEW_GO(false, false);
#undef FEW_GO
        return;
    }
#define PLAIN_GO(VEC_, VEC_V_, FULL_) attn_plain_kernel<T, NT, VEC_, VEC_V_, FULL_><<<grid, 256, 0, stream>>>(q, ldq, out, ldo, k_pages, v_pages, \
        table, width, base, n_pages, tok_seq, tok_pos, N, nh, nkv, hd, scale, window, run, part_o, part_ml)
    // A page's keys at once beside its values cost registers: heads of 256 fit one workgroup a compute unit instead of two, of 128 in bfloat16
    // two instead of three.  Faster at every size for shorter heads of floats; else where the others would have no work anyway,
    // or where one token's chain bounds the time.  us, keys one after another and at once, 32-bit, heads of 256: 8 over 4, 421 tokens
    // (212 workgroups) 67 and 51, 700 (352) 101 and 99, 800 (400) 118 and 124, 2,000 335 and 386; 16 over 8, 6,000 2,029 and 2,458;
    // 64 tokens apart behind 1,000 keys (512) 257 and 239.  bfloat16: 8 over 4, 500 tokens (252) 70 and 65, 521 (264) 81 and 84, 2,000 334
    // and 444; 64 apart behind 200 keys (256) 47 and 38, 128 (512) 63 and 73; heads of 128, 16 over 4, 500 tokens (500) 49 and 45, 521
    // (524) 56 and 60, 32 over 16, 33 apart behind 1,000 keys (528) 148 and 169, 64 (1,024) 292 and 187.
    const long wgs = (long)grid.x * splits;
    const bool floats = sizeof(T) == 4;
    bool full = NT <= 4 && hd == NT * 64;
    if (NT == 4) full = full && ((floats && one_token_each) || wgs <= (floats ? 360 : COMPUTE_UNITS));
    if (NT == 2 && !floats) full = full && (wgs <= 2 * COMPUTE_UNITS || (one_token_each && wgs > 3 * COMPUTE_UNITS));
    if (vec && full) PLAIN_GO(true, true, (NT <= 4));
    else if (vec) PLAIN_GO(true, true, false);
    else if (vec_v) PLAIN_GO(false, true, false);
    else PLAIN_GO(false, false, false);
#undef PLAIN_GO
    if (splits > 1) attn_plain_merge_kernel<T><<<N * nh, 128, 0, stream>>>(part_o, part_ml, out, ldo, nh, hd, splits);
}

template <typename T>
static void launch_type(const void* q, long ldq, void* out, long ldo, const void* k_pages, const void* v_pages, const int* table, int width,
                        const int* base, int n_pages, const int* tok_seq, const int* tok_pos, int N, int nh, int nkv, int hd, float scale,
                        int window, bool few_keys, bool one_token_each, int run, int turns, int splits, float* part_o, float* part_ml, hipStream_t stream) {
#define ROWS_GO(NT_) launch_rows<T, NT_>((const T*)q, ldq, (T*)out, ldo, (const T*)k_pages, (const T*)v_pages, table, width, base, n_pages, \
                                         tok_seq, tok_pos, N, nh, nkv, hd, scale, window, few_keys, one_token_each, run, turns, splits, part_o, part_ml, stream)
    if (hd <= 64) ROWS_GO(1);
    else if (hd <= 128) ROWS_GO(2);
    else if (hd <= 256) ROWS_GO(4);
    else ROWS_GO(8);
#undef ROWS_GO
}

// How many workgroups share a row's pages when every sequence brings one token and spans at most `span` pages: a page each at
// least, and no more workgroups in all than fill the compute units once.
extern "C" int agave_attn_plain_splits(int N, int nh, int nkv, int span) {
    if (N <= 0 || nh <= 0 || nkv <= 0 || nh % nkv != 0) return 1;
    const long wgs = (long)N * nkv * ((nh / nkv + ROWS - 1) / ROWS);
    long z = COMPUTE_UNITS / wgs;
    if (z > span) z = span;
    if (z > MOST_SPLITS) z = MOST_SPLITS;
    return z < 1 ? 1 : (int)z;
}

// How many neighbouring tokens a workgroup takes.
// Neighbouring tokens share a page's keys where there are enough of them to fill the compute units without.  us, a token a
// workgroup and several, 32-bit: 16 heads of 128 over 4, 64 tokens (256 workgroups) 10.5 and 11.2, 96 tokens 18.1 and 16.2, 421
// tokens 99 and 47; 8 heads of 256 over 4, 64 tokens 14.1 and 15.8, 96 tokens 27.3 and 24.5; 4 heads of 64 over one, 256
// tokens 17.6 and 18.1, 300 tokens 22.4 and 20.9; 8 heads of 64 over 8, 64 tokens (512 workgroups) 8.4 and 8.8, 96 tokens 13.2 and 11.9.
extern "C" int agave_attn_plain_run(int N, int nh, int nkv) {
    if (N <= 0 || nh <= 0 || nkv <= 0 || nh % nkv != 0) return 1;
    const int G = nh / nkv;
    return G >= ROWS || (long)N * nkv <= COMPUTE_UNITS ? 1 : ROWS / G;
}

// one_token_each: neighbouring tokens are of different sequences (a decode step), so a workgroup takes one.  most_seqs: of as
// many sequences at most are any `agave_attn_plain_run` tokens from a multiple of it on.  most_keys: no token sees more keys than
// this, 0 where that is not known.  (No result depends on either being right.)  splits > 1: part_o [N][nh][splits][hd] and part_ml
// [N][nh][splits][2] receive what a row's workgroups leave.
extern "C" int agave_attn_plain(int dtype, const void* q, long ldq, void* out, long ldo, const void* k_pages,
                                const void* v_pages, const int* table, int width, const int* base, int n_pages,
                                const int* tok_seq, const int* tok_pos, int N, int nh, int nkv, int hd, float scale,
                                int window, int one_token_each, int most_seqs, int most_keys, int splits, float* part_o, float* part_ml, hipStream_t stream) {
    AGAVE_CHECK(N >= 0 && nh > 0 && nkv > 0 && hd > 0, "attn_plain: bad sizes N=%d nh=%d nkv=%d hd=%d", N, nh, nkv, hd);
    AGAVE_CHECK(nh % nkv == 0, "attn_plain: %d query heads are not a multiple of %d kv heads", nh, nkv);
    AGAVE_CHECK(hd <= 512, "attn_plain: head_dim %d exceeds the supported maximum %d", hd, 512);
    AGAVE_CHECK(ldq >= (long)nh * hd && ldo >= (long)nh * hd, "attn_plain: a row stride is below nh*hd");
    AGAVE_CHECK(window >= 0, "attn_plain: negative window");
    AGAVE_CHECK(q && out && k_pages && v_pages && table && base && tok_seq && tok_pos && width > 0 && n_pages > 0,
                "attn_plain: null buffer or empty table");
    AGAVE_CHECK((long)N * nh < 2147483647L, "attn_plain: too many (token, head) pairs");
    AGAVE_CHECK(splits >= 1 && splits <= MOST_SPLITS && (splits == 1 || (part_o && part_ml)), "attn_plain: %d splits (1 to %d, with buffers for what they leave)",
                splits, MOST_SPLITS);
    AGAVE_CHECK(dtype == AGAVE_F32 || dtype == AGAVE_BF16, "attn_plain: unknown dtype %d", dtype);
    AGAVE_CHECK(most_seqs >= 1, "attn_plain: %d sequences a workgroup", most_seqs);
    if (N == 0) return 0;
    // Few keys and few rows: beyond, tiles of rows share what they load (the longest times of the few-key kernel over those of the
    // tiles, over 16 head shapes and types: 16 keys and 1,024 rows 1.01, 2,048 rows 2.9; 48 and 512 1.01, 1,024 1.4; 64 and 256 1.03, 512 1.13).
    const bool few_keys = splits == 1 && most_keys > 0 && most_keys <= 64 && (long)N * nh <= (most_keys <= 16 ? 1024 : most_keys <= 48 ? 512 : 256);
    const int run = one_token_each ? 1 : agave_attn_plain_run(N, nh, nkv);
    // A workgroup for each of a run's sequences from three on (of two, one waits for the other).  40 tokens behind 1,000 keys
    // each and a prompt of 64 tokens, 32 bits, us, one after another and so: 8 heads of 64 over 8 885 and 75, 8 of 256 over 4 1,548
    // and 260 (a workgroup per token and head 148 and 400).
    const int most_turns = most_seqs < run ? most_seqs : run, turns = most_turns > 2 ? most_turns : 1;
    if (dtype == AGAVE_F32)
        launch_type<float>(q, ldq, out, ldo, k_pages, v_pages, table, width, base, n_pages, tok_seq, tok_pos, N, nh, nkv, hd, scale, window,
                           few_keys, one_token_each != 0, run, turns, splits, part_o, part_ml, stream);
    else
        launch_type<bf16>(q, ldq, out, ldo, k_pages, v_pages, table, width, base, n_pages, tok_seq, tok_pos, N, nh, nkv, hd, scale, window,
                          few_keys, one_token_each != 0, run, turns, splits, part_o, part_ml, stream);
    AGAVE_LAUNCH_CHECK("attn_plain");
    return 0;
}
