// Decode steps of the attention whose query heads all read one wide key row per position ([c | r], up to 576 elements)
// and whose values are the row's first elements (c, up to 512), for gfx950 (bfloat16, pages in operand order, see
// row_pages.h).  One row a sequence.
//
//   latent_decode    scores, softmax and the sums over the cached rows.  A workgroup of eight waves takes a page at a
//                    time, all waves together: with sixteen query heads as columns, wave w multiplies key block w % 4 over
//                    half of the row's elements, the halves meet in LDS, every wave makes the page's softmax for itself
//                    (the scores a lane reads are the ones its operand of the next product holds), and then adds its
//                    own share of the value columns.  So a page is one round trip to memory however wide its rows are: a
//                    wave's share of the keys and of the values is asked for at once, and the next page's while this one
//                    is multiplied.  `splits` workgroups share a sequence's pages; each leaves its reference, its sum
//                    and its unnormalised sums over the rows.
//                    Bound by that round trip and the chain behind it: 16 heads of 576, 4 sequences of 1,000 in 32 shares
//                    10.9 -> 9.6 to 10.5 us, the step 0.493 -> 0.485 ms, since a share of one page reads nothing behind it
//                    (without that branch 12.3 us for both kernels instead of 11.7).
//   latent_values    merges the shares of a (row, head) and multiplies the merged row by the head's value matrix:
//                    y = W_h x, times the sigmoid of a gate where there is one.  The matrix is asked for before the shares.
//
// A window limits the keys to positions p-W+1 .. p; a sink per head is one more term of the softmax's denominator.
#include "common_impl.h"
#include "mfma.h"
#include "row_pages.h"
#include <math.h>

struct LatentDecodeArgs {
    const bf16* q; long ldq;                 // [rows][heads * kd]
    const bf16* k_pages; const bf16* v_pages; const int* table; int width; const int* base; int n_pages;
    const int* tok_pos;                      // row b is sequence b's
    int heads, kd, vd;
    float scale;
    int window;                              // 0: all earlier keys
    const float* sink;                       // [heads] or null
    int splits;
    float* part_o;                           // [rows][heads][splits][vd]
    float* part_ml;                          // [rows][heads][splits][2]: reference (base 2), sum
};

// A barrier that leaves loads from memory in flight: only the wave's LDS accesses are waited for.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// KH: steps of 32 elements a wave multiplies (half of the row's); VW: blocks of 16 value columns a wave adds
template <int KH, int VW>
__global__ __launch_bounds__(512) void latent_decode_kernel(LatentDecodeArgs A) {
    __shared__ f32x4_t sums[2][2][4][64];                    // [turn][half of the row][key block][lane]
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4, kb = w & 3, half = w >> 2;
    const int b = blockIdx.x / A.splits, sp = blockIdx.x % A.splits;
    // what names the pages is asked for at once: the position, the table's first column's page, a table column a lane
    const int pos = A.tok_pos[b], pbase = A.base[b];
    const int* row_table = A.table + (size_t)b * A.width;
    const int column = row_table[lane < A.width ? lane : A.width - 1];
    const int head = blockIdx.y * 16 + c;
    const bool valid = head < A.heads;
    const int ksl = (A.kd + 31) / 32, k0 = half ? (ksl + 1) / 2 : 0, k_end = half ? ksl : (ksl + 1) / 2;
    const int n_vb = A.vd / 16;
    frag16 q[KH];
    const bf16* qrow = A.q + (size_t)b * A.ldq + (size_t)(valid ? head : 0) * A.kd;
#pragma unroll
    for (int i = 0; i < KH; ++i) {
        const int e = 32 * (k0 + i) + 8 * g;
        q[i].u = *reinterpret_cast<const uint4*>(qrow + (k0 + i < k_end && e < A.kd ? e : 0));     // (emptied outside the row below)
    }
    const float LOG2E = 1.4426950408889634f, scale2 = A.scale * LOG2E;
    float m = -INFINITY, l = 0.f;
    if (A.sink && sp == 0) {
        m = A.sink[valid ? head : 0] * LOG2E;
        l = g == 0 ? 1.f : 0.f;                              // (the lane groups' sums are added up at the end)
    }
    f32x4_t o[VW];
#pragma unroll
    for (int j = 0; j < VW; ++j) o[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const int W = A.window, lo = W > 0 ? max(0, pos - W + 1) : 0;
    const int first = lo / AGAVE_PAGE, n_pg = pos / AGAVE_PAGE - first + 1;
    // The page of the idx-th place in two steps: its id is asked for a page ahead of its use, by a load at one place for the whole wave
    // (scalar: a load by the lanes is waited for with all the page's loads before it, and a sequence of more than 64 pages then asks
    // for its second page when the first is there).  16 heads of 576, with lanes' loads and now, us: one sequence of 6,000 15.2 and 14.7,
    // of 30,000 31.3 and 28.5, 4 of 1,000 11.8 and 11.7.
    const auto scalar_table = (const __attribute__((address_space(4))) int*)row_table;
    auto ask_id = [&](int idx) -> int {
        const int col = first + idx - pbase;
        return scalar_table[col < 0 ? 0 : (col < A.width ? col : A.width - 1)];
    };
    auto page_at = [&](int idx, int id) -> int {
        const int col = first + idx - pbase;
        return idx >= n_pg || col < 0 || col >= A.width || id >= A.n_pages ? -1 : id;
    };
    // Loads without conditions: where a page is not there, all lanes read one place of page 0, and nothing uses it.  (A whole page 0 was
    // read behind every sequence's last, and the first page's loads waited for the queries'.)
    auto fetch = [&](int pg, frag16 (&k)[KH], frag16 (&v)[VW][2]) {
        const size_t at = pg < 0 ? 0 : pg;
        const int place = pg < 0 ? 0 : lane;
        const u32x4_t* kt = (const u32x4_t*)A.k_pages + (at * 4 + kb) * ksl * 64 + place;
        const u32x4_t* vt = (const u32x4_t*)A.v_pages + at * n_vb * 2 * 64 + place;
#pragma unroll
        for (int i = 0; i < KH; ++i) k[i].r = kt[(size_t)min(k0 + i, ksl - 1) * 64];      // (past my half q is empty)
#pragma unroll
        for (int j = 0; j < VW; ++j) {
            const int nb = w + 8 * j < n_vb ? w + 8 * j : 0;
#pragma unroll
            for (int h = 0; h < 2; ++h) v[j][h].r = vt[(size_t)(nb * 2 + h) * 64];
        }
    };
    int turn = 0;                                            // (the scores' place: the one before last's readers are done when it comes round)
    auto use = [&](int idx, frag16 (&k)[KH], frag16 (&v)[VW][2]) {
        f32x4_t s0 = f32x4_t{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
        for (int i = 0; i < KH; i += 2) {
            s0 = mfma_16x16x32(k[i], q[i], s0);
            if (i + 1 < KH) s1 = mfma_16x16x32(k[i + 1 < KH ? i + 1 : i], q[i + 1 < KH ? i + 1 : i], s1);
        }
        sums[turn][half][kb][lane] = s0 + s1;
        lds_barrier();
        // the page's scores of my column: key block kb2 holds keys 32 (kb2 / 2) + 8 g + 4 (kb2 % 2) + e
        float s[4][4], top = -INFINITY;
        const int d0 = pos - (first + idx) * AGAVE_PAGE - 8 * g;          // distance to the lane group's first key
#pragma unroll
        for (int kb2 = 0; kb2 < 4; ++kb2) {
            const f32x4_t x = sums[turn][0][kb2][lane], y = sums[turn][1][kb2][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int dist = d0 - (32 * (kb2 >> 1) + 4 * (kb2 & 1) + e);
                const bool see = dist >= 0 && (W == 0 || dist < W);
                s[kb2][e] = see ? (x[e] + y[e]) * scale2 : -INFINITY;
                top = fmaxf(top, s[kb2][e]);
            }
        }
        top = rows_max(top);
        const float m_new = fmaxf(m, top), ref = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - ref);
        float sum = 0.f;
        frag16 p[2];
#pragma unroll
        for (int kb2 = 0; kb2 < 4; ++kb2) {
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[e] = __builtin_amdgcn_exp2f(s[kb2][e] - ref);           // 2^(-inf) = 0 for what is not seen
                sum += x[e];
            }
            p[kb2 >> 1].r[2 * (kb2 & 1)] = f32x2_to_bf16x2(x[0], x[1]);
            p[kb2 >> 1].r[2 * (kb2 & 1) + 1] = f32x2_to_bf16x2(x[2], x[3]);
        }
        l = l * alpha + sum;
        m = m_new;
        turn ^= 1;
#pragma unroll
        for (int j = 0; j < VW; ++j) {
            o[j] *= alpha;
            o[j] = mfma_16x16x32(v[j][0], p[0], o[j]);
            o[j] = mfma_16x16x32(v[j][1], p[1], o[j]);
        }
    };
    // two sets of operands take turns; which pages there are is the same for all waves, so all of them meet at every barrier
    frag16 ka[KH], va[VW][2], kc[KH], vc[VW][2];
    const int col0 = first + sp - pbase;
    int idx = sp, pg = page_at(idx, col0 >= 0 && col0 < 64 ? __builtin_amdgcn_readlane(column, col0) : ask_id(idx)), id = ask_id(idx + A.splits);
    fetch(pg, ka, va);
#pragma unroll
    for (int i = 0; i < KH; ++i)
        if (!(k0 + i < k_end && 32 * (k0 + i) + 8 * g < A.kd && valid)) q[i].u = make_uint4(0, 0, 0, 0);
    if (idx + A.splits >= n_pg) {                            // one page at most: nothing is asked for behind it
        if (pg >= 0) use(idx, ka, va);
        idx = n_pg;
    }
    while (idx < n_pg) {
        const int next = idx + A.splits, pg_next = page_at(next, id);
        id = ask_id(next + A.splits);
        fetch(pg_next, kc, vc);
        if (pg >= 0) use(idx, ka, va);
        if (next >= n_pg) break;
        idx = next + A.splits;
        pg = page_at(idx, id);
        id = ask_id(idx + A.splits);
        fetch(pg, ka, va);
        if (pg_next >= 0) use(next, kc, vc);
    }
    l = rows_sum(l);
    if (!valid) return;
    const size_t mine = ((size_t)b * A.heads + head) * A.splits + sp;
    if (w == 0 && g == 0) {
        A.part_ml[mine * 2] = m;
        A.part_ml[mine * 2 + 1] = l;
    }
#pragma unroll
    for (int j = 0; j < VW; ++j) {
        const int nb = w + 8 * j;
        if (nb < n_vb) *reinterpret_cast<f32x4_t*>(A.part_o + mine * A.vd + 16 * nb + 4 * g) = o[j];
    }
}

#define LATENT_MAX_KEY 576
#define LATENT_MAX_VALUE 512
#define LATENT_MAX_SPLITS 64

// 1 if these sizes run on the kernels of this file
extern "C" int agave_latent_decode_ok(int kd, int vd, int out, int ldq) {
    return kd > 0 && vd > 0 && vd <= kd && kd % 8 == 0 && kd <= LATENT_MAX_KEY && vd % 16 == 0 && vd <= LATENT_MAX_VALUE && out > 0 && ldq % 8 == 0;
}

template <int KH, int VW> static void launch_latent_decode(const LatentDecodeArgs& A, dim3 grid, hipStream_t stream) {
    latent_decode_kernel<KH, VW><<<grid, 512, 0, stream>>>(A);
}

extern "C" int agave_latent_decode(const void* q, long ldq, const void* k_pages, const void* v_pages, const int* table, int width,
                                   const int* base, int n_pages, const int* tok_pos, int rows, int heads, int kd, int vd, float scale,
                                   int window, const float* sink, int splits, float* part_o, float* part_ml, hipStream_t stream) {
    AGAVE_CHECK(rows >= 0 && heads > 0 && width > 0 && n_pages > 0 && window >= 0, "latent_decode: bad sizes rows=%d heads=%d", rows, heads);
    AGAVE_CHECK(agave_latent_decode_ok(kd, vd, 1, (int)(ldq % 8)), "latent_decode: rows of %d / %d elements are not taken", kd, vd);
    AGAVE_CHECK(splits >= 1 && splits <= LATENT_MAX_SPLITS, "latent_decode: %d shares of a row (1 to %d)", splits, LATENT_MAX_SPLITS);
    AGAVE_CHECK(q && k_pages && v_pages && table && base && tok_pos && part_o && part_ml, "latent_decode: null buffer");
    AGAVE_CHECK(ldq >= (long)heads * kd && ((uintptr_t)q % 16) == 0 && ((uintptr_t)part_o % 16) == 0, "latent_decode: query rows too short, or not aligned to 16 bytes");
    AGAVE_CHECK((long)rows * splits < 2147483647L && (heads + 15) / 16 <= 65535, "latent_decode: too many rows or heads");
    if (rows == 0) return 0;
    LatentDecodeArgs A{(const bf16*)q, ldq, (const bf16*)k_pages, (const bf16*)v_pages, table, width, base, n_pages, tok_pos, heads, kd, vd,
                       scale, window, sink, splits, part_o, part_ml};
    const dim3 grid(rows * splits, (heads + 15) / 16);
    const int kh = ((kd + 31) / 32 + 1) / 2, vw = (vd / 16 + 7) / 8;
    if (kh <= 2 && vw <= 1) launch_latent_decode<2, 1>(A, grid, stream);
    else if (kh <= 5 && vw <= 2) launch_latent_decode<5, 2>(A, grid, stream);
    else launch_latent_decode<9, 4>(A, grid, stream);
    AGAVE_LAUNCH_CHECK("latent_decode");
    return 0;
}

// ------------------------------------------------------------------ the shares merged, and the head's value matrix
struct LatentValuesArgs {
    const float* part_o; const float* part_ml; int splits;
    const bf16* w;                           // [heads][out][vd]
    bf16* y; long ldy;                       // [rows][heads * out]
    const float* gate; long ldg;             // [rows][heads * out] logits, or null
    int heads, vd, out;
};

// One workgroup or a few per (row, head), eight waves.  The merge: four groups of 128 threads take the shares in turn, a thread four
// neighbouring elements.  The product: a wave per block of 16 outputs, the merged row as all sixteen columns of the
// operand.  VK: steps of 32 elements along the row.  SR: shares of a group at most.
// Bound by the ways to memory, one after the other: everything that is read (the shares' sums, then their rows, the first block's
// matrix and gate) is asked for before anything is waited for, and in the order in which it is needed, and every wave has all shares'
// weights in its lanes.  us, with the shares' sums waited for first and a workgroup a (row, head), and so, 16 heads of 512 by 128: 1 row
// of 64 shares 7.1 and 4.3, 4 rows 7.2 and 4.8, 6 rows of 42 7.9 and 6.3, 16 rows of 16 7.6 and 7.3, 64 rows of 4 25.0 and 23.6; 128 heads,
// 8 rows of 4 23.0 and 22.8.
template <int VK, int SR>
__global__ __launch_bounds__(512) void latent_values_kernel(LatentValuesArgs A) {
    __shared__ f32x4_t part[4][LATENT_MAX_VALUE / 4];
    __shared__ __attribute__((aligned(16))) bf16 row[LATENT_MAX_VALUE + 32];
    const int r = blockIdx.x / A.heads, h = blockIdx.x % A.heads, tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
    const int vd = A.vd, out = A.out, splits = A.splits;
    // this workgroup's blocks of outputs
    const int all = (out + 15) / 16, per = (all + gridDim.y - 1) / gridDim.y, ob0 = blockIdx.y * per, n_ob = min(ob0 + per, all);
    const bf16* w = A.w + (size_t)h * out * vd;
    const size_t first = (size_t)blockIdx.x * splits;
    const float* ml = A.part_ml + (first + (lane < splits ? lane : 0)) * 2;
    const float share_m = ml[0], share_l = ml[1];
    const int grp = wv >> 1, d = (tid & 127) * 4;
    f32x4_t x[SR] = {};
    // (fewer shares than groups: a group without one would read another's again.  33 rows of 128 heads in one share, latent_decode with it,
    // 106.6 us so, 104.1; 64 rows of 128 181 and 177)
    if (grp < splits) {
        const float* src = A.part_o + first * vd + (d < vd ? d : 0);
#pragma unroll
        for (int j = 0; j < SR; ++j) {
            const int s = grp + 4 * j;                       // (past the last share: the last one again, of weight 0)
            x[j] = *reinterpret_cast<const f32x4_t*>(src + (size_t)(s < splits ? s : splits - 1) * vd);
        }
    }
    // the first block's share of the matrix travels while the shares are merged
    frag16 f[VK];
    auto ask = [&](int ob) {
        const int o = 16 * ob + c;
        const bf16* wr = w + (size_t)(o < out ? o : out - 1) * vd;
#pragma unroll
        for (int k = 0; k < VK; ++k) {
            const int e = 32 * k + 8 * g;
            f[k].u = *reinterpret_cast<const uint4*>(wr + (e < vd ? e : 0));       // (the row is empty there)
        }
    };
    float gate[4];
    auto ask_gate = [&](int ob) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = 16 * ob + 4 * g + e;
            gate[e] = A.gate ? A.gate[(size_t)r * A.ldg + (size_t)h * out + (n < out ? n : out - 1)] : 0.f;
        }
    };
    if (ob0 + wv < n_ob) {
        ask(ob0 + wv);
        ask_gate(ob0 + wv);
    }
    __builtin_amdgcn_sched_barrier(0);
    float weight;                                            // of share `lane`
    {
        const float m = lane < splits ? share_m : -INFINITY, top = wave_max(m);
        const float e = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - top);
        const float total = wave_sum(e * share_l);
        weight = total > 0.f ? e / total : 0.f;
    }
    {
        f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < SR; ++j) {
            const int s = grp + 4 * j;
            const float ws = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(weight), s));      // (SR <= 16: s < 64)
            acc += x[j] * (s < splits ? ws : 0.f);
        }
        part[grp][tid & 127] = acc;
    }
    __syncthreads();
    if (tid < 128) {
        uint2 p = make_uint2(0, 0);
        if (d < vd) {
            const f32x4_t sum = part[0][tid] + part[1][tid] + part[2][tid] + part[3][tid];
            p = make_uint2(f32x2_to_bf16x2(sum[0], sum[1]), f32x2_to_bf16x2(sum[2], sum[3]));
        }
        *reinterpret_cast<uint2*>(row + d) = p;              // (elements past the row's end are zeros)
    }
    __syncthreads();
    for (int ob = ob0 + wv; ob < n_ob; ob += 8) {
        if (ob != ob0 + wv) {
            ask(ob);
            ask_gate(ob);
        }
        f32x4_t y = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < VK; ++k) {
            frag16 in;
            in.u = *reinterpret_cast<const uint4*>(row + 32 * k + 8 * g);
            y = mfma_16x16x32(f[k], in, y);
        }
        if (c == 0) {                                        // all columns are the same row: outputs 16 ob + 4 g + e
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = 16 * ob + 4 * g + e;
                if (n >= out) continue;
                float v = y[e];
                if (A.gate) v *= 1.0f / (1.0f + expf(-gate[e]));
                A.y[(size_t)r * A.ldy + (size_t)h * out + n] = f32_to_bf16(v);
            }
        }
    }
}

template <int VK>
static void launch_latent_values(const LatentValuesArgs& A, unsigned wgs, hipStream_t stream) {
    // As many workgroups a (row, head) as leave one a compute unit: what a compute unit takes from memory bounds them, and each merges the
    // shares for itself.  us, 1, 2, 4 and 8 of them (16 heads of 512 by 128): 1 row of 64 shares 7.0 5.5 4.6 4.2, 4 rows 7.2 5.7 4.9
    // 7.4, 6 rows of 42 shares 7.6 6.3 8.4 10.3, 16 rows of 16 shares 7.3 9.8 13.6 21.2.
    const int blocks = (A.out + 15) / 16;
    unsigned parts = 1;
    while (2 * parts * wgs <= 256 && 2 * parts <= (unsigned)blocks) parts *= 2;
    const dim3 grid(wgs, parts);
    if (A.splits <= 4) latent_values_kernel<VK, 1><<<grid, 512, 0, stream>>>(A);
    else if (A.splits <= 8) latent_values_kernel<VK, 2><<<grid, 512, 0, stream>>>(A);
    else if (A.splits <= 16) latent_values_kernel<VK, 4><<<grid, 512, 0, stream>>>(A);
    else if (A.splits <= 32) latent_values_kernel<VK, 8><<<grid, 512, 0, stream>>>(A);
    else if (A.splits <= 48) latent_values_kernel<VK, 12><<<grid, 512, 0, stream>>>(A);
    else latent_values_kernel<VK, 16><<<grid, 512, 0, stream>>>(A);
}

extern "C" int agave_latent_values(const float* part_o, const float* part_ml, int splits, const void* w, void* y, long ldy,
                                   const float* gate, long ldg, int rows, int heads, int vd, int out, hipStream_t stream) {
    AGAVE_CHECK(rows >= 0 && heads > 0 && vd > 0 && vd % 16 == 0 && vd <= LATENT_MAX_VALUE && out > 0, "latent_values: bad sizes rows=%d heads=%d vd=%d out=%d", rows, heads, vd, out);
    AGAVE_CHECK(splits >= 1 && splits <= LATENT_MAX_SPLITS && part_o && part_ml && w && y, "latent_values: null buffer or %d shares", splits);
    AGAVE_CHECK(ldy >= (long)heads * out && (!gate || ldg >= (long)heads * out) && ((uintptr_t)part_o % 16) == 0 && ((uintptr_t)w % 16) == 0,
                "latent_values: rows too short, or not aligned to 16 bytes");
    AGAVE_CHECK((long)rows * heads < 2147483647L, "latent_values: too many (row, head) pairs");
    if (rows == 0) return 0;
    LatentValuesArgs A{part_o, part_ml, splits, (const bf16*)w, (bf16*)y, ldy, gate, ldg, heads, vd, out};
    if (vd <= 128) launch_latent_values<4>(A, rows * heads, stream);
    else if (vd <= 256) launch_latent_values<8>(A, rows * heads, stream);
    else launch_latent_values<16>(A, rows * heads, stream);
    AGAVE_LAUNCH_CHECK("latent_values");
    return 0;
}
