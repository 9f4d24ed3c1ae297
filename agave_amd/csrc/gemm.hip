// Plain matrix product for gfx950: C[M,N] = A[M,K] * W[N,K]^T with 32-bit products and 32-bit
// accumulation, for any M, N, K and any mix of float / bf16 operands.
//
// This is the true 32-bit path of the linear layers and the fallback for sizes the bfloat16 kernels
// refuse.  It runs on the matrix cores' 32-bit instructions (v_mfma_f32_*: operands and sums are whole
// floats, nothing is narrowed), which do twice the multiply-adds a clock of the vector units; products of floats of 17 rows
// and more, where that is faster (split_instead), on the bfloat16 instructions, each float as three bfloat16 pieces that
// hold all its bits, in 32-bit sums.
// Weights are row-major [out, in] and used as y = W x, as in the reference
// (src/backend/backend.zig:474, 481).
//
// With few rows (decode steps, short prompts) the weights' way from memory bounds the product, with more the
// multiply-adds do: a kernel for up to eight rows, one for up to 64, one for more, and one for one or two rows that four
// elements do not fit.
#include "common_impl.h"
#include "fours.h"
#include "gate_act.h"
#include "mfma.h"

// ---------------------------------------------------------------- one or two rows that fours do not fit
// A wave per column of C, the lanes along K.  Bound by its trips to memory: a lane's loads are single elements, and a wave's 64 lie
// next to each other, where the kernel below asks for sixteen rows' lines with each.  The sums are held in double, which costs
// nothing here: in 32 bits they would be a lane's few products added across 64 lanes, and up to a third less exact than below.
// Measured, us, with the kernel below and so: 1 row by 130 x 2,049 in 32 bits 12.7 and 4.1, by 30,000 x 515 28.4 and 15.7, in bfloat16 40.0
// and 14.8, by 1,000 x 33 3.6 and 3.1; 2 rows by 16 x 4,097 29.5 and 5.1.  Errors against 64 bits 0.25 to 0.3e-7 after 0.6 to 1.6e-7.
#define FEW_ROWS 2
template <typename TA, typename TW, typename TC>
__global__ __launch_bounds__(256) void gemm_f32_few_rows_kernel(const TA* __restrict__ A, long lda, const TW* __restrict__ W, long ldw,
                                                                TC* __restrict__ C, long ldc, int M, int N, int K) {
    const int lane = threadIdx.x & 63, n = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (n >= N) return;
    const TW* w = W + (size_t)n * ldw;
    const TA* a[FEW_ROWS] = {A, A + (size_t)(M - 1) * lda};   // (a single row is made twice)
    double acc[FEW_ROWS] = {};
#pragma unroll 8
    for (int k = lane; k < K; k += 64) {
        const double wk = ld(w + k);
#pragma unroll
        for (int m = 0; m < FEW_ROWS; ++m) acc[m] = fma((double)ld(a[m] + k), wk, acc[m]);
    }
#pragma unroll
    for (int o = 1; o < 64; o *= 2)
#pragma unroll
        for (int m = 0; m < FEW_ROWS; ++m) acc[m] += __shfl_xor(acc[m], o);
    if (lane < M) st(C + (size_t)lane * ldc + n, (float)acc[lane == 0 ? 0 : 1]);
}

// ---------------------------------------------------------------- few rows
// A workgroup makes 16 columns of C for up to 64 rows (MT tiles of 16; more rows are cut into groups of
// 64, blockIdx.y); its NW waves share K and add their sums through LDS.  Per k-step of 16 a lane brings
// 16 bytes of a weight row and 16 of each A tile's row, straight from memory into the registers of
// v_mfma_f32_16x16x4_f32: that takes k in any order as long as both operands agree, so lane group g holds
// k = 4g .. 4g+3 and element e of the four goes into the e-th of four instructions.  U steps are asked
// for together, 256 bytes of every weight row.
// Bound by the weights' way from memory: NW is chosen so that about 2,048 waves stand in flight (see
// launch_skinny).  Measured in 32 bits, N x K = 10,752 x 2,048: 16 rows 31 us (2.8 TB/s), 64 rows 76 us; 2,048 x 5,376: 16 rows
// 26 us, 64 rows 64 us.  A wave per column with lanes along K took 82, 256, 89 us,
// vector tiles with 64 rows 646 us.
// A sum of K products in 32 bits loses more the longer its one running sum is.  One tile of rows keeps a
// running sum per step and element (16 a lane, of which each takes K / (16 NW) products), added in pairs
// at the end; with more tiles there is one per tile.
template <typename TA, typename TW, typename TC, int MT, int NW, bool VEC>
__global__ __launch_bounds__(NW * 64) void gemm_f32_skinny_kernel(const TA* __restrict__ A, long lda, const TW* __restrict__ W, long ldw,
                                                                  TC* __restrict__ C, long ldc, int M, int N, int K) {
    constexpr int U = MT > 2 ? 2 : 4;
    constexpr int S = MT == 1 ? 4 * U : 1;                        // running sums
    __shared__ float part[NW][MT * 256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 64;
    const TW* w = W + (size_t)min(n0 + r, N - 1) * ldw;           // (rows and columns outside are computed from the last one and not stored)
    const TA* a[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) a[t] = A + (size_t)min(m0 + 16 * t + r, M - 1) * lda;
    f32x4_t acc[S][MT] = {};
    for (int k0 = wave * U * 16; k0 < K; k0 += NW * U * 16) {
        f32x4_t wv[U], av[U][MT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + 16 * u + 4 * g;
            wv[u] = ld4<VEC>(w, k, K);
#pragma unroll
            for (int t = 0; t < MT; ++t) av[u][t] = ld4<VEC>(a[t], k, K);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    f32x4_t& sum = acc[(4 * u + e) % S][t];
                    sum = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u][t][e], wv[u][e], sum, 0, 0, 0);
                }
    }
#pragma unroll
    for (int s = S / 2; s > 0; s /= 2)
#pragma unroll
        for (int i = 0; i < s; ++i)
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[i][t] += acc[i + s][t];
    // acc[0][t][e] is row 16 t + 4 g + e, column r
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) part[wave][t * 256 + (4 * g + e) * 16 + r] = acc[0][t][e];
    __syncthreads();
    for (int i = threadIdx.x; i < MT * 256; i += NW * 64) {
        const int m = m0 + (i >> 4), n = n0 + (i & 15);
        if (m >= M || n >= N) continue;
        float sums[NW];
#pragma unroll
        for (int v = 0; v < NW; ++v) sums[v] = part[v][i];
#pragma unroll
        for (int s = NW / 2; s > 0; s /= 2)
#pragma unroll
            for (int v = 0; v < s; ++v) sums[v] += sums[v + s];
        st(C + (size_t)m * ldc + n, sums[0]);
    }
}

// ---------------------------------------------------------------- up to eight rows
// A workgroup makes 8 columns of C; its NW waves share K.  Eight rows fill half of v_mfma_f32_16x16x4_f32's sixteen, so the other
// half of rows and columns takes 16 further k: rows i and columns j of the result belong together where both are below 8 or
// both are not, and those two quarters are added at the end (the other two mean nothing).  A wave's load is then 128
// bytes, a whole line, of each of 8 weight rows, where sixteen rows took 64 of each; and 2,048 columns make a workgroup for each
// of the 256 compute units (with 16 a workgroup 128 of them pulled 2.2 TB/s).  Three chunks of 64 k are in flight a wave: a load leaves as
// soon as the chunk three before it is multiplied, without a condition around it (past the end it repeats the last four
// elements, which are not used), so that a wait leaves the younger ones in flight.
// Bound by the weights' way from memory.  Measured in 32 bits, us, three rows, before (sixteen columns a workgroup, four loads at a
// time) and now: 10,752 x 2,048 23.7 and 20.7 (4.3 TB/s), 2,048 x 5,376 20.3 and 13.0, 3,072 x 2,048 9.8 and 8.9, 2,048 x 2,048 9.0 and 6.2,
// 32,768 x 2,048 61 and 51 (5.3 TB/s); eight rows 26.8 and 22.5, 22.2 and 15.7, 10.4 and 10.9, 9.5 and 7.3, 67 and 55.
// A running sum per step and element, eight a lane in each half of k, as many as sixteen rows have.  Where fewer than sixteen waves share
// K they are added up half way and begun anew, so that each is of no more products than in groups of sixteen rows, which have twice
// the waves there.  Root mean square of the error against 64 bits over that of the result, in 1e-7, groups of sixteen, as one run and so:
// 3,072 x 2,048 0.94, 1.03, 0.94; 2,304 x 5,376 1.14, 1.38, 1.14; 5,376 x 2,048 1.03, 1.23, 1.03; 8,176 x 5,376 1.37, 1.78, 1.38; 32,768 x
// 5,376 1.78, 1.78, 1.38, in the same time.
// GATED (R = 2): W holds N rows of the gate matrix and behind them N of the up matrix; a workgroup makes 8 columns of either and leaves
// act(gate) * up.  The activation as a kernel of its own cost its start, its end and a round trip to memory, 2.8 us of some 21 (2 x 5,376
// columns of 2,048, three rows): 12 decode steps of 8 layers 7.37 -> 7.10 ms.
template <typename TA, typename TW, typename TC, int NW, int R, bool GATED>
__global__ __launch_bounds__(NW * 64, R == 2 ? 3 : 4) void gemm_f32_eight_rows_kernel(const TA* __restrict__ A, long lda, const TW* __restrict__ W,
                                                                      long ldw, TC* __restrict__ C, long ldc, int M, int N, int K, int act, float p0, float p1) {
    static_assert(!GATED || R == 2, "a block of the gate's columns and one of the up matrix's");
    constexpr int U = 2, CHUNK = U * 32, S = 3;
    __shared__ float part[NW][R * 64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 7, h = (lane >> 3) & 1, g = lane >> 4;
    const int n0 = blockIdx.x * 8 * (GATED ? 1 : R);
    const TW* w[R];                                               // (rows and columns outside are computed from the last one and not stored)
#pragma unroll
    for (int i = 0; i < R; ++i) w[i] = W + (GATED ? (size_t)i * N + min(n0 + r, N - 1) : (size_t)min(n0 + 8 * i + r, N - 1)) * ldw;
    const TA* a = A + (size_t)min(r, M - 1) * lda;
    const int lane_k = 16 * h + 4 * g;
    const int n_chunks = (K + CHUNK - 1) / CHUNK, n_iter = (n_chunks + NW - 1) / NW;
    f32x4_t acc[4 * U][R] = {};
    f32x4_t wv[S][U][R], av[S][U];
    // Chunks are dealt to the waves in turn, from another one on in every workgroup: rows that lie a multiple of 4 KB apart have
    // their like columns in one channel of the L2, and all workgroups would ask the same few at a time.
    const int first = (int)(blockIdx.x >> 3) % n_chunks;
    auto chunk_of = [&](int it) {
        const int c = min(it * NW + wave, n_chunks - 1) + first;
        return c < n_chunks ? c : c - n_chunks;
    };
    auto load = [&](int st, int it) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(chunk_of(it) * CHUNK + 32 * u + lane_k, K - 4);
#pragma unroll
            for (int i = 0; i < R; ++i) wv[st][u][i] = ld4<true>(w[i], k, K);
            av[st][u] = ld4<true>(a, k, K);
        }
    };
    auto add_up = [&]() {                                         // all running sums of a column block into the first
#pragma unroll
        for (int s = 2 * U; s > 0; s /= 2)
#pragma unroll
            for (int i = 0; i < s; ++i)
#pragma unroll
                for (int j = 0; j < R; ++j) acc[i][j] += acc[i + s][j];
    };
    f32x4_t first_half[R] = {};
    const int half = NW < 16 ? n_iter / 2 : 0;
    auto use = [&](int st, int it) {
        if (it * NW + wave >= n_chunks) return;
        if (NW < 16 && half > 0 && it == half) {
            add_up();
#pragma unroll
            for (int j = 0; j < R; ++j) first_half[j] = acc[0][j];
#pragma unroll
            for (int i = 0; i < 4 * U; ++i)
#pragma unroll
                for (int j = 0; j < R; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
        const int c = chunk_of(it);
        if ((c + 1) * CHUNK > K) {                                // the last chunk, where columns are missing from it
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (c * CHUNK + 32 * u + lane_k >= K) {
                    av[st][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int i = 0; i < R; ++i) wv[st][u][i] = av[st][u];
                }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < R; ++i)
                    acc[4 * u + e][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[st][u][e], wv[st][u][i][e], acc[4 * u + e][i], 0, 0, 0);
    };
    if (n_iter < S) {                                             // (nothing is asked for twice)
        load(0, 0);
        if (n_iter > 1) load(1, 1);
        use(0, 0);
        if (n_iter > 1) use(1, 1);
    } else {
#pragma unroll
        for (int st = 0; st < S; ++st) load(st, st);
        int it = 0;
        for (; it + 2 * S <= n_iter; it += S)                     // every load is of a chunk that exists
#pragma unroll
            for (int st = 0; st < S; ++st) {
                __builtin_amdgcn_sched_barrier(0);
                use(st, it + st);
                __builtin_amdgcn_sched_barrier(0);
                load(st, it + st + S);
            }
#pragma unroll
        for (int st = 0; st < S; ++st) {                          // the last S to 2 S - 1
            __builtin_amdgcn_sched_barrier(0);
            use(st, it + st);
            __builtin_amdgcn_sched_barrier(0);
            if (it + st + S < n_iter) load(st, it + st + S);
        }
#pragma unroll
        for (int st = 0; st < S - 1; ++st) use(st, it + st + S);
    }
    add_up();
    if (NW < 16)
#pragma unroll
        for (int j = 0; j < R; ++j) acc[0][j] += first_half[j];
    // acc[0][i][e] is row 4 g + e, column lane % 16; the quarters that mean something: rows below 8 in lane groups 0 and 1 with
    // columns below 8, and what lies 8 rows (two lane groups) and 8 columns further, 40 lanes in all
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float sum = acc[0][i][e] + __shfl_xor(acc[0][i][e], 40, 64);
            if (h == 0 && g < 2) part[wave][(4 * g + e) * 8 * R + 8 * i + r] = sum;
        }
    __syncthreads();
    const int m = threadIdx.x / (8 * R), n = n0 + threadIdx.x % (GATED ? 8 : 8 * R);
    if (m >= M || (!GATED && n >= N)) return;                     // (GATED: all sixteen lanes of a row stay for the exchange)
    float sums[NW];
#pragma unroll
    for (int v = 0; v < NW; ++v) sums[v] = part[v][threadIdx.x];
#pragma unroll
    for (int s = NW / 2; s > 0; s /= 2)
#pragma unroll
        for (int v = 0; v < s; ++v) sums[v] += sums[v + s];
    if (GATED) {
        const float up = __shfl_xor(sums[0], 8);                  // column n of the up matrix lies eight lanes further
        if ((threadIdx.x & 8) == 0 && n < N) st(C + (size_t)m * ldc + n, gate_form(sums[0], up, act, p0, p1));
    } else {
        st(C + (size_t)m * ldc + n, sums[0]);
    }
}

// ---------------------------------------------------------------- more rows
// A workgroup of 4 waves makes BM x 64 of C.  Stages of 32 k go through LDS in two buffers: while a
// stage is multiplied the next one's loads are in flight into registers.  v_mfma_f32_32x32x2_f32 takes
// k in any order as long as both operands agree: a lane reads 16 bytes of a row (k = 8 j + 4 h .. + 3 for
// half h of the wave) and the four elements go into four instructions.  Rows of 36 floats keep the
// 16-byte reads of neighbouring rows on different banks.
// Bound by the multiply-adds: 4 waves keep the CU's matrix units busy from 37 KB of LDS a workgroup, so
// that others stand by for the barriers.  BM = 64: a wave per quarter of the tile.  BM = 32, where the
// larger tiles would leave compute units without one: two waves side by side, two sharing every
// stage's k, added at the end.  Tiles one below the other follow each other on an XCD (workgroups go
// to the 8 XCDs in turn), so that a panel of weights is read into one L2.
// Measured in 32 bits: 777 rows by 10,752 x 2,048 352 us (97 TFLOP/s), by 2,048 x 5,376 213 us; 2,048 rows
// by 10,752 x 2,048 840 us (107 TFLOP/s).  Vector multiply-adds from 64 x 64 tiles took 1,280, 837 and 2,471 us.
#define TN 64
#define TK 32
#define TS (TK + 4)
// S: running sums of an element (of each half of k where BM = 32); two where few rows come here that groups of rows, with a running
// sum per quarter of k, would otherwise take, and beside the rings (2,048 columns 8.1e-7 of the result with one, 5.7e-7 with two, in the same
// time).
template <typename TA, typename TW, typename TC, int BM, bool VEC, int S>
__global__ __launch_bounds__(256) void gemm_f32_tiled_kernel(const TA* __restrict__ A, long lda, const TW* __restrict__ W, long ldw,
                                                             TC* __restrict__ C, long ldc, int M, int N, int K, int m_tiles, int tiles) {
    constexpr int AR = BM / 32;                                   // rows of A a thread brings per stage
    __shared__ float As[2][BM * TS], Ws[2][TN * TS];
    const int tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int m0 = tile % m_tiles * BM, n0 = tile / m_tiles * TN;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wn = wave & 1;                                      // which 32 columns
    const int wm = BM == 64 ? wave >> 1 : 0;                      // which 32 rows
    const int wk = BM == 64 ? 0 : wave >> 1;                      // which half of a stage's k
    const int lr = threadIdx.x >> 3, lk = (threadIdx.x & 7) * 4;  // loader: a row, 4 neighbouring k
    const TA* a[AR];
    const TW* w[2];
#pragma unroll
    for (int i = 0; i < AR; ++i) a[i] = A + (size_t)min(m0 + lr + 32 * i, M - 1) * lda;
#pragma unroll
    for (int i = 0; i < 2; ++i) w[i] = W + (size_t)min(n0 + lr + 32 * i, N - 1) * ldw;
    f32x4_t ra[AR], rw[2];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < AR; ++i) ra[i] = ld4<VEC>(a[i], k0 + lk, K);
#pragma unroll
        for (int i = 0; i < 2; ++i) rw[i] = ld4<VEC>(w[i], k0 + lk, K);
    };
    auto put = [&](int b) {
#pragma unroll
        for (int i = 0; i < AR; ++i) *(f32x4_t*)&As[b][(lr + 32 * i) * TS + lk] = ra[i];
#pragma unroll
        for (int i = 0; i < 2; ++i) *(f32x4_t*)&Ws[b][(lr + 32 * i) * TS + lk] = rw[i];
    };
    f32x16_t sums[S] = {};
    fetch(0);
    put(0);
    __syncthreads();
    const int row = (lane & 31) * TS + (lane >> 5) * 4;
    for (int k0 = 0, b = 0; k0 < K; k0 += TK, b ^= 1) {
        if (k0 + TK < K) fetch(k0 + TK);
        const float* pa = &As[b][wm * 32 * TS + row];
        const float* pw = &Ws[b][wn * 32 * TS + row];
#pragma unroll
        for (int j = 0; j < (BM == 64 ? 4 : 2); ++j) {
            const int o = 8 * j + (BM == 64 ? 0 : 16 * wk);
            const f32x4_t va = *(const f32x4_t*)(pa + o), vw = *(const f32x4_t*)(pw + o);
#pragma unroll
            for (int e = 0; e < 4; ++e) sums[e % S] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[e], vw[e], sums[e % S], 0, 0, 0);
        }
        if (k0 + TK < K) put(b ^ 1);                              // (the other buffer was last read before the barrier below)
        __syncthreads();
    }
    f32x16_t acc = sums[0];
    if (S == 2) acc += sums[S - 1];
    if (BM == 32) {                                               // the second pair's sums, 32 x 64 floats, through the first buffer
        static_assert(64 * 17 * 2 <= 2 * 32 * TS, "a wave's sums, padded by one float a lane, fit");
        float* half = &As[0][0] + wn * 64 * 17;
        if (wk == 1)
#pragma unroll
            for (int e = 0; e < 16; ++e) half[lane * 17 + e] = acc[e];
        __syncthreads();
        if (wk == 1) return;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] += half[lane * 17 + e];
    }
    // acc[e] is row 8 (e/4) + 4 (lane/32) + e%4, column lane%32
    const int n = n0 + wn * 32 + (lane & 31);
    if (n >= N) return;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm * 32 + 8 * (e / 4) + 4 * (lane >> 5) + e % 4;
        if (m < M) st(C + (size_t)m * ldc + n, acc[e]);
    }
}

// ---------------------------------------------------------------- more rows, 32-bit operands that fours fit
// WM x WN waves make BM x BN of C, a wave BM/WM x BN/WN in tiles of 32 x 32.  Stages of 32 k come into LDS straight from memory, in a
// ring of NS buffers: while a stage is multiplied the next NS - 1 are on their way, and no wave spends registers or LDS writes on
// bringing them (the kernel above does, and waits for a stage's loads with nothing else in flight).  A row's eight 16-byte pieces are
// permuted by its number, so that the 32 rows of a read lie on different banks.  The waits are for "all but the youngest n": loads
// and LDS reads come back in the order they were asked for.
// Bound by the multiply-adds (64 clocks for 32 x 32 x 2).  The ring of 32 x 128 tiles is made so large (80 KB) that two workgroups share a
// compute unit: a third (64 x 64 tiles in 48 KB) made 624 tiles 16 % slower.  Measured in 32 bits, us, the kernel above and this one:
// 777 rows by 10,752 x 2,048 370 and 309 (111 TFLOP/s), by 2,048 x 5,376 208 and 174, by 2,048 x 2,048 85 and 72, by 3,072 x 2,048 122 and
// 108; 300 rows by 10,752 x 2,048 175 and 134; 2,048 rows 870 and 730 (124 TFLOP/s).
// S running sums of an element, each of every S-th k.
template <int BM, int BN, int WM, int WN, int S, int NS>
__global__ __launch_bounds__(WM * WN * 64) void gemm_f32_ring_kernel(const float* __restrict__ A, long lda, const float* __restrict__ W,
                                                                     long ldw, float* __restrict__ C, long ldc, int M, int N, int K,
                                                                     int m_tiles, int tiles) {
    constexpr int NWV = WM * WN, MT = BM / WM / 32, NT = BN / WN / 32;
    constexpr int LA = BM / 8 / NWV, LW = BN / 8 / NWV, LOADS = LA + LW;      // of a kilobyte, eight rows, a wave and stage
    static_assert(LA * NWV * 8 == BM && LW * NWV * 8 == BN && MT * WM * 32 == BM && NT * WN * 32 == BN, "whole loads and tiles a wave");
    constexpr int A_BYTES = BM * 128, STAGE = (BM + BN) * 128;
    __shared__ __attribute__((aligned(16))) unsigned char ring[NS * STAGE];
    // (tiles one below the other follow each other on an XCD, as above)
    const int tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int m0 = tile % m_tiles * BM, n0 = tile / m_tiles * BN;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave % WN, wm = wave / WN, r = lane & 31, h = lane >> 5;
    const unsigned char* ap = (const unsigned char*)(A + (size_t)m0 * lda);
    const unsigned char* wp = (const unsigned char*)(W + (size_t)n0 * ldw);
    unsigned aoff[LA], woff[LW];                                  // (rows outside: the last one again, not stored)
    const int row0 = wave * 8 + (lane >> 3);                      // this lane's row of load 0; a load further: 8 NWV rows
    auto piece = [&](int i) { return (lane & 7) ^ (((row0 + i * NWV * 8) >> 1) & 7); };       // the four k it brings
#pragma unroll
    for (int i = 0; i < LA; ++i) aoff[i] = (unsigned)min(row0 + i * NWV * 8, M - 1 - m0) * (unsigned)(lda * 4) + piece(i) * 16;
#pragma unroll
    for (int i = 0; i < LW; ++i) woff[i] = (unsigned)min(row0 + i * NWV * 8, N - 1 - n0) * (unsigned)(ldw * 4) + piece(i) * 16;
    auto to_lds = [&](const unsigned char* src, int at) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)(ring + at), 16, 0, 0);
    };
    const int n_stage = (K + 31) / 32, rest = K & 31;             // rest: k of a broken last stage
    auto mend = [&]() {                                           // pieces past the last k: the stage's first one, zeroed when read
#pragma unroll
        for (int i = 0; i < LA; ++i) aoff[i] -= piece(i) * 4 >= rest ? piece(i) * 16 : 0;
#pragma unroll
        for (int i = 0; i < LW; ++i) woff[i] -= piece(i) * 4 >= rest ? piece(i) * 16 : 0;
    };
    auto fetch = [&](int buf) {
#pragma unroll
        for (int i = 0; i < LA; ++i) to_lds(ap + aoff[i], buf + (i * NWV + wave) * 1024);
#pragma unroll
        for (int i = 0; i < LW; ++i) to_lds(wp + woff[i], buf + A_BYTES + (i * NWV + wave) * 1024);
        ap += 128;
        wp += 128;
    };
    // v_mfma_f32_32x32x2_f32 takes k in any order as long as both operands agree: the four elements of piece 2 j + h go into four
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)ring;
    unsigned at[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) at[j] = lds0 + r * 128 + (((2 * j + h) ^ ((r >> 1) & 7)) * 16);
    const unsigned a_wave = wm * MT * 4096, w_wave = A_BYTES + wn * NT * 4096;
    f32x16_t sums[S][MT][NT] = {};
    static_for<0, NS - 1>([&](auto p) {
        if (p.value < n_stage) {
            if (p.value == n_stage - 1 && rest != 0) mend();
            fetch(p.value * STAGE);
        }
    });
    int buf = 0, free_buf = (NS - 1) * STAGE;
    // a stage; FLIGHT: loads of the stages behind it that may still be on their way; ASK: another stage's are asked for; BROKEN:
    // pieces of it lie past the last k
    auto stage = [&](auto flight, auto ask, auto broken) {
        constexpr int n = decltype(flight)::value;
        static_assert(n < 64, "the counter holds six bits");
        __builtin_amdgcn_s_waitcnt(0x0F70 | (n & 15) | ((n >> 4) << 14));
        __builtin_amdgcn_s_barrier();                             // (all that this stage needs has come, and the one before it is read)
        frag16 va[4][MT], vw[4][NT];
        static_for<0, 4>([&](auto j) {
            static_for<0, MT>([&](auto t) { lds_read16<t.value * 4096>(va[j.value][t.value], at[j.value] + a_wave + buf); });
            static_for<0, NT>([&](auto t) { lds_read16<t.value * 4096>(vw[j.value][t.value], at[j.value] + w_wave + buf); });
        });
        if constexpr (decltype(ask)::value != 0) fetch(free_buf);
        static_for<0, 4>([&](auto j) {
            __builtin_amdgcn_sched_barrier(0);                    // (each piece's multiplications as soon as it is here)
            lds_settle_to<(3 - j.value) * (MT + NT)>();
#pragma unroll
            for (int t = 0; t < MT; ++t) lds_use(va[j.value][t]);
#pragma unroll
            for (int t = 0; t < NT; ++t) lds_use(vw[j.value][t]);
            if (decltype(broken)::value != 0 && (2 * j.value + h) * 4 >= rest) {
#pragma unroll
                for (int t = 0; t < MT; ++t) va[j.value][t].u = uint4{0, 0, 0, 0};
#pragma unroll
                for (int t = 0; t < NT; ++t) vw[j.value][t].u = uint4{0, 0, 0, 0};
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int u = 0; u < NT; ++u)
                        sums[e % S][t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(f32x4_t, va[j.value][t].r)[e],
                                                                                 __builtin_bit_cast(f32x4_t, vw[j.value][u].r)[e],
                                                                                 sums[e % S][t][u], 0, 0, 0);
        });
        free_buf = buf;
        buf = buf == (NS - 1) * STAGE ? 0 : buf + STAGE;
    };
    for (int st = 0; st + NS < n_stage; ++st) stage(IntC<(NS - 2) * LOADS>{}, IntC<1>{}, IntC<0>{});
    if (n_stage >= NS) {                                          // the last stage's loads
        if (rest != 0) mend();
        stage(IntC<(NS - 2) * LOADS>{}, IntC<1>{}, IntC<0>{});
    }
    static_for<0, NS - 2>([&](auto p) {                           // NS - 1 stages are left, or all that there are
        constexpr int left = NS - 1 - p.value;
        if (n_stage >= left) stage(IntC<(left - 1) * LOADS>{}, IntC<0>{}, IntC<0>{});
    });
    if (rest != 0) stage(IntC<0>{}, IntC<0>{}, IntC<1>{});
    else stage(IntC<0>{}, IntC<0>{}, IntC<0>{});
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) {
#pragma unroll
            for (int s = S / 2; s > 0; s /= 2)
#pragma unroll
                for (int i = 0; i < s; ++i) sums[i][t][u] += sums[i + s][t][u];
            // element e is row 8 (e/4) + 4 (lane/32) + e%4, column lane%32
            const int n = n0 + (wn * NT + u) * 32 + r;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + (wm * MT + t) * 32 + 8 * (e / 4) + 4 * h + e % 4;
                if (m < M && n < N) C[(size_t)m * ldc + n] = sums[0][t][u][e];
            }
        }
}

// ---------------------------------------------------------------- more rows, on the bfloat16 instructions
// A float is the sum of three bfloat16 values exactly (24 bits are three times 8: the nearest bfloat16, the nearest of what is left, and
// the rest) if its last bit is one that a bfloat16 can hold: not below 2^-133, where a float's go down to 2^-149.  So both operands are
// cut as PIECES_UP times as large, and the sums brought down again (uncut so, rows of 2^-112, -116, -120 and -124 had errors of 2.4e-7,
// 2.2e-6, 3.5e-5 and 5.6e-4).  A product of floats is then the sum of nine exact products of pieces.  The six large ones are made here on
// v_mfma_f32_16x16x32_bf16, whose sums are 32-bit; the three left out are below 2^-24 of the product.  The large pieces' products have a
// running sum of their own, the five corrections another.  That sum takes 32 products an instruction, the 32-bit
// instruction two or four, and so rounds a sixteenth as often.
// Bound by the multiply-adds and, where a stage's tiles are few, by their chain of loads, cuts and barriers.  us, the kernels above and
// this one with its sums of slices: 777 rows by 10,752 x 2,048 325 and 232 (147 TFLOP/s; the 32-bit instructions reach 153 on the largest
// products), by 2,048 x 5,376 174 and 110, by 2,048 x 2,048 71 and 51, by 3,072 x 2,048 119 and 76; 2,048 rows by 10,752 x 2,048 728 and
// 456 (198 TFLOP/s); 64 rows 41 and 31, 58 and 25, 25 and 15, 25 and 17.  Making the operands larger takes 2 to 3 % of it, with up to 64
// rows by many columns up to 8.  Root mean
// square of the error against 64 bits over that of the result, in 1e-7: 2,048 columns 5.7 (rings) and 2.7 whole, 1.9 in two slices, 1.3
// in four; 5,376 9.3 and 4.6, 3.2, 2.2.
// A piece of an infinity or NaN is none of the two, and floats from 2^104 on and sums from 2^80 on leave 32 bits when they are made so much
// larger: an element that does not come out finite is made again from the floats themselves, in 64 bits.
// WM x WN = 2 x 2 waves make BM rows x BN columns of C.  A stage of 32 k is brought into registers a stage ahead, cut into pieces there
// and put into LDS in the order the instruction reads its operands; two workgroups share a compute unit, and one cuts while the other
// multiplies.
#define PIECES_UP 0x1p24f
struct Pieces { uint32_t u[3]; };                                 // two floats' pieces, largest first, side by side
__device__ __forceinline__ Pieces pieces_of(float a, float b) {
    Pieces p;
    a *= PIECES_UP, b *= PIECES_UP;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        p.u[i] = f32x2_to_bf16x2(a, b);
        a -= __builtin_bit_cast(float, p.u[i] << 16);
        b -= __builtin_bit_cast(float, p.u[i] & 0xffff0000u);
    }
    return p;
}
template <int BM, int BN>
__global__ __launch_bounds__(256, 2) void gemm_f32_split_kernel(const float* __restrict__ A, long lda, const float* __restrict__ W,
                                                                long ldw, float* __restrict__ C, long ldc, int M, int N, int K,
                                                                int m_tiles, int tiles, long part_stride) {
    constexpr int ROWS = BM + BN, UNITS = ROWS / 64;              // 8 k of a row: a unit; so many of a stage a thread
    constexpr int MT = BM / 32, NT = BN / 32;                     // tiles of 16 x 16 of a wave
    constexpr int PLANE = ROWS * 64;                              // bytes of one piece of all rows
    static_assert(BM % 64 == 0 && BN % 64 == 0, "a pass of the loads is of rows of A or of W");
    __shared__ __attribute__((aligned(16))) unsigned char stage[3 * PLANE];
    const int tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);      // (one below the other on an XCD, as above)
    if (tile >= tiles) return;
    const int m0 = tile % m_tiles * BM, n0 = tile / m_tiles * BN;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave & 1, wn = wave >> 1, j = lane & 15, g = lane >> 4;
    // gridDim.y workgroups share a tile's k and leave their sums in slices of C
    const int stages = (K + 31) / 32;
    const int st0 = (int)((long)blockIdx.y * stages / gridDim.y), st_end = (int)((long)(blockIdx.y + 1) * stages / gridDim.y);
    C += (size_t)blockIdx.y * part_stride;

    const int ug = threadIdx.x & 3, ur = threadIdx.x >> 2;        // unit u: row ur + 64 u of the stage, k 8 ug .. + 8
    const float* src[UNITS];
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {                             // (rows outside: the last one again, not stored)
        const int row = ur + 64 * u;
        src[u] = row < BM ? A + (size_t)min(m0 + row, M - 1) * lda : W + (size_t)min(n0 + row - BM, N - 1) * ldw;
    }
    f32x4_t raw[UNITS][2];
    auto fetch = [&](int st) {
        const int k = st * 32 + 8 * ug;                           // (K is a multiple of 4; past it the last four again, cleared below)
#pragma unroll
        for (int u = 0; u < UNITS; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i) raw[u][i] = *reinterpret_cast<const f32x4_t*>(src[u] + min(k + 4 * i, K - 4));
    };
    // a unit's place: tile of 16 rows, lane row % 16 + 16 ug of the operand, moved so that a store's lanes take different banks
    const unsigned put = (ur >> 4) * 1024 + ug * 256 + (((ur & 15) ^ (2 * ug)) * 16);
    const unsigned get = g * 256 + ((j ^ (2 * g)) * 16);
    f32x4_t high[MT][NT] = {}, low[MT][NT] = {};
    if (st0 < st_end) fetch(st0);
    for (int st = st0; st < st_end; ++st) {
        uint4 cut[UNITS][3];
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            if (st * 32 + 32 > K) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    if (st * 32 + 8 * ug + 4 * i >= K) raw[u][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
            const Pieces a = pieces_of(raw[u][0][0], raw[u][0][1]), b = pieces_of(raw[u][0][2], raw[u][0][3]);
            const Pieces c = pieces_of(raw[u][1][0], raw[u][1][1]), d = pieces_of(raw[u][1][2], raw[u][1][3]);
#pragma unroll
            for (int p = 0; p < 3; ++p) cut[u][p] = make_uint4(a.u[p], b.u[p], c.u[p], d.u[p]);
        }
        __builtin_amdgcn_s_barrier();                             // (every wave has its operands of the stage before this one)
#pragma unroll
        for (int u = 0; u < UNITS; ++u)
#pragma unroll
            for (int p = 0; p < 3; ++p) *reinterpret_cast<uint4*>(stage + p * PLANE + u * 4096 + put) = cut[u][p];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        fetch(st + 1 < st_end ? st + 1 : st);                     // (the last stage's once more, not used)
        __builtin_amdgcn_sched_barrier(0);                        // (or the compiler asks when it needs them)
        frag16 w[NT][3];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int p = 0; p < 3; ++p)
                w[t][p].u = *reinterpret_cast<const uint4*>(stage + p * PLANE + (BM / 16 + wn * NT + t) * 1024 + get);
#pragma unroll
        for (int r = 0; r < MT; ++r) {
            frag16 x[3];
#pragma unroll
            for (int p = 0; p < 3; ++p) x[p].u = *reinterpret_cast<const uint4*>(stage + p * PLANE + (wm * MT + r) * 1024 + get);
#pragma unroll
            for (int t = 0; t < NT; ++t) high[r][t] = mfma_16x16x32(w[t][0], x[0], high[r][t]);
#pragma unroll
            for (int t = 0; t < NT; ++t) low[r][t] = mfma_16x16x32(w[t][2], x[0], low[r][t]);
#pragma unroll
            for (int t = 0; t < NT; ++t) low[r][t] = mfma_16x16x32(w[t][0], x[2], low[r][t]);
#pragma unroll
            for (int t = 0; t < NT; ++t) low[r][t] = mfma_16x16x32(w[t][1], x[1], low[r][t]);
#pragma unroll
            for (int t = 0; t < NT; ++t) low[r][t] = mfma_16x16x32(w[t][1], x[0], low[r][t]);
#pragma unroll
            for (int t = 0; t < NT; ++t) low[r][t] = mfma_16x16x32(w[t][0], x[1], low[r][t]);
        }
    }
    // high[r][t][e]: row 16 r + j, column 16 t + 4 g + e of the wave's
    const bool fours = ldc % 4 == 0 && ((uintptr_t)C & 15) == 0;
#pragma unroll
    for (int r = 0; r < MT; ++r) {
        const int m = m0 + (wm * MT + r) * 16 + j;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int n = n0 + (wn * NT + t) * 16 + 4 * g;
            f32x4_t s = (high[r][t] + low[r][t]) * (1.0f / (PIECES_UP * PIECES_UP));
            if (m >= M || n >= N) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (!(__builtin_fabsf(s[e]) < __builtin_inff()) && n + e < N) {
                    double again = 0.0;
                    const float *pa = A + (size_t)m * lda, *pw = W + (size_t)(n + e) * ldw;
                    for (int k = st0 * 32; k < min(st_end * 32, K); ++k) again = fma((double)pa[k], (double)pw[k], again);
                    s[e] = (float)again;
                }
            float* dst = C + (size_t)m * ldc + n;
            if (fours && n + 4 <= N) {
                *reinterpret_cast<f32x4_t*>(dst) = s;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) dst[e] = s[e];
            }
        }
    }
}

template <int BM, int BN>
static void launch_split(const float* A, long lda, const float* W, long ldw, float* C, long ldc, int M, int N, int K, int slices, long part_stride,
                         hipStream_t stream) {
    const int m_tiles = (M + BM - 1) / BM, tiles = m_tiles * ((N + BN - 1) / BN);
    gemm_f32_split_kernel<BM, BN><<<dim3((tiles + 7) / 8 * 8, slices), 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, m_tiles, tiles, part_stride);
}

// ---------------------------------------------------------------- launch
#define SKINNY_M 64
#define COMPUTE_UNITS 256

template <typename TA, typename TW, typename TC, int MT, bool VEC>
static void launch_skinny(const TA* A, long lda, const TW* W, long ldw, TC* C, long ldc, int M, int N, int K, hipStream_t stream) {
    const dim3 groups((N + 15) / 16, (M + 63) / 64);
    // waves a workgroup: enough for 2,048 in all, as far as K has a stretch for each
    const int want = (2048 + groups.x - 1) / groups.x, most = (K + 63) / 64;
    const int waves = want < most ? want : most;
    if (waves > 8 && MT <= 2)
        gemm_f32_skinny_kernel<TA, TW, TC, MT <= 2 ? MT : 1, 16, VEC><<<groups, 1024, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K);
    else if (waves > 4)
        gemm_f32_skinny_kernel<TA, TW, TC, MT, 8, VEC><<<groups, 512, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K);
    else
        gemm_f32_skinny_kernel<TA, TW, TC, MT, 4, VEC><<<groups, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K);
}

// Up to eight rows: 16 waves for each of up to 256 workgroups of one block of columns, 8 for up to 512 (two a compute unit), and beyond
// that two blocks a workgroup of 4 waves, which take the rows of A once for both (of 512 columns and less only from 768 blocks on: 4
// waves have two chunks each then; 5,376 x 512, one row, 5.85 us with four and 5.53 with eight, 8,176 x 512 6.0 and 7.0).
template <typename TA, typename TW, typename TC>
static void launch_eight_rows(const TA* A, long lda, const TW* W, long ldw, TC* C, long ldc, int M, int N, int K, hipStream_t stream) {
    const int blocks = (N + 7) / 8;
    if (blocks <= COMPUTE_UNITS) gemm_f32_eight_rows_kernel<TA, TW, TC, 16, 1, false><<<blocks, 1024, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, 0, 0.f, 0.f);
    else if (blocks <= (K > 512 ? 2 : 3) * COMPUTE_UNITS) gemm_f32_eight_rows_kernel<TA, TW, TC, 8, 1, false><<<blocks, 512, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, 0, 0.f, 0.f);
    else gemm_f32_eight_rows_kernel<TA, TW, TC, 4, 2, false><<<(blocks + 1) / 2, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, 0, 0.f, 0.f);
}

template <int BM, int BN, int WM, int WN, int S, int NS>
static void launch_ring(const float* A, long lda, const float* W, long ldw, float* C, long ldc, int M, int N, int K, hipStream_t stream) {
    const int m_tiles = (M + BM - 1) / BM, tiles = m_tiles * ((N + BN - 1) / BN);
    gemm_f32_ring_kernel<BM, BN, WM, WN, S, NS><<<(tiles + 7) / 8 * 8, WM * WN * 64, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, m_tiles, tiles);
}

// Rows a tile of gemm_f32_ring_kernel, 0: not that kernel.  Tiles of 32 x 128, two at a time on a compute unit, or, where that is less by
// the times of so many tiles a compute unit (measured at 2,048 columns, us; what is left over after whole rounds takes as long as if it
// were alone), of 128 x 128, 130 us each.  The kernel of 32 x 64 tiles keeps products of one round of those (37.5 us), which halve the k
// between waves.  Up to 64 rows stay in groups of 64 rows where these have eight running sums a product or more (under 8,192 columns), and
// are added up as in groups with four.
static const double RING_32[] = {0, 44, 72, 109, 146, 195};
static int ring_rows(int M, int N) {
    auto a_unit = [&](int bm) { return (((long)M + bm - 1) / bm * (((long)N + 127) / 128) + COMPUTE_UNITS - 1) / COMPUTE_UNITS; };
    if (M <= SKINNY_M) return N >= (M > 32 ? 8192 : 16384) ? 32 : 0;
    if ((long)((M + 31) / 32) * ((N + TN - 1) / TN) <= COMPUTE_UNITS) return 0;
    const long n32 = a_unit(32);
    // three tiles of 32 x 128 a unit, of which two run at a time, take 117 to 133, and three of 64 x 64 in the kernel above 118 (5,376 columns
    // 320 to 338 and 298; 1,500 rows by 2,048 x 2,048 132.8 and 118.3, 512 by 5,376 x 10,752 667 and 591)
    if (n32 == 3 && ((long)M + 63) / 64 * (((long)N + TN - 1) / TN) <= 3 * COMPUTE_UNITS) return 0;
    return (n32 <= 5 ? RING_32[n32] : 35.0 * n32) <= 130.0 * a_unit(128) ? 32 : 128;
}

// Microseconds of a product on a tile shape of gemm_f32_split_kernel: of a launch, and of a stage of 32 k with so many tiles a compute unit
// (two workgroups share a unit, up to four of the smaller tiles).  Least squares over the times of 500 products of 33 to 6,000 rows by 512
// to 11,000 x 512 to 11,000 in up to eight slices, from which they are 3 to 4 % off.
struct SplitShape { int bm, bn; double start, stage[12]; };
static const double SPLIT_TILES[12] = {0.25, 0.5, 1, 1.25, 1.5, 2, 2.5, 3, 4, 5, 6, 8};
static const SplitShape SPLIT_SHAPES[4] = {
    {128, 128, 6.4, {1.63, 1.66, 1.71, 2.06, 2.11, 2.38, 4.05, 4.28, 4.59, 6.46, 7.04, 9.73}},
    {64, 128, 5.2, {1.12, 1.12, 1.15, 1.36, 1.37, 1.48, 2.12, 2.25, 3.02, 3.48, 4.28, 5.61}},
    {128, 64, 5.1, {1.06, 1.05, 1.09, 1.30, 1.32, 1.45, 2.03, 2.15, 2.94, 3.41, 4.18, 5.56}},
    {64, 64, 4.4, {0.74, 0.74, 0.76, 0.87, 0.88, 0.92, 1.33, 1.39, 1.62, 2.04, 2.52, 3.20}}};
// (just past a whole number of tiles a unit some have one more, which is what the others then wait for: as long as the next measured load, or
// with more than three as the next whole number.  135 rows by 10,896 x 4,888 in tiles of 64 x 64, 2.004 a unit: 206, taken for 2 of them 149)
static double split_stage(const SplitShape& s, double tiles_a_unit) {
    double t = tiles_a_unit;
    if (t > 3) t = ceil(t);
    else if (t > 2 && t < 2.5) t = 2.5;
    else if (t > 1 && t < 1.25) t = 1.25;
    if (t <= SPLIT_TILES[0]) return s.stage[0];
    for (int i = 1; i < 12; ++i)
        if (t <= SPLIT_TILES[i]) return s.stage[i - 1] + (s.stage[i] - s.stage[i - 1]) * (t - SPLIT_TILES[i - 1]) / (SPLIT_TILES[i] - SPLIT_TILES[i - 1]);
    return s.stage[11] * t / SPLIT_TILES[11];
}
struct SplitPlan { int shape, slices; double us; };
// The fastest shape in so many slices.  Adding them up takes a launch, and 4 bytes each of them and the result at 3.5 TB/s; large operands
// come at 5 TB/s (33 rows by 10,240 x 4,096 in eight slices 43 us).
static SplitPlan split_in(int M, int N, int K, int slices) {
    SplitPlan best = {0, slices, 1e30};
    const int stages = ((K + 31) / 32 + slices - 1) / slices;
    const double memory = ((double)M + N) * K * 4 / 5.0e6;
    for (int i = 0; i < 4; ++i) {
        const SplitShape& s = SPLIT_SHAPES[i];
        const double tiles = (double)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn);
        double us = s.start + std::max(split_stage(s, tiles * slices / COMPUTE_UNITS) * stages, memory);
        if (slices > 1) us += 2.0 + (slices + 1.0) * M * N * 4 / 3.5e6;
        if (us < best.us) best.shape = i, best.us = us;
    }
    return best;
}
// The fastest of `least` to `most` slices, powers of two, of eight stages and more; rather one than slices that are as fast (1,200 rows by
// 10,752 x 4,096 578 and 622 in two, taken for 593 and 589).
static SplitPlan plan_split(int M, int N, int K, int least, int most) {
    SplitPlan best = {0, least, 1e30};
    const int stages = (K + 31) / 32;
    for (int z = least; z <= most && (z == 1 || stages / z >= 8); z *= 2) {
        const SplitPlan of_z = split_in(M, N, K, z);
        if (of_z.us < (best.slices == 1 && z > 1 ? 0.99 : 1.0) * best.us) best = of_z;
    }
    return best;
}
static void launch_split(const SplitPlan& plan, const float* A, long lda, const float* W, long ldw, float* C, long ldc, int M, int N, int K,
                         long part_stride, hipStream_t stream) {
    switch (plan.shape) {
        case 0: return launch_split<128, 128>(A, lda, W, ldw, C, ldc, M, N, K, plan.slices, part_stride, stream);
        case 1: return launch_split<64, 128>(A, lda, W, ldw, C, ldc, M, N, K, plan.slices, part_stride, stream);
        case 2: return launch_split<128, 64>(A, lda, W, ldw, C, ldc, M, N, K, plan.slices, part_stride, stream);
        default: return launch_split<64, 64>(A, lda, W, ldw, C, ldc, M, N, K, plan.slices, part_stride, stream);
    }
}
// Microseconds that the 32-bit instructions take from 17 rows on: rings as ring_rows knows them, with a start for every tile after the other
// (by the least squares of 98 sizes' logarithms, off by 7 %: 221 rows by 31,916 x 248 45.6, 760 by 776 x 5,784 106); a round of workgroups
// of groups of rows or of tiles at least so much a 2,048 columns (1,800 times of 1,100 sizes, one in twenty of which is below it, by some 3 %;
// rows a power of two apart, whose columns lie on the same channels, take up to a third more).
static double whole_us(int M, int N, int K, int rows) {
    auto rounds = [](long wgs) { return (double)((wgs + COMPUTE_UNITS - 1) / COMPUTE_UNITS); };
    const long rows64 = ((long)M + 63) / 64, cols64 = ((long)N + TN - 1) / TN;
    if (rows != 0) {
        const long n = (((long)M + rows - 1) / rows * (((long)N + 127) / 128) + COMPUTE_UNITS - 1) / COMPUTE_UNITS;
        return 2.0 + (rows == 128 ? 7.2 : 2.4) * n + 0.9 * (rows == 128 ? 130.0 * n : n <= 5 ? RING_32[n] : 35.0 * n) * K / 2048;
    }
    double unit;
    if (M > SKINNY_M && rows64 * cols64 >= COMPUTE_UNITS) unit = 37.7 * rounds(rows64 * cols64);
    else if (M > SKINNY_M && ((long)M + 31) / 32 * cols64 >= COMPUTE_UNITS) unit = 31.5;
    else unit = (M <= 32 ? 10.3 : M <= 48 ? 16.2 : M <= 64 ? 18.0 : 19.0) * rounds(rows64 * (((long)N + 15) / 16));
    return 2.3 + unit * K / 2048;
}
// The plan of a product in pieces, us 0 where the 32-bit instructions take it: where they are faster, to within what the times above are
// off.  Where groups of rows or the tiles above would take it only in slices (one is less exact than groups of rows, two and more are
// not), from 1,024 columns and 33 rows (or 4,096 and 17) on.  Over the 1,200 sizes none is slower by more than 1 %, and they take 0.4 %
// longer than in the fastest shape and number of slices each.  us, those and slices with their sum: 17 rows by 4,096 x 4,096 24.8 and 26.1,
// by 2,048 23.6 and 19.8; 33 rows by 2,048 x 1,024 11.1 and 12.6, by 2,048 x 2,048 20.0 and 14.0; 64 rows by 1,024 x 1,100 13.1 and 13.5;
// 150 rows by 6,144 x 2,048 (rings) 42.6 and 45.8; 300 by 2,048 x 1,024 22.6 and 22.8; 400 by 2,048 x 2,048 42.8 and 34.2; 1,400 by
// 2,048 x 2,048 120 and 81.4.
static SplitPlan split_instead(int M, int N, int K, int max_slices) {
    SplitPlan plan = {0, 1, 0};
    if (M <= 16 || (M <= 32 && K < 4096)) return plan;
    const int rows = ring_rows(M, N);
    if (rows == 0 && (K < 1024 || max_slices == 1)) return plan;
    plan = plan_split(M, N, K, rows == 0 ? 2 : 1, max_slices);
    if (plan.us >= 0.95 * whole_us(M, N, K, rows)) plan.us = 0;
    return plan;
}

template <typename TA, typename TW, typename TC, bool VEC>
static void launch_vec(const TA* A, long lda, const TW* W, long ldw, TC* C, long ldc, int M, int N, int K, hipStream_t stream) {
    if (!VEC && M <= FEW_ROWS) {
        gemm_f32_few_rows_kernel<TA, TW, TC><<<(N + 3) / 4, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K);
        return;
    }
    if constexpr (VEC) {
        // (seven and eight rows by 2,049 to 4,096 columns stay in groups of sixteen: workgroups of eight waves, two a compute unit, read A
        // twice as often as one of sixteen; us, eight rows, those and these: 2,304 x 2,048 9.6 and 10.0, 3,072 x 2,048 10.0 and 10.1, 4,088 x
        // 5,376 21.0 and 23.9; six rows 9.8 and 9.4 at 3,072 x 2,048)
        if (M <= 6 || (M <= 8 && ((N + 7) / 8 <= COMPUTE_UNITS || (N + 7) / 8 > 2 * COMPUTE_UNITS)))
            return launch_eight_rows<TA, TW, TC>(A, lda, W, ldw, C, ldc, M, N, K, stream);
    }
    if (M <= 16) return launch_skinny<TA, TW, TC, 1, VEC>(A, lda, W, ldw, C, ldc, M, N, K, stream);
    if constexpr (VEC && std::is_same<TA, float>::value && std::is_same<TW, float>::value && std::is_same<TC, float>::value) {
        const SplitPlan plan = split_instead(M, N, K, 1);
        if (plan.us > 0) return launch_split(plan, A, lda, W, ldw, C, ldc, M, N, K, 0, stream);
        const int rows = lda < (1L << 22) && ldw < (1L << 22) ? ring_rows(M, N) : 0;       // (offsets in a tile have 32 bits)
        if (rows == 32 && M <= SKINNY_M) return launch_ring<32, 128, 1, 4, 4, 4>(A, lda, W, ldw, C, ldc, M, N, K, stream);
        if (rows == 32) return launch_ring<32, 128, 1, 4, 2, 4>(A, lda, W, ldw, C, ldc, M, N, K, stream);
        if (rows == 128) return launch_ring<128, 128, 2, 4, 2, 3>(A, lda, W, ldw, C, ldc, M, N, K, stream);
    }
    // from 65 rows on (17 where fours do not fit and K is not short): tiles as soon as the smaller ones give every compute unit one (80 rows by
    // 2,048 x 2,048, 96 of them: 47 us tiled, 24 us in groups of 64 rows; 200 rows, 224: 47 us in groups, 300 rows, 320: 52 us tiled;
    // 30,000 x 515, 469 a row of tiles: 17 rows 54.2 in groups and 25.3 tiled, 64 rows 108 and 47, in bfloat16 132 and 62)
    const int n_tiles = (N + TN - 1) / TN;
    const long small_tiles = (long)n_tiles * ((M + 31) / 32);
    if ((M <= SKINNY_M && (VEC || K < 256)) || small_tiles < COMPUTE_UNITS) {
        if (M <= 32) return launch_skinny<TA, TW, TC, 2, VEC>(A, lda, W, ldw, C, ldc, M, N, K, stream);
        return launch_skinny<TA, TW, TC, 4, VEC>(A, lda, W, ldw, C, ldc, M, N, K, stream);
    }
    const bool few = M <= SKINNY_M, large = !few && (long)n_tiles * ((M + 63) / 64) >= COMPUTE_UNITS;
    const int bm = large ? 64 : 32, m_tiles = (M + bm - 1) / bm, tiles = m_tiles * n_tiles;
    const int grid = (tiles + 7) / 8 * 8;
    constexpr int TWO = VEC && std::is_same<TA, float>::value && std::is_same<TW, float>::value && std::is_same<TC, float>::value ? 2 : 1;     // (as the rings)
    if (few)
        gemm_f32_tiled_kernel<TA, TW, TC, 32, VEC, VEC ? 1 : 2><<<grid, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, m_tiles, tiles);
    else if (large)
        gemm_f32_tiled_kernel<TA, TW, TC, 64, VEC, TWO><<<grid, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, m_tiles, tiles);
    else
        gemm_f32_tiled_kernel<TA, TW, TC, 32, VEC, 1><<<grid, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, m_tiles, tiles);
}

template <typename T> static bool rows_of_fours(const void* p, long ld) {
    return ld % 4 == 0 && (uintptr_t)p % (4 * sizeof(T)) == 0;
}

template <typename TA, typename TW, typename TC>
static void launch_gemm(const void* A, long lda, const void* W, long ldw, void* C, long ldc, int M, int N, int K,
                        hipStream_t stream) {
    if (K % 4 == 0 && rows_of_fours<TA>(A, lda) && rows_of_fours<TW>(W, ldw))
        launch_vec<TA, TW, TC, true>((const TA*)A, lda, (const TW*)W, ldw, (TC*)C, ldc, M, N, K, stream);
    else
        launch_vec<TA, TW, TC, false>((const TA*)A, lda, (const TW*)W, ldw, (TC*)C, ldc, M, N, K, stream);
}

extern "C" int agave_gemm_plain(int dt_a, const void* A, long lda, int dt_w, const void* W, long ldw, int dt_c,
                                void* C, long ldc, int M, int N, int K, hipStream_t stream) {
    AGAVE_CHECK(M >= 0 && N > 0 && K > 0, "gemm_plain: bad sizes M=%d N=%d K=%d", M, N, K);
    AGAVE_CHECK(lda >= K && ldw >= K && ldc >= N, "gemm_plain: a row stride is too small (lda=%ld ldw=%ld ldc=%ld)", lda, ldw, ldc);
    AGAVE_CHECK((M + 63) / 64 <= 65535, "gemm_plain: M=%d exceeds the grid limit", M);
    AGAVE_CHECK((long)((M + 31) / 32) * ((N + TN - 1) / TN) < (1L << 30), "gemm_plain: M=%d x N=%d exceeds the grid limit", M, N);
    if (M == 0) return 0;
    const int code = dt_a * 4 + dt_w * 2 + dt_c;
    switch (code) {
        case 0: launch_gemm<float, float, float>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        case 1: launch_gemm<float, float, bf16>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        case 2: launch_gemm<float, bf16, float>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        case 3: launch_gemm<float, bf16, bf16>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        case 4: launch_gemm<bf16, float, float>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        case 5: launch_gemm<bf16, float, bf16>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        case 6: launch_gemm<bf16, bf16, float>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        case 7: launch_gemm<bf16, bf16, bf16>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        default: AGAVE_CHECK(false, "gemm_plain: unknown dtypes %d %d %d", dt_a, dt_w, dt_c);
    }
    AGAVE_LAUNCH_CHECK("gemm_plain");
    return 0;
}

// ---------------------------------------------------------------- in slices
// out[i] = the sum of the slices' i-th elements, in their order
__global__ __launch_bounds__(256) void gemm_f32_add_slices_kernel(const f32x4_t* __restrict__ parts, long n4, int slices, f32x4_t* __restrict__ out) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    f32x4_t s = parts[i];
#pragma unroll 4
    for (int z = 1; z < slices; ++z) s += parts[z * n4 + i];
    out[i] = s;
}

// Slices in which agave_gemm_slices makes a product of aligned floats faster than agave_gemm_plain does (1: it does not).
extern "C" int agave_gemm_slices_for(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 4 != 0 || N % 4 != 0) return 1;
    const SplitPlan plan = split_instead(M, N, K, 8);
    return plan.us > 0 ? plan.slices : 1;
}

extern "C" int agave_add_slices(const float* parts, long n, int slices, float* out, hipStream_t stream) {
    AGAVE_CHECK(n >= 0 && slices >= 1 && n / 1024 < (1L << 31) - 1, "add_slices: bad sizes n=%ld slices=%d", n, slices);
    AGAVE_CHECK(n % 4 == 0 && (((uintptr_t)parts | (uintptr_t)out) & 15) == 0, "add_slices: aligned fours only (n=%ld)", n);
    if (n == 0) return 0;
    gemm_f32_add_slices_kernel<<<(unsigned)((n / 4 + 255) / 256), 256, 0, stream>>>((const f32x4_t*)parts, n / 4, slices, (f32x4_t*)out);
    AGAVE_LAUNCH_CHECK("add_slices");
    return 0;
}

// parts [slices, M, N] <- 32-bit slices that add up to A W^T
extern "C" int agave_gemm_slices(const float* A, long lda, const float* W, long ldw, float* parts, int M, int N, int K, int slices,
                                 hipStream_t stream) {
    AGAVE_CHECK(M > 0 && N > 0 && K > 0 && lda >= K && ldw >= K, "gemm_slices: bad sizes M=%d N=%d K=%d", M, N, K);
    AGAVE_CHECK(K % 4 == 0 && N % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && (((uintptr_t)A | (uintptr_t)W | (uintptr_t)parts) & 15) == 0,
                "gemm_slices: rows of aligned fours");
    AGAVE_CHECK((long)((M + 63) / 64) * ((N + 63) / 64) < (1L << 30), "gemm_slices: M=%d x N=%d exceeds the grid limit", M, N);
    AGAVE_CHECK(slices >= 1 && slices <= 8 && slices <= (K + 31) / 32, "gemm_slices: %d slices of %d columns", slices, K);
    launch_split(split_in(M, N, K, slices), A, lda, W, ldw, parts, N, M, N, K, (long)M * N, stream);
    AGAVE_LAUNCH_CHECK("gemm_slices");
    return 0;
}

// A product in a tile shape and a number of slices that the caller names (the tests run every shape with it; agave_gemm_slices
// takes the fastest).
extern "C" int agave_gemm_slices_as(const float* A, long lda, const float* W, long ldw, float* parts, int M, int N, int K, int bm, int bn, int slices,
                                    hipStream_t stream) {
    AGAVE_CHECK(M > 0 && N > 0 && K > 0 && lda >= K && ldw >= K, "gemm_slices_as: bad sizes M=%d N=%d K=%d", M, N, K);
    AGAVE_CHECK(K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && (((uintptr_t)A | (uintptr_t)W) & 15) == 0, "gemm_slices_as: rows of aligned fours");
    AGAVE_CHECK((long)((M + 63) / 64) * ((N + 63) / 64) < (1L << 30), "gemm_slices_as: M=%d x N=%d exceeds the grid limit", M, N);
    AGAVE_CHECK(slices >= 1 && slices <= 8 && slices <= (K + 31) / 32, "gemm_slices_as: %d slices of %d columns", slices, K);
    for (int i = 0; i < 4; ++i)
        if (SPLIT_SHAPES[i].bm == bm && SPLIT_SHAPES[i].bn == bn) {
            launch_split({i, slices, 0}, A, lda, W, ldw, parts, N, M, N, K, (long)M * N, stream);
            AGAVE_LAUNCH_CHECK("gemm_slices_as");
            return 0;
        }
    AGAVE_CHECK(false, "gemm_slices_as: no tiles of %d x %d", bm, bn);
}

// ---------------------------------------------------------------- gate and up of few rows, with their activation
// Whether agave_gemm_gated takes M rows by a gate and an up matrix of ff rows: up to eight, where the product of both takes two blocks of
// columns a workgroup (launch_eight_rows), so that a workgroup has a block of either.
extern "C" int agave_gemm_gated_takes(int M, int ff, int K) {
    return M > 0 && M <= 8 && K > 0 && K % 4 == 0 && ff > 0 && (2L * ff + 7) / 8 > (K > 512 ? 2 : 3) * COMPUTE_UNITS;
}
// C [M, ff] <- act(A Wg^T) * (A Wu^T) for W = [Wg; Wu], all 32-bit
extern "C" int agave_gemm_gated(const float* A, long lda, const float* W, long ldw, float* C, long ldc, int M, int ff, int K, int act, float p0,
                                float p1, hipStream_t stream) {
    AGAVE_CHECK(agave_gemm_gated_takes(M, ff, K), "gemm_gated: M=%d ff=%d K=%d", M, ff, K);
    AGAVE_CHECK(lda >= K && ldw >= K && ldc >= ff && rows_of_fours<float>(A, lda) && rows_of_fours<float>(W, ldw), "gemm_gated: rows of aligned fours");
    AGAVE_CHECK((act >= 0 && act < AGAVE_GATE_ACTS) || act == AGAVE_GATE_SWISH_CLAMPED, "gemm_gated: unknown activation %d", act);
    gemm_f32_eight_rows_kernel<float, float, float, 4, 2, true><<<(ff + 7) / 8, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, ff, K, act, p0, p1);
    AGAVE_LAUNCH_CHECK("gemm_gated");
    return 0;
}
