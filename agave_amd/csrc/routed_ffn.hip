// A routed feed-forward (mixture of experts) for gfx950: the choice of experts per token and the
// experts' products over the tokens that chose them.
//
//   s = softmax(z) over all R router outputs (32-bit);  choice score c = s + correction;
//   the R outputs form `groups` equal groups of neighbours, a group's score is its largest c, only
//   the outputs of the `keep` best groups can be chosen; the `top` largest c among them are
//   chosen (the lower index wins a tie); the weight of a chosen output is s * scale.
//   Outputs e >= E are identity experts: their result is the feed-forward's input row itself.
//   Expert e < E: W_down[e] (act(W_gate[e] x) * (W_up[e] x)).
//   The other way of scoring (mode 1): the logits z + bias decide, the `top` largest are chosen, and the weights are
//   the softmax over the chosen logits alone, times scale.
//   A third way (mode 2): s = sigmoid(z), each output on its own; choice and groups as with the softmax over all.
//   `group_top` 2: a group's score is the sum of its two largest c instead of its largest.  `normalise`: the chosen
//   outputs' weights are divided by their sum + 1e-20 before the factor.
//   A shared expert, which every token runs through, may be one more expert of the products: the choice then ends every token's
//   pairs with it, weighted by the sigmoid of its gate's logit.
//   The router matrix may carry further rows behind its R outputs (`extra`): their products with the token are handed
//   out as they are (the logit of a gate on the shared expert), so that they cost no kernel of their own.
//
// A (token, slot) pair p = t * top + slot names one chosen output.  The plain kernels take the pairs
// as they come (a wave per pair and output column).  The matrix-core kernels take them sorted by
// expert, in tiles of 16, 64 or 128 pairs that never span two experts (`route_sort` makes the list and the
// tiles' table on the device, so a step's launches never depend on the choice), or, of few pairs, find an expert's from the
// choices themselves.
#include "common_impl.h"
#include "fours.h"
#include "mfma.h"
#include <math.h>

#define ROUTE_MAX 1024        // router outputs at most

// ------------------------------------------------------------------ the choice
// One thread per token; `s` [N][R] is scratch that receives the softmax.
__global__ void route_topk_kernel(const float* __restrict__ z, long ldz, const float* __restrict__ correction,
                                  float* __restrict__ s, int N, int R, int groups, int keep, int top, float scale,
                                  int* __restrict__ choice, float* __restrict__ weight) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= N) return;
    const float* zr = z + (size_t)t * ldz;
    float* sr = s + (size_t)t * R;
    float mx = -INFINITY;
    for (int e = 0; e < R; ++e) mx = fmaxf(mx, zr[e]);
    float sum = 0.f;
    for (int e = 0; e < R; ++e) {
        const float w = expf(zr[e] - mx);
        sr[e] = w;
        sum += w;
    }
    const float inv = 1.0f / sum;
    for (int e = 0; e < R; ++e) sr[e] *= inv;
    // groups that may be chosen from: a bit per group (at most 64 groups)
    const int gs = R / groups;
    unsigned long long open = ~0ull;
    if (keep < groups) {
        open = 0ull;
        for (int r = 0; r < keep; ++r) {
            int best = -1;
            float best_v = -INFINITY;
            for (int g = 0; g < groups; ++g) {
                if ((open >> g) & 1ull) continue;
                float gv = -INFINITY;
                for (int e = g * gs; e < (g + 1) * gs; ++e) gv = fmaxf(gv, sr[e] + (correction ? correction[e] : 0.f));
                if (best < 0 || gv > best_v) {
                    best = g;
                    best_v = gv;
                }
            }
            open |= 1ull << best;
        }
    }
    // the `top` best of what is open; what was chosen is marked in the scratch row's sign (s >= 0)
    for (int r = 0; r < top; ++r) {
        int best = -1;
        float best_v = -INFINITY;
        for (int e = 0; e < R; ++e) {
            const float se = sr[e];
            if (se < 0.f || !((open >> (e / gs)) & 1ull)) continue;
            const float c = se + (correction ? correction[e] : 0.f);
            if (best < 0 || c > best_v) {
                best = e;
                best_v = c;
            }
        }
        // (top <= open outputs is checked on the host, so best >= 0)
        choice[(size_t)t * top + r] = best;
        weight[(size_t)t * top + r] = sr[best] * scale;
        sr[best] = -1.0f - sr[best];
    }
}

extern "C" int agave_route_topk(const float* z, long ldz, const float* correction, float* scratch, int N, int R, int groups,
                                int keep, int top, float scale, int* choice, float* weight, hipStream_t stream) {
    AGAVE_CHECK(N >= 0 && R > 0 && R <= ROUTE_MAX, "route_topk: %d router outputs (1 to %d)", R, ROUTE_MAX);
    AGAVE_CHECK(groups > 0 && groups <= 64 && R % groups == 0, "route_topk: %d outputs in %d groups (equal groups, at most 64)", R, groups);
    AGAVE_CHECK(keep > 0 && keep <= groups, "route_topk: %d of %d groups kept", keep, groups);
    AGAVE_CHECK(top > 0 && top <= keep * (R / groups), "route_topk: %d chosen of %d that are open", top, keep * (R / groups));
    AGAVE_CHECK(z && scratch && choice && weight && ldz >= R, "route_topk: bad buffers");
    if (N == 0) return 0;
    route_topk_kernel<<<(N + 63) / 64, 64, 0, stream>>>(z, ldz, correction, scratch, N, R, groups, keep, top, scale, choice, weight);
    AGAVE_LAUNCH_CHECK("route_topk");
    return 0;
}

// ------------------------------------------------------------------ router product and choice in one kernel
// A workgroup takes RR tokens: its waves share the router's outputs (a wave per output in turn, the lanes
// along the width, a weight row read once for all of the workgroup's tokens), the logits wait in LDS, and one
// thread per token then chooses as route_topk_kernel does.  The router matrix is 32-bit; the rows may be bfloat16.
// eight neighbours along the width as floats (16 bytes of bfloat16, 32 of float)
__device__ __forceinline__ void load8(const bf16* p, float* v) {
    const uint4 u = *reinterpret_cast<const uint4*>(p);
    const uint32_t r[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(r[i] << 16);
        v[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
    }
}
__device__ __forceinline__ void load8(const float* p, float* v) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// WIDE: the width is a multiple of 8 and the rows are aligned, so a lane takes eight neighbours at a time (a
// fraction of the loads, many of them in flight); otherwise element by element.  The workgroup's waves (4, or 16
// where few tokens leave the chip idle) take the outputs in turn.
// RR tokens a workgroup: eight where there are many, one where few tokens would leave the chip idle (a wave then holds
// a whole row's share of loads in flight at once).
// OUT outputs a wave at a time: one, or two, w and w + nw, whose rows are one round trip to memory (a wave without a second
// one reads its first again).
// TILES > 0 (many tokens, RR = 16): the matrix cores' 32-bit instruction makes the product, TILES tiles of 16 outputs by the
// workgroup's 16 tokens, and plain multiply-adds up to two outputs behind them (a shared expert's gate would else cost a
// tile).  The sixteen waves take runs of 32 columns in turn, lane i + 16 g columns 8 g .. 8 g + 7 of row i of either
// operand, which is the same order for both; four running sums a tile, so that none is longer than a lane's of the other way.
// That one reads every token's row once for each output (pair) and is bound by these reads from the compute unit's cache; here a
// row is read once.  3,001 tokens of 2,048 by 17 outputs, in a prompt: 30.1 -> 13.7 us.
template <typename T, bool WIDE, int RR, int OUT, int TILES>
__global__ __launch_bounds__(1024) void route_rows_kernel(const T* __restrict__ x, long ldx, const float* __restrict__ router,
                                                          const float* __restrict__ correction, int N, int K, int R, int groups,
                                                          int keep, int top, float scale, int* __restrict__ choice,
                                                          float* __restrict__ weight, int mode, int extra,
                                                          float* __restrict__ extra_out, int group_top, int normalise, int stride,
                                                          int shared_at) {
    extern __shared__ float zs[];                      // [RR][R + extra], then the corrections [R]
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int Rt = R + extra;
    float* corr = zs + RR * Rt;                // (read many times by the one thread that chooses: from LDS, not memory)
    for (int e = threadIdx.x; e < R; e += blockDim.x) corr[e] = correction ? correction[e] : 0.f;
    const int t0 = blockIdx.x * RR;
    const int rows = min(RR, N - t0);
    if constexpr (TILES > 0) {
        constexpr int NW = 16, REST = 2;
        float* part = corr + R;                // [NW][RR][Rt]
        const int i = lane & 15, g = lane >> 4, tiled = min(Rt, 16 * TILES), rest = Rt - tiled;
        const T* xr = x + (size_t)(t0 + min(i, rows - 1)) * ldx + 8 * g;
        const float* wt[TILES];
#pragma unroll
        for (int j = 0; j < TILES; ++j) wt[j] = router + (size_t)min(16 * j + i, Rt - 1) * K + 8 * g;     // (outputs past the end: never stored)
        const float* wr[REST];
#pragma unroll
        for (int j = 0; j < REST; ++j) wr[j] = router + (size_t)min(tiled + j, Rt - 1) * K + 8 * g;
        f32x4_t acc[TILES][4] = {};
        float more[REST][2] = {};
#pragma unroll(TILES == 1 ? 4 : TILES == 2 ? 2 : 1)
        for (int k = 32 * w; k < K; k += 32 * NW) {
            float xv[8], wv[TILES][8], rv[REST][8];
            load8(xr + k, xv);
#pragma unroll
            for (int j = 0; j < TILES; ++j) load8(wt[j] + k, wv[j]);
#pragma unroll
            for (int j = 0; j < REST; ++j)
                if (j < rest) load8(wr[j] + k, rv[j]);
#pragma unroll
            for (int m = 0; m < 8; ++m) {
#pragma unroll
                for (int j = 0; j < TILES; ++j) acc[j][m & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[m], wv[j][m], acc[j][m & 3], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < REST; ++j)
                    if (j < rest) more[j][m & 1] = fmaf(xv[m], rv[j][m], more[j][m & 1]);
            }
        }
        // a tile: lane holds tokens 4 g + e of output 16 j + i; the rest: lane holds a fourth of token i's sum
        float* mine = part + w * RR * Rt;
#pragma unroll
        for (int j = 0; j < TILES; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (16 * j + i < tiled) mine[(4 * g + e) * Rt + 16 * j + i] = (acc[j][0][e] + acc[j][1][e]) + (acc[j][2][e] + acc[j][3][e]);
#pragma unroll
        for (int j = 0; j < REST; ++j)
            if (j < rest) {
                float sum = more[j][0] + more[j][1];
                sum += __shfl_xor(sum, 16);
                sum += __shfl_xor(sum, 32);
                if (g == 0) mine[i * Rt + tiled + j] = sum;
            }
        __syncthreads();
        for (int at = threadIdx.x; at < RR * Rt; at += 64 * NW) {
            float sum[NW];
#pragma unroll
            for (int o = 0; o < NW; ++o) sum[o] = part[o * RR * Rt + at];
#pragma unroll
            for (int half = NW / 2; half > 0; half /= 2)
#pragma unroll
                for (int o = 0; o < half; ++o) sum[o] += sum[o + half];
            zs[at] = sum[0];
        }
    }
    for (int r = w; TILES == 0 && r < Rt; r += OUT * nw) {
        const bool second = OUT == 2 && r + nw < Rt;
        const float* wr = router + (size_t)r * K;
        const float* wr2 = second ? wr + (size_t)nw * K : wr;
        float acc[RR], acc2[RR];
#pragma unroll
        for (int i = 0; i < RR; ++i) acc[i] = acc2[i] = 0.f;
        if (WIDE) {
#pragma unroll(RR == 1 ? 4 : 3 - OUT)
            for (int k = 8 * lane; k < K; k += 512) {
                float wk[8], wk2[8] = {};
                load8(wr + k, wk);
                if (OUT == 2) load8(wr2 + k, wk2);
#pragma unroll
                for (int i = 0; i < RR; ++i) {
                    const int t = t0 + (i < rows ? i : 0);
                    float xv[8];
                    load8(x + (size_t)t * ldx + k, xv);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        acc[i] = fmaf(xv[j], wk[j], acc[i]);
                        if (OUT == 2) acc2[i] = fmaf(xv[j], wk2[j], acc2[i]);
                    }
                }
            }
        } else {
            for (int k = lane; k < K; k += 64) {
                const float wk = wr[k], wk2 = OUT == 2 ? wr2[k] : 0.f;
#pragma unroll
                for (int i = 0; i < RR; ++i) {
                    const int t = t0 + (i < rows ? i : 0);
                    const float xv = ld(x + (size_t)t * ldx + k);
                    acc[i] = fmaf(xv, wk, acc[i]);
                    if (OUT == 2) acc2[i] = fmaf(xv, wk2, acc2[i]);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < RR; ++i) {
            const float sum = wave_sum(acc[i]), sum2 = OUT == 2 ? wave_sum(acc2[i]) : 0.f;
            if (lane == 0) {
                zs[i * Rt + r] = sum;
                if (second) zs[i * Rt + r + nw] = sum2;
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; extra_out && i < rows * extra; i += blockDim.x)
        extra_out[(size_t)(t0 + i / extra) * extra + i % extra] = zs[(i / extra) * Rt + R + i % extra];
    // the choice: a wave per token, the lanes along the outputs
    const int gs = R / groups;
    for (int i = w; i < rows; i += nw) {
        float* sr = zs + (size_t)i * Rt;
        const int t = t0 + i;
        if (shared_at >= 0 && lane == 0) {          // the shared expert: every token's last pair, weighted by its gate
            choice[(size_t)t * stride + top] = shared_at;
            weight[(size_t)t * stride + top] = extra ? 1.0f / (1.0f + expf(-sr[R])) : 1.0f;
        }
        if (mode == 1 && R <= 64 && R <= 6 * top) {
            // An output a lane, its place among all counted at once, R turns; the loop below is `top` chains of two maxima over the lanes.
            // us, the loop and so, 6 tokens of 2,048: 17 outputs 2 chosen 5.7 and 5.9, 4 6.3 and 6.0, 8 7.6 and 6.0; 32 4 7.2 and 7.5, 8 8.5 and
            // 7.6; 64 4 10.2 and 11.7, 8 11.6 and 11.7.  Logits that are not finite keep that loop's order.
            const float z = lane < R ? sr[lane] + corr[lane] : 0.f;
            if (!__any(!(fabsf(z) < INFINITY))) {
                int place = 0;
                for (int f = 0; f < R; ++f) {
                    const float zf = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(z), f));
                    place += (zf > z || (zf == z && f < lane)) ? 1 : 0;
                }
                const bool chosen = lane < R && place < top;
                __builtin_amdgcn_wave_barrier();
                if (chosen) sr[place] = z;
                __builtin_amdgcn_wave_barrier();
                const float first_v = sr[0];
                float sum = 0.f;
                for (int r = 0; r < top; ++r) sum += expf(sr[r] - first_v);
                if (chosen) {
                    choice[(size_t)t * stride + place] = lane;
                    weight[(size_t)t * stride + place] = expf(z - first_v) / sum * scale;
                }
                continue;
            }
        }
        if (mode == 1) {
            // the largest logits (bias added) are chosen, the lower index among equals; a chosen place is marked by
            // -infinity; lane r keeps round r's logit, and the weights are the softmax over those (top <= 64)
            for (int e = lane; e < R; e += 64) sr[e] += corr[e];
            __builtin_amdgcn_wave_barrier();
            int my_choice = 0;
            float my_logit = 0.f, first_v = 0.f, sum = 0.f;
            for (int r = 0; r < top; ++r) {
                float best_v = -INFINITY;
                int best = -1;
                for (int e = lane; e < R; e += 64) {
                    const float se = sr[e];
                    if (se == -INFINITY) continue;
                    if (best < 0 || se > best_v) {
                        best = e;
                        best_v = se;
                    }
                }
                const float top_v = wave_max(best >= 0 ? best_v : -INFINITY);
                int chosen = (int)(-wave_max((best >= 0 && best_v == top_v) ? -(float)best : -INFINITY));
                if (chosen < 0 || chosen >= R) chosen = 0;          // (every open logit is -infinity or not a number)
                if (r == 0) first_v = top_v;
                sum += expf(top_v - first_v);
                if (r == lane) {
                    my_choice = chosen;
                    my_logit = top_v;
                }
                if (lane == 0) sr[chosen] = -INFINITY;
                __builtin_amdgcn_wave_barrier();
            }
            if (lane < top) {
                choice[(size_t)t * stride + lane] = my_choice;
                weight[(size_t)t * stride + lane] = expf(my_logit - first_v) / sum * scale;
            }
            continue;
        }
        if (mode == 2) {
            for (int e = lane; e < R; e += 64) sr[e] = 1.0f / (1.0f + expf(-sr[e]));
        } else {
            float mx = -INFINITY;
            for (int e = lane; e < R; e += 64) mx = fmaxf(mx, sr[e]);
            mx = wave_max(mx);
            float sum = 0.f;
            for (int e = lane; e < R; e += 64) {
                const float v = expf(sr[e] - mx);
                sr[e] = v;
                sum += v;
            }
            const float inv = 1.0f / wave_sum(sum);
            for (int e = lane; e < R; e += 64) sr[e] *= inv;
        }
        __builtin_amdgcn_wave_barrier();
        // the groups that stay open: lane g holds group g's score (at most 64 groups)
        unsigned long long open = ~0ull;
        if (keep < groups) {
            float gv = -INFINITY;
            if (lane < groups) {
                float second = -INFINITY;
                for (int e = lane * gs; e < (lane + 1) * gs; ++e) {
                    const float c = sr[e] + corr[e];
                    if (c > gv) {
                        second = gv;
                        gv = c;
                    } else {
                        second = fmaxf(second, c);
                    }
                }
                if (group_top == 2 && gs > 1) gv += second;
            }
            open = 0ull;
            for (int r = 0; r < keep; ++r) {
                const float cand = (lane < groups && !((open >> lane) & 1ull)) ? gv : -INFINITY;
                const float best_v = wave_max(cand);
                // the lowest group among equals
                const float first = wave_max((lane < groups && !((open >> lane) & 1ull) && cand == best_v) ? -(float)lane : -INFINITY);
                open |= 1ull << (int)(-first);
            }
        }
        // the `top` best of what is open; what was chosen is marked in the row's sign (s >= 0)
        int my_choice = 0;
        float my_weight = 0.f, chosen_sum = 0.f;
        for (int r = 0; r < top; ++r) {
            float best_v = -INFINITY;
            int best = -1;
            for (int e = lane; e < R; e += 64) {
                const float se = sr[e];
                if (se < 0.f || !((open >> (e / gs)) & 1ull)) continue;
                const float c = se + corr[e];
                if (best < 0 || c > best_v) {          // (a lane's outputs come in rising order: the first of equals stays)
                    best = e;
                    best_v = c;
                }
            }
            const float top_v = wave_max(best >= 0 ? best_v : -INFINITY);
            const int chosen = (int)(-wave_max((best >= 0 && best_v == top_v) ? -(float)best : -INFINITY));
            // (top <= open outputs is checked on the host, so some lane has a candidate)
            const float s_chosen = sr[chosen];
            chosen_sum += s_chosen;
            if ((r & 63) == lane) {             // lane r keeps round r's result; the results leave in one store at the end
                my_choice = chosen;
                my_weight = s_chosen * scale;
            }
            if (lane == 0) sr[chosen] = -1.0f - s_chosen;
            // (a wave's LDS accesses happen in the order they were issued: the next round's reads see this write)
            __builtin_amdgcn_wave_barrier();
            if ((r & 63) == 63 || r == top - 1) {
                const int at = (r & ~63) + lane;
                if (at <= r) {
                    choice[(size_t)t * stride + at] = my_choice;
                    weight[(size_t)t * stride + at] = normalise ? my_weight / (chosen_sum + 1e-20f) : my_weight;      // (normalise: top <= 64, one batch)
                }
            }
        }
    }
}

extern "C" int agave_route_rows(int dtype, const void* x, long ldx, const float* router, const float* correction, int N, int K,
                                int R, int groups, int keep, int top, float scale, int* choice, float* weight, int mode,
                                int extra, float* extra_out, int group_top, int normalise, int stride, int shared_at, hipStream_t stream) {
    AGAVE_CHECK(stride >= top + (shared_at >= 0 ? 1 : 0) && (shared_at < 0 || extra <= 1), "route_rows: rows of %d pairs do not hold %d chosen and the shared expert, which has one gate at most", stride, top);
    AGAVE_CHECK(mode == 0 || mode == 2 || (mode == 1 && top <= 64 && groups == 1), "route_rows: the softmax over the chosen logits takes at most 64 of them and no groups");
    AGAVE_CHECK((group_top == 1 || group_top == 2) && (!normalise || (top <= 64 && mode != 1)), "route_rows: a group counts by its largest or its two largest; weights are divided by their sum for at most 64 chosen");
    AGAVE_CHECK(extra >= 0 && extra <= 64 && (extra == 0 || extra_out || shared_at >= 0), "route_rows: %d further rows of the router (0 to 64, with a place for their products)", extra);
    AGAVE_CHECK(N >= 0 && K > 0 && R > 0 && R <= ROUTE_MAX, "route_rows: %d router outputs (1 to %d)", R, ROUTE_MAX);
    AGAVE_CHECK(groups > 0 && groups <= 64 && R % groups == 0, "route_rows: %d outputs in %d groups (equal groups, at most 64)", R, groups);
    AGAVE_CHECK(keep > 0 && keep <= groups, "route_rows: %d of %d groups kept", keep, groups);
    AGAVE_CHECK(top > 0 && top <= keep * (R / groups), "route_rows: %d chosen of %d that are open", top, keep * (R / groups));
    AGAVE_CHECK(x && router && choice && weight && ldx >= K, "route_rows: bad buffers");
    if (N == 0) return 0;
    const bool wide = K % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x % 32) == 0 && ((uintptr_t)router % 32) == 0;
    AGAVE_CHECK(dtype == AGAVE_F32 || dtype == AGAVE_BF16, "route_rows: unknown dtype %d", dtype);
    const bool f32 = dtype == AGAVE_F32;
    // Many tokens, more than a few outputs and whole runs of 32 columns: tiles of 16 outputs on the matrix cores, a last tile of one
    // or two left to plain multiply-adds.  From 2,049 tokens on, where eight a workgroup are more than one round of
    // workgroups.  us, the other way and this, bfloat16 rows of 2,048: 17 outputs 2,000 tokens 13.6 and 13.3, 3,001 22.4 and 13.3, 12,000
    // 51.9 and 35.4; 32 outputs 13.5 and 16.2, 22.4 and 16.4, 66.7 and 45.4; 49 outputs 21.6 and 21.6, 37.5 and 22.1, 105 and 63;
    // 8 outputs 12,000 tokens 27.5 and 27.6, rows of 512 17.5 and 18.2.
    const int outputs_all = R + extra, tiles = outputs_all < 16 || outputs_all % 16 > 2 ? (outputs_all + 15) / 16 : outputs_all / 16;
    if (wide && K % 32 == 0 && N > 2048 && outputs_all > 8 && tiles <= 3) {
        const size_t lds_tiles = ((size_t)17 * 16 * outputs_all + R) * sizeof(float);
#define ROUTE_TILES(T_, TILES_) route_rows_kernel<T_, true, 16, 1, TILES_><<<(N + 15) / 16, 1024, lds_tiles, stream>>>((const T_*)x, ldx, router, correction, \
        N, K, R, groups, keep, top, scale, choice, weight, mode, extra, extra_out, group_top, normalise, stride, shared_at)
        if (f32) { if (tiles == 1) ROUTE_TILES(float, 1); else if (tiles == 2) ROUTE_TILES(float, 2); else ROUTE_TILES(float, 3); }
        else if (tiles == 1) ROUTE_TILES(bf16, 1); else if (tiles == 2) ROUTE_TILES(bf16, 2); else ROUTE_TILES(bf16, 3);
#undef ROUTE_TILES
        AGAVE_LAUNCH_CHECK("route_rows");
        return 0;
    }
    const int rows = N <= 64 ? 1 : 8, blocks = (N + rows - 1) / rows;
    const int threads = blocks <= 512 ? 1024 : 256;            // (more waves to share the outputs while they all fit the chip at once)
    const size_t lds = (size_t)(rows * (R + extra) + R) * sizeof(float);
    // Two outputs a wave at a time where there are more than one for each wave.  With a token a workgroup not where the last two
    // turns would be one for most waves, and of one or two tokens only where they are little more than one turn: a wave's second
    // row is then work for nothing, or more than one compute unit takes from memory at once.  us, one and two, routers from memory, rows
    // of 2,048: 16 outputs, 6 tokens 5.2 and 6.1, 3,001 tokens 18.6 and 22.0; 17 outputs 6.5 and 6.1, 26.3 and 22.2; 32 outputs, one
    // token 8.7 and 9.0, 64 tokens 8.5 and 8.1; 48 outputs, 6 tokens 11.1 and 11.9, 3,001 tokens 41.1 and 37.6; 128 outputs, one
    // token 24.3 and 25.1, 12 tokens 22.8 and 21.1.
    const int waves = threads / 64, outputs = R + extra, last = outputs % (2 * waves);
    const bool two = outputs > waves && (rows == 8 || (N > 2 ? last == 0 || last <= waves / 2 || last > waves : last > waves && last <= waves * 3 / 2));
#define ROUTE_GO(T_, W_, RR_, OUT_) route_rows_kernel<T_, W_, RR_, OUT_, 0><<<blocks, threads, lds, stream>>>((const T_*)x, ldx, router, correction, N, K, R, groups, \
        keep, top, scale, choice, weight, mode, extra, extra_out, group_top, normalise, stride, shared_at)
#define ROUTE_ROWS(T_, W_) do { if (rows == 1 && two) ROUTE_GO(T_, W_, 1, 2); else if (rows == 1) ROUTE_GO(T_, W_, 1, 1); \
        else if (two) ROUTE_GO(T_, W_, 8, 2); else ROUTE_GO(T_, W_, 8, 1); } while (0)
    if (f32 && wide) ROUTE_ROWS(float, true); else if (f32) ROUTE_ROWS(float, false); else if (wide) ROUTE_ROWS(bf16, true); else ROUTE_ROWS(bf16, false);
#undef ROUTE_ROWS
#undef ROUTE_GO
    AGAVE_LAUNCH_CHECK("route_rows");
    return 0;
}

// ------------------------------------------------------------------ activations of the experts' gates
// Of the products' 32-bit sums: nothing is rounded before the result, the inner row, which is what the down product reads.
// act(gate) * up for activations 0 to 3; 6 ("swish_clamped"): g = min(gate, p0), u = clamp(up, -p0, p0),
// g sigmoid(p1 g) (u + 1)
__device__ __forceinline__ float expert_act(float x, int act);
__device__ __forceinline__ float expert_gated(float gate, float up, int act, float p0, float p1) {
    if (act == 6) {
        const float g = fminf(gate, p0), u = fminf(fmaxf(up, -p0), p0);
        return g / (1.0f + expf(-p1 * g)) * (u + 1.0f);
    }
    return expert_act(gate, act) * up;
}
__device__ __forceinline__ float expert_act(float x, int act) {
    switch (act) {
        case 0: { const float c = 0.7978845608028654f; return 0.5f * x * (1.0f + tanhf(c * (x + 0.044715f * x * x * x))); }
        case 1: return x / (1.0f + expf(-x));
        case 2: return 0.5f * x * (1.0f + erff(x * 0.7071067811865476f));
        default: return x > 0.f ? x : 0.f;
    }
}

// ------------------------------------------------------------------ plain products, pair by pair
// act[p][f] = act(W_gate[e] x_t . f) * (W_up[e] x_t . f): a wave per (pair, f), lanes along K
template <typename T>
__global__ __launch_bounds__(256) void routed_gate_up_plain_kernel(const T* __restrict__ x, long ldx, const int* __restrict__ choice,
                                                                   const T* __restrict__ wg, const T* __restrict__ wu,
                                                                   T* __restrict__ act_out, int top, int E, int ff, int K, int act,
                                                                   float p0, float p1) {
    const int p = blockIdx.x;
    const int e = choice[p];
    if (e < 0 || e >= E) return;
    const int lane = threadIdx.x & 63;
    const int f = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (f >= ff) return;
    const T* xr = x + (size_t)(p / top) * ldx;
    const T* g = wg + ((size_t)e * ff + f) * K;
    const T* u = wu + ((size_t)e * ff + f) * K;
    float ag = 0.f, au = 0.f;
    for (int k = lane; k < K; k += 64) {
        const float xv = ld(xr + k);
        ag = fmaf(xv, ld(g + k), ag);
        au = fmaf(xv, ld(u + k), au);
    }
    ag = wave_sum(ag);
    au = wave_sum(au);
    if (lane == 0) st(act_out + (size_t)p * ff + f, expert_gated(ag, au, act, p0, p1));
}

// y[p][c] = W_down[e][c] . act[p]: a wave per (pair, c), lanes along ff; y is 32-bit
template <typename T>
__global__ __launch_bounds__(256) void routed_down_plain_kernel(const T* __restrict__ act_in, const int* __restrict__ choice,
                                                                const T* __restrict__ wd, float* __restrict__ y, int E, int ff,
                                                                int hidden) {
    const int p = blockIdx.x;
    const int e = choice[p];
    if (e < 0 || e >= E) return;
    const int lane = threadIdx.x & 63;
    const int c = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (c >= hidden) return;
    const T* a = act_in + (size_t)p * ff;
    const T* w = wd + ((size_t)e * hidden + c) * ff;
    float acc = 0.f;
    for (int f = lane; f < ff; f += 64) acc = fmaf(ld(a + f), ld(w + f), acc);
    acc = wave_sum(acc);
    if (lane == 0) y[(size_t)p * hidden + c] = acc;
}

// out[t] = sum over the token's pairs of weight * (expert row, or the input row for an identity expert) + shared[t].
// `place` (may be null): where pair p's row lies in y (a sorted list); null: at p.
// A thread makes V neighbours of a row: 4 in steps of many tokens where rows and sizes allow accesses of four elements (bound by
// memory: 3,001 tokens of 4 pairs and 2,048 columns, 135 MB, 21.6 us; one element a thread 35.8), 1 otherwise.
template <typename T, int V>
__global__ void routed_combine_kernel(const float* __restrict__ y, const int* __restrict__ place, const int* __restrict__ choice,
                                      const float* __restrict__ weight, const T* __restrict__ x, long ldx,
                                      const T* __restrict__ shared, long lds, const float* __restrict__ shared_gate,
                                      T* __restrict__ out, long ldo, int N, int top, int E, int hidden) {
    const long idx = ((long)blockIdx.x * blockDim.x + threadIdx.x) * V;
    if (idx >= (long)N * hidden) return;
    const int t = (int)(idx / hidden), c = (int)(idx % hidden);
    // (no load under a per-lane condition: the input row's element is read once, an expert row's from a row that exists
    // whatever the choice, and what does not count is left out afterwards)
    float xv[V], sv[V], acc[V];
    load_near<V>(x + (size_t)t * ldx + c, xv);
    load_near<V>((shared ? shared : x) + (size_t)t * (shared ? lds : ldx) + c, sv);
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = 0.f;
#pragma unroll 4
    for (int r = 0; r < top; ++r) {
        const int p = t * top + r;
        const int e = choice[p];
        const float w = weight[p];
        const bool expert = e >= 0 && e < E;
        int row = place ? place[p] : p;
        row = (expert && row >= 0) ? row : 0;
        float yv[V] = {};
        if (y) load_near<V>(y + (size_t)row * hidden + c, yv);
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] = fmaf(w, e >= E ? xv[i] : (expert ? yv[i] : 0.f), acc[i]);
    }
    // (the shared expert's row, times the sigmoid of a logit per token where it has a gate)
#pragma unroll
    for (int i = 0; i < V; ++i)
        if (shared) acc[i] = shared_gate ? fmaf(1.0f / (1.0f + expf(-shared_gate[t])), sv[i], acc[i]) : acc[i] + sv[i];
    store_near<V>(out + (size_t)t * ldo + c, acc);
}

extern "C" int agave_routed_experts_plain(int dtype, const void* x, long ldx, const int* choice, const void* wg, const void* wu,
                                          const void* wd, void* act_rows, float* y, int N, int top, int E, int ff, int hidden,
                                          int act, float p0, float p1, hipStream_t stream) {
    AGAVE_CHECK(N >= 0 && top > 0 && E >= 0 && ff > 0 && hidden > 0, "routed_experts: bad sizes");
    AGAVE_CHECK((act >= 0 && act < 4) || act == 6, "routed_experts: unknown activation %d", act);
    AGAVE_CHECK(x && choice && act_rows && y && ldx >= hidden && (E == 0 || (wg && wu && wd)), "routed_experts: bad buffers");
    AGAVE_CHECK((ff + 3) / 4 <= 65535 && (hidden + 3) / 4 <= 65535, "routed_experts: too many columns for the grid");
    if (N == 0 || E == 0) return 0;
    const dim3 g1(N * top, (ff + 3) / 4), g2(N * top, (hidden + 3) / 4);
    if (dtype == AGAVE_F32) {
        routed_gate_up_plain_kernel<float><<<g1, 256, 0, stream>>>((const float*)x, ldx, choice, (const float*)wg, (const float*)wu,
                                                                   (float*)act_rows, top, E, ff, hidden, act, p0, p1);
        routed_down_plain_kernel<float><<<g2, 256, 0, stream>>>((const float*)act_rows, choice, (const float*)wd, y, E, ff, hidden);
    } else if (dtype == AGAVE_BF16) {
        routed_gate_up_plain_kernel<bf16><<<g1, 256, 0, stream>>>((const bf16*)x, ldx, choice, (const bf16*)wg, (const bf16*)wu,
                                                                  (bf16*)act_rows, top, E, ff, hidden, act, p0, p1);
        routed_down_plain_kernel<bf16><<<g2, 256, 0, stream>>>((const bf16*)act_rows, choice, (const bf16*)wd, y, E, ff, hidden);
    } else
        AGAVE_CHECK(false, "routed_experts: unknown dtype %d", dtype);
    AGAVE_LAUNCH_CHECK("routed_experts_plain");
    return 0;
}

extern "C" int agave_routed_combine(int dtype, const float* y, const int* place, const int* choice, const float* weight,
                                    const void* x, long ldx, const void* shared, long lds, const float* shared_gate, void* out,
                                    long ldo, int N, int top, int E, int hidden, hipStream_t stream) {
    AGAVE_CHECK(N >= 0 && top > 0 && hidden > 0, "routed_combine: bad sizes");
    AGAVE_CHECK(choice && weight && x && out && (E == 0 || y) && ldx >= hidden && ldo >= hidden && (!shared || lds >= hidden),
                "routed_combine: bad buffers");
    if (N == 0) return 0;
    AGAVE_CHECK(dtype == AGAVE_F32 || dtype == AGAVE_BF16, "routed_combine: unknown dtype %d", dtype);
    const uintptr_t wide = 4 * (dtype == AGAVE_F32 ? 4 : 2);           // bytes of four neighbours in a row
    // (Few elements leave most of the chip without a thread when each takes four.  us, 1 and 4, bfloat16, 2,048 columns of 4 pairs: 6
    // tokens 2.8 and 3.1, 64 3.0 and 3.2, 100 3.24 and 3.16, 300 4.8 and 3.5; 4,096 columns of 2 pairs, 32 2.84 and 2.96, 48 2.95 and 2.89.)
    const bool fours = (long)N * hidden >= 3 << 16 && hidden % 4 == 0 && ldx % 4 == 0 && ldo % 4 == 0 && (!shared || lds % 4 == 0) && (uintptr_t)x % wide == 0 &&
                       (uintptr_t)out % wide == 0 && (uintptr_t)shared % wide == 0 && (uintptr_t)y % 16 == 0;
    const long blocks = ((long)N * hidden / (fours ? 4 : 1) + 255) / 256;
#define COMBINE_GO(T_, V_) routed_combine_kernel<T_, V_><<<(unsigned)blocks, 256, 0, stream>>>(y, place, choice, weight, (const T_*)x, ldx, \
        (const T_*)shared, lds, shared_gate, (T_*)out, ldo, N, top, E, hidden)
    if (dtype == AGAVE_F32) {
        if (fours) COMBINE_GO(float, 4); else COMBINE_GO(float, 1);
    } else {
        if (fours) COMBINE_GO(bf16, 4); else COMBINE_GO(bf16, 1);
    }
#undef COMBINE_GO
    AGAVE_LAUNCH_CHECK("routed_combine");
    return 0;
}

// ------------------------------------------------------------------ the pairs' sum, straight into the residual stream
// b = sum over the token's pairs of weight * expert row + shared row (as routed_combine_kernel, no identity experts);
// h[t] += post_gain ? rmsnorm(b) * post_gain : b;  out[t] = pre_gain ? rmsnorm(h[t]) * pre_gain : h[t].
// A workgroup a token, its row in registers; everything is asked for before anything is used, the pairs' rows PB at a time.  As a
// row of its own the sum cost a kernel, its write and its read.
// Bound by memory with many tokens, by its round trips with few.  us, the two kernels and this one, 2,048 columns, 5 pairs a token: 6 tokens
// 5.8 and 4.0, 300 9.6 and 6.0, 3,001 50.3 and 37.0 (185 MB); 4,096 columns of 2 pairs, 64 6.4 and 4.4, 2,000 44.3 and 27.8.
template <typename T, int VPT, int PB>
__global__ void routed_norm_kernel(float* __restrict__ h, const float* __restrict__ y, const int* __restrict__ place, const int* __restrict__ choice,
                                   const float* __restrict__ weight, int top, int E, const T* __restrict__ shared, long lds,
                                   const float* __restrict__ shared_gate, const float* __restrict__ post_gain, float post_eps, T* __restrict__ out,
                                   long ldo, const float* __restrict__ pre_gain, float pre_eps, int e) {
    __shared__ float red[2][16];
    const int t = blockIdx.x;
    float* hr = h + (size_t)t * e;
    f32x4_t hv[VPT], g1[VPT], g2[VPT], b[VPT] = {}, yv[PB][VPT];
    float sv[VPT][4];
    int col[VPT];
    bool in[VPT];
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
        const int c = (threadIdx.x + v * blockDim.x) * 4;
        in[v] = c < e;
        col[v] = in[v] ? c : 0;                              // (a lane past the row's end reads its start and uses nothing of it)
        hv[v] = *reinterpret_cast<const f32x4_t*>(hr + col[v]);
        g1[v] = *reinterpret_cast<const f32x4_t*>((post_gain ? post_gain : hr) + col[v]);       // (a gain that is not there: the row, not used)
        g2[v] = *reinterpret_cast<const f32x4_t*>((pre_gain ? pre_gain : hr) + col[v]);
        if (shared) load_near<4>(shared + (size_t)t * lds + col[v], sv[v]);
    }
    for (int r0 = 0; r0 < top; r0 += PB) {
        float w[PB];
        bool live[PB];
#pragma unroll
        for (int u = 0; u < PB; ++u) {                       // (a pair past the last: the last one again, not added)
            const int p = t * top + min(r0 + u, top - 1), ex = choice[p];
            live[u] = ex >= 0 && ex < E && r0 + u < top;
            int row = place ? place[p] : p;
            row = live[u] && row >= 0 ? row : 0;
            w[u] = weight[p];
#pragma unroll
            for (int v = 0; v < VPT; ++v) yv[u][v] = *reinterpret_cast<const f32x4_t*>(y + (size_t)row * e + col[v]);
        }
#pragma unroll
        for (int u = 0; u < PB; ++u)
#pragma unroll
            for (int v = 0; v < VPT; ++v)
#pragma unroll
                for (int i = 0; i < 4; ++i) b[v][i] = live[u] ? fmaf(w[u], yv[u][v][i], b[v][i]) : b[v][i];
    }
    if (shared) {
        const float sg = shared_gate ? 1.0f / (1.0f + expf(-shared_gate[t])) : 1.0f;
#pragma unroll
        for (int v = 0; v < VPT; ++v)
#pragma unroll
            for (int i = 0; i < 4; ++i) b[v][i] = fmaf(sg, sv[v][i], b[v][i]);
    }
    // (rounded as the row that routed_combine leaves: whether a step takes that kernel and the norm's or this one shows in the order
    // of the norms' sums only)
#pragma unroll
    for (int v = 0; v < VPT; ++v)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            T rounded;
            st(&rounded, b[v][i]);
            b[v][i] = ld(&rounded);
        }
    auto squares = [&](const f32x4_t& x) { return x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3]; };
    if (post_gain) {
        float ss = 0.f;
#pragma unroll
        for (int v = 0; v < VPT; ++v) ss += in[v] ? squares(b[v]) : 0.f;
        const float inv = 1.0f / sqrtf(block_sum(ss, red[0]) / (float)e + post_eps);
#pragma unroll
        for (int v = 0; v < VPT; ++v) b[v] = b[v] * inv * g1[v];
    }
    float ss = 0.f;
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
        hv[v] += b[v];
        if (in[v]) {
            *reinterpret_cast<f32x4_t*>(hr + col[v]) = hv[v];
            ss += squares(hv[v]);
        }
    }
    float inv = 1.0f;
    if (pre_gain) inv = 1.0f / sqrtf(block_sum(ss, red[1]) / (float)e + pre_eps);
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = pre_gain ? hv[v][i] * inv * g2[v][i] : hv[v][i];
        if (in[v]) store_near<4>(out + (size_t)t * ldo + col[v], o);
    }
}

extern "C" int agave_routed_norm(int dtype, float* h, const float* y, const int* place, const int* choice, const float* weight, int top, int E,
                                 const void* shared, long lds, const float* shared_gate, const float* post_gain, float post_eps, void* out, long ldo,
                                 const float* pre_gain, float pre_eps, int N, int e, hipStream_t stream) {
    AGAVE_CHECK(N >= 0 && top > 0 && E > 0 && e > 0 && e % 4 == 0 && e <= 16384, "routed_norm: bad sizes N=%d top=%d E=%d e=%d", N, top, E, e);
    AGAVE_CHECK(h && y && choice && weight && out && ldo >= e && ldo % 4 == 0 && (!shared || (lds >= e && lds % 4 == 0)), "routed_norm: bad buffers");
    AGAVE_CHECK((((uintptr_t)h | (uintptr_t)y | (uintptr_t)shared | (uintptr_t)post_gain | (uintptr_t)out | (uintptr_t)pre_gain) & 15) == 0,
                "routed_norm: rows must be aligned to 16 bytes");
    AGAVE_CHECK(dtype == AGAVE_F32 || dtype == AGAVE_BF16, "routed_norm: unknown dtype %d", dtype);
    if (N == 0) return 0;
    // threads as residual_norm takes them: one float4 each in steps of few tokens, two (four) in steps of many.  More than eight pairs
    // of more than 2,048 columns go in twos with few tokens, too: two batches of eight float4 and 1,024 threads wait for one another
    // (4,096 columns of nine pairs, 64 tokens 6.9 us, so 4.8; a kernel for the sum and one for the norm 7.3).  In twos five
    // pairs a batch are as fast as eight for six to eight pairs but for 0.4 to 0.6 us of few tokens, and faster from some 300 tokens
    // on (5,120 columns of eight, 800 tokens 31.0 and 33.4) and for five, nine and ten pairs.
    int threads;
    if (e <= 1024 || (N <= 64 && e <= (top > 8 ? 2048 : 4096))) threads = 64 * ((e / 4 + 63) / 64);
    else {
        const int per = e / 4 <= 2048 ? 2 : 4;
        threads = 64 * ((e / 4 + per * 64 - 1) / (per * 64));
    }
    const int vpt = (e / 4 + threads - 1) / threads;
#define NORM_GO(T_, V_, P_) routed_norm_kernel<T_, V_, P_><<<N, threads, 0, stream>>>(h, y, place, choice, weight, top, E, (const T_*)shared, lds, shared_gate, \
        post_gain, post_eps, (T_*)out, ldo, pre_gain, pre_eps, e)
#define NORM_T(T_) do { if (vpt <= 1) { if (top > 4) NORM_GO(T_, 1, 8); else NORM_GO(T_, 1, 4); } else if (vpt <= 2) { if (top > 4) NORM_GO(T_, 2, 5); else NORM_GO(T_, 2, 4); } \
        else NORM_GO(T_, 4, 2); } while (0)
    if (dtype == AGAVE_F32) NORM_T(float); else NORM_T(bf16);
#undef NORM_T
#undef NORM_GO
    AGAVE_LAUNCH_CHECK("routed_norm");
    return 0;
}

// ------------------------------------------------------------------ the pairs sorted by expert
// One workgroup.  Every expert's pairs get a run of whole tiles of TM sorted rows (the last one padded):
//   place[p]        sorted row of pair p (-1: the pair's choice is an identity expert)
//   sorted_pair[r]  pair in sorted row r (-1: padding)
//   tile_expert[t]  expert of tile t (-1: no such tile)
// The order of an expert's pairs among themselves is whatever the atomics make it; every row's result is
// its own, so nothing depends on it.
// A thread keeps its pairs' choices and ranks in registers (SORT_PER of them; of more pairs the ranks wait in `place`), all loads
// of choices leave together and the experts' first tiles are counted up across the lanes.  12,004 pairs of 16
// experts, tiles of 128: 9.1 us, with a load, an atomic and a store at a time and one thread for the tiles 16.1; 32,768 of 64 20.7
// and 55.0.
#define SORT_PER 32
__global__ __launch_bounds__(1024) void route_sort_kernel(const int* __restrict__ choice, int P, int E, int TM, int cap,
                                                          int max_tiles, int* __restrict__ place,
                                                          int* __restrict__ sorted_pair, int* __restrict__ tile_expert) {
    __shared__ int counts[ROUTE_MAX];
    __shared__ int first_row[ROUTE_MAX];
    __shared__ int wave_tiles[16];
    const int tid = threadIdx.x;
    const bool kept = P <= SORT_PER * 1024;
    int e[SORT_PER], rank[SORT_PER];
    if (kept) {
#pragma unroll
        for (int u = 0; u < SORT_PER; ++u) {
            if (u * 1024 >= P) break;
            e[u] = choice[min(tid + u * 1024, P - 1)];
        }
    }
    counts[tid] = 0;                                       // (ROUTE_MAX is the workgroup's size)
    for (int r = tid; r < cap; r += 1024) sorted_pair[r] = -1;
    __syncthreads();
    if (kept) {
#pragma unroll
        for (int u = 0; u < SORT_PER; ++u) {
            if (u * 1024 >= P) break;
            if (tid + u * 1024 >= P || e[u] >= E) e[u] = -1;
            rank[u] = e[u] >= 0 ? atomicAdd(&counts[e[u]], 1) : 0;
        }
    } else {
        for (int p = tid; p < P; p += 1024) {
            const int ep = choice[p];
            place[p] = (ep >= 0 && ep < E) ? atomicAdd(&counts[ep], 1) : -1;        // for now: the pair's rank within its expert
        }
    }
    __syncthreads();
    const int lane = tid & 63, w = tid >> 6, tiles = tid < E ? (counts[tid] + TM - 1) / TM : 0;      // of expert `tid`
    int upto = tiles;
#pragma unroll
    for (int o = 1; o < 64; o *= 2) {
        const int below = __shfl_up(upto, o);
        if (lane >= o) upto += below;
    }
    if (lane == 63) wave_tiles[w] = upto;
    __syncthreads();
    int all = 0;
#pragma unroll
    for (int o = 0; o < 16; ++o) {
        if (o == w) upto += all;
        all += wave_tiles[o];
    }
    first_row[tid] = (upto - tiles) * TM;
    for (int t = upto - tiles; t < upto && t < max_tiles; ++t) tile_expert[t] = tid;
    for (int t = all + tid; t < max_tiles; t += 1024) tile_expert[t] = -1;
    __syncthreads();
    // (a row beyond cap cannot be: cap holds every pair and every expert's padding)
    if (kept) {
#pragma unroll
        for (int u = 0; u < SORT_PER; ++u) {
            if (u * 1024 >= P) break;
            const int p = tid + u * 1024;
            if (p >= P) continue;
            const int r = e[u] >= 0 ? first_row[e[u]] + rank[u] : -1;
            place[p] = r < cap ? r : -1;
            if (r >= 0 && r < cap) sorted_pair[r] = p;
        }
    } else {
        for (int p = tid; p < P; p += 1024) {
            const int ep = choice[p];
            if (ep >= 0 && ep < E) {
                const int r = first_row[ep] + place[p];
                place[p] = r < cap ? r : -1;
                if (r < cap) sorted_pair[r] = p;
            }
        }
    }
}

// Up to 64 pairs and 64 experts (a decode step of few tokens): one wave, a lane per pair and per expert, the experts' tiles counted
// up across the lanes, so that no thread walks the experts alone.  us, with the kernel above and so, tiles
// of 16: 8 pairs of 8 experts 3.2 and 2.2, 24 of 16 4.4 and 2.4, 32 of 64 9.1 and 3.1.
#define FEW_CAP (65 * 64)      // sorted rows: 64 experts and a tile more, in tiles of up to 64
__global__ __launch_bounds__(64) void route_sort_few_kernel(const int* __restrict__ choice, int P, int E, int TM, int cap, int max_tiles,
                                                            int* __restrict__ place, int* __restrict__ sorted_pair,
                                                            int* __restrict__ tile_expert) {
    __shared__ int count[64], first[64], sorted[FEW_CAP];
    const int lane = threadIdx.x;
    const int chosen = lane < P ? choice[lane] : -1, mine = chosen < E ? chosen : -1;
    count[lane] = 0;
    for (int r = lane; r < cap; r += 64) sorted[r] = -1;
    __syncthreads();
    const int rank = mine >= 0 ? atomicAdd(&count[mine], 1) : 0;
    __syncthreads();
    const int tiles = (count[lane] + TM - 1) / TM;           // of expert `lane`
    int upto = tiles;
#pragma unroll
    for (int o = 1; o < 64; o *= 2) {
        const int below = __shfl_up(upto, o);
        if (lane >= o) upto += below;
    }
    first[lane] = (upto - tiles) * TM;
    for (int t = upto - tiles; t < upto; ++t) tile_expert[t] = lane;
    for (int t = __shfl(upto, 63) + lane; t < max_tiles; t += 64) tile_expert[t] = -1;
    __syncthreads();
    const int row = mine >= 0 ? first[mine] + rank : -1;
    if (row >= 0) sorted[row] = lane;                        // (cap holds every pair and every expert's padding)
    __syncthreads();
    for (int r = lane; r < cap; r += 64) sorted_pair[r] = sorted[r];
    if (lane < P) place[lane] = row;
}

extern "C" int agave_route_sort(const int* choice, int P, int E, int TM, int cap, int max_tiles, int* place, int* sorted_pair,
                                int* tile_expert, hipStream_t stream) {
    AGAVE_CHECK(P >= 0 && E > 0 && E <= ROUTE_MAX && (TM == 16 || TM == 64 || TM == 128), "route_sort: bad sizes P=%d E=%d TM=%d", P, E, TM);
    AGAVE_CHECK(max_tiles >= (P + TM - 1) / TM + E && cap >= max_tiles * TM, "route_sort: %d tiles of %d rows do not hold %d pairs of %d experts",
                max_tiles, TM, P, E);
    AGAVE_CHECK(choice && place && sorted_pair && tile_expert, "route_sort: null buffer");
    if (P == 0) return 0;
    if (P <= 64 && E <= 64 && cap <= FEW_CAP) {
        route_sort_few_kernel<<<1, 64, 0, stream>>>(choice, P, E, TM, cap, max_tiles, place, sorted_pair, tile_expert);
        AGAVE_LAUNCH_CHECK("route_sort");
        return 0;
    }
    route_sort_kernel<<<1, 1024, 0, stream>>>(choice, P, E, TM, cap, max_tiles, place, sorted_pair, tile_expert);
    AGAVE_LAUNCH_CHECK("route_sort");
    return 0;
}

// ------------------------------------------------------------------ the experts' products on the matrix cores
// A workgroup takes one tile of TM = 16 MI sorted rows (one expert) and 64 NJ output columns, 16 NJ a wave; both operands
// come straight from memory in the order v_mfma_f32_16x16x32_bf16 reads them (a lane's eight neighbours along K are
// 16 bytes of a row of X or of W[e]).  GATED: two products (gate and up) side by side, ending in act(gate) * up,
// rows gathered from X through the sorted pairs; otherwise one product of the sorted inner rows, 32-bit out.
template <int MI, int NJ, bool GATED>
__global__ __launch_bounds__(256) void routed_product_mfma_kernel(const bf16* __restrict__ x, long ldx, const int* __restrict__ sorted_pair,
                                                                  const int* __restrict__ tile_expert, const bf16* __restrict__ w0,
                                                                  const bf16* __restrict__ w1, void* __restrict__ out_, int top,
                                                                  int n_out, int K, int act, int wpacked, float p0, float p1) {
    const int e = tile_expert[blockIdx.x];
    if (e < 0) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int c = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * 16 * MI;
    // A tile of 16 rows (MI == 1) streams its weights once: its four waves take the same 16 NJ columns and a quarter of
    // K each, so that a wave's chain of loads is a quarter as long, and wave 0 adds the four sums through LDS.
    constexpr bool KSPLIT = MI == 1;
    const int col0 = KSPLIT ? blockIdx.y * (16 * NJ) : blockIdx.y * (64 * NJ) + w * (16 * NJ);
    if (col0 >= n_out) return;                                  // (the whole workgroup where the waves split K)
    const int k_share = KSPLIT ? ((K + 127) / 128) * 32 : K;    // whole steps of 32
    const int k_begin = KSPLIT ? min(K, w * k_share) : 0, k_end = KSPLIT ? min(K, k_begin + k_share) : K;
    // A rows: 16 i + c of the tile
    const bf16* arow[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int r = row0 + 16 * i + c;
        if (GATED) {
            const int p = sorted_pair[r];
            arow[i] = x + (size_t)(p >= 0 ? p / top : 0) * ldx + 8 * g;       // (a padding row computes on row 0 and is never read)
        } else {
            arow[i] = x + (size_t)r * ldx + 8 * g;
        }
    }
    // B rows: output columns col0 + 16 j + c of expert e (clamped; columns past the end are not stored)
    const bf16* b0[NJ];
    const bf16* b1[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        int col = col0 + 16 * j + c;
        if (col >= n_out) col = n_out - 1;
        // (wpacked: W[e] in tiles of 16 rows x 32 columns, each the 64 lanes' operands in a row, a row block's tiles one
        // after another: a whole operand is one load of a kilobyte)
        const size_t at0 = wpacked ? (((size_t)e * (n_out / 16) + col / 16) * (K / 32) * 64 + lane) * 8
                                   : ((size_t)e * n_out + col) * K + 8 * g;
        b0[j] = w0 + at0;
        b1[j] = GATED ? w1 + at0 : nullptr;
    }
    f32x4_t acc0[MI][NJ], acc1[MI][GATED ? NJ : 1];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            acc0[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            if (GATED) acc1[i][GATED ? j : 0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    int k_done = k_begin;
    if constexpr (MI == 1) {
        // a tile of 16 rows streams its weights once and waits for memory, not for the matrix cores: the loads of
        // eight steps are asked for before the first is used
        constexpr int U = 8;
        for (; k_done + 32 * U <= k_end; k_done += 32 * U) {
            frag16 a[U], bw0[U][NJ], bw1[U][NJ];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k0 = k_done + 32 * u;
                a[u].u = *reinterpret_cast<const uint4*>(arow[0] + k0);
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    bw0[u][j].u = *reinterpret_cast<const uint4*>(b0[j] + (wpacked ? k0 * 16 : k0));
                    if (GATED) bw1[u][j].u = *reinterpret_cast<const uint4*>(b1[j] + (wpacked ? k0 * 16 : k0));
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    acc0[0][j] = mfma_16x16x32(a[u], bw0[u][j], acc0[0][j]);
                    if (GATED) acc1[0][GATED ? j : 0] = mfma_16x16x32(a[u], bw1[u][j], acc1[0][GATED ? j : 0]);
                }
        }
    }
    for (int k0 = k_done; k0 < k_end; k0 += 32) {
        // (loads without conditions, from inside the row; a lane past the row's end reads its start and is emptied)
        const bool in = k0 + 8 * g < K;
        const int at = in ? k0 : -8 * g;
        const int bat = wpacked ? k0 * 16 : at;
        frag16 a[MI], bw0[NJ], bw1[NJ];
#pragma unroll
        for (int i = 0; i < MI; ++i) a[i].u = *reinterpret_cast<const uint4*>(arow[i] + at);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            bw0[j].u = *reinterpret_cast<const uint4*>(b0[j] + bat);
            if (GATED) bw1[j].u = *reinterpret_cast<const uint4*>(b1[j] + bat);
        }
        if (!in) {
#pragma unroll
            for (int i = 0; i < MI; ++i) a[i].u = make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                acc0[i][j] = mfma_16x16x32(a[i], bw0[j], acc0[i][j]);
                if (GATED) acc1[i][GATED ? j : 0] = mfma_16x16x32(a[i], bw1[j], acc1[i][GATED ? j : 0]);
            }
    }
    if constexpr (KSPLIT) {
        __shared__ float part[3][2][NJ][256];
        if (w > 0) {
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4) {
                    part[w - 1][0][j][e4 * 64 + lane] = acc0[0][j][e4];
                    if (GATED) part[w - 1][1][j][e4 * 64 + lane] = acc1[0][GATED ? j : 0][e4];
                }
        }
        __syncthreads();
        if (w > 0) return;
#pragma unroll
        for (int ow = 0; ow < 3; ++ow)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4) {
                    acc0[0][j][e4] += part[ow][0][j][e4 * 64 + lane];
                    if (GATED) acc1[0][GATED ? j : 0][e4] += part[ow][1][j][e4 * 64 + lane];
                }
    }
    // D[i][j]: lane holds rows 4 g + e4 of the row block, column c of the column block
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int col = col0 + 16 * j + c;
            if (col >= n_out) continue;
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                const size_t r = (size_t)row0 + 16 * i + 4 * g + e4;
                if (GATED) {
                    ((bf16*)out_)[r * n_out + col] = f32_to_bf16(expert_gated(acc0[i][j][e4], acc1[i][GATED ? j : 0][e4], act, p0, p1));
                } else {
                    ((float*)out_)[r * n_out + col] = acc0[i][j][e4];
                }
            }
        }
}

// Few pairs, weights in tile order, K a multiple of 1,024 (KQ = K / 128 steps of 32 a wave): bound by the weights' way from
// memory.  A workgroup takes a tile of 16 sorted rows through `blocks` blocks of columns (GATED: 16 columns of the gate and the
// up matrix, otherwise 32), its four waves a quarter of K each.  A wave keeps its quarter of the rows in registers for all
// blocks (loaded again for every block, the rows were a third and a half of what the kernel above asks for) and streams its
// weights, two tiles of a kilobyte a step, through a ring of NS steps in LDS of its own: it waits for nobody but its own loads,
// and the loads of the next block's first steps are on their way while this one's sums meet in LDS.
// Measured, us, both products, with the kernel above and so, 1, 2, 4 and 16 rows: 16 experts of 2,048 by 2,048, 4 a row, 34 44 78 117
// and 30 43 57 87; 32 of 1,024 by 1,024, 4 a row, 18 21 27 49 and 15 20 24 38; 8 of 4,096 by 4,096, 2 a row, 44 118 116 185 and 48
// 96 107 153; 8 of 4,096 inner rows by 1,024, 2 a row, 25 33 40 49 and 21 27 39 46.
// Of up to FEW_PAIRS pairs a workgroup finds its own rows from the pairs' choices (CHOSEN): which of them chose the same expert
// as it takes a vote a bit of the expert's number, and a tile is then led by every sixteenth pair of an expert, tiles counted in the
// pairs' order.  The rows of either product are the pairs themselves, and there is no sorted list to wait for, neither its kernel nor
// two loads one after the other at the start of both products.  us, sorting and both products, and so: 17 experts of 2,048 by
// 2,048, 5 a row, 1 row 37.2 and 35.4, 6 rows 93.4 and 76.7, 16 rows 89.6 and 81.6, 48 rows 114 and 100; 32 of 1,024 by 2,048, 4 a row,
// 23.6 and 15.8, 53.5 and 47.7, 71.5 and 62.4, 86.1 and 79.2; 8 of 4,096 by 4,096, 2 a row, 59.5 and 44.1, 123 and 112, 149 and 141, 176 and 154;
// 256 of 1,024 by 1,024, 8 a row, 22.7 and 14.5, 73.3 and 65.1, 133 and 118, 32 rows 211 and 185.  A thread looks at one pair, which is the
// limit; more pairs are sorted as before, in a time that is little of theirs.
#define FEW_PAIRS 256
// The expert of tile `tile` (-1: no such tile) and in mine[16], of this wave, the pairs of its rows (-1: no such row).  With `runs` > 0
// `tile` is a workgroup's number among so many runs of every tile that there is, the first runs of all tiles first, and its own run
// comes back in `run`.  LDS, 16-byte pieces nobody else uses until all waves are back: `counts` 4 E + 6 words, `mine` the waves' rows
// `stride` words apart.
__device__ __forceinline__ int few_tile(const int* __restrict__ choice, int P, int E, int tile, int runs, int& run, int* counts, int* mine, int stride) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool alone = P <= 64;                                   // (every wave looks at all pairs and needs no other)
    const int pair = alone ? lane : (int)threadIdx.x;
    const int chosen = choice[min(pair, P - 1)];
    const bool valid = pair < P && (unsigned)chosen < (unsigned)E;
    if (lane < 16) mine[w * stride + lane] = -1;
    if (!alone)
        for (int i = threadIdx.x; i < 4 * E; i += 256) counts[i] = 0;
    unsigned long long same = __ballot(valid);
    for (int b = 0; (E - 1) >> b; ++b) {
        const bool bit = (chosen >> b) & 1;
        const unsigned long long ones = __ballot(bit);
        same &= bit ? ones : ~ones;
    }
    const unsigned long long below = (1ull << lane) - 1;
    int rank = __popcll(same & below);                            // of the pair among its expert's
    if (!alone) {
        __syncthreads();
        if (valid && (same >> lane) == 1) counts[w * E + chosen] = rank + 1;       // (its expert's last of the wave)
        __syncthreads();
        for (int o = 0; o < w; ++o)
            if (valid) rank += counts[o * E + chosen];
    }
    const unsigned long long leaders = __ballot(valid && (rank & 15) == 0);
    int first = 0, e = -1, base = 0, all = __popcll(leaders);
    if (!alone) {
        if (lane == 0) counts[4 * E + w] = __popcll(leaders);
        __syncthreads();
        all = 0;
        for (int o = 0; o < 4; ++o) {
            if (o == w) first = all;
            all += counts[4 * E + o];
        }
    }
    all = __builtin_amdgcn_readfirstlane(all);
    if (tile >= (runs ? all * runs : all)) return -1;
    if (runs) {
        run = tile / all;
        tile -= run * all;
    }
    const unsigned long long leads = __ballot(((leaders >> lane) & 1) && first + __popcll(leaders & below) == tile);
    if (leads) {
        const int at = __ffsll(leads) - 1;
        e = __builtin_amdgcn_readlane(chosen, at);
        base = __builtin_amdgcn_readlane(rank, at);
    }
    if (alone) {
        if (valid && chosen == e && rank >= base && rank < base + 16) mine[w * stride + rank - base] = pair;
    } else {
        if (leads && lane == 0) {
            counts[4 * E + 4] = e;
            counts[4 * E + 5] = base;
        }
        __syncthreads();
        e = counts[4 * E + 4];
        base = counts[4 * E + 5];
        if (valid && chosen == e && rank >= base && rank < base + 16)
            for (int o = 0; o < 4; ++o) mine[o * stride + rank - base] = pair;
        __syncthreads();
    }
    __builtin_amdgcn_wave_barrier();                              // (a wave's LDS accesses happen in the order they were issued)
    return __builtin_amdgcn_readfirstlane(e);
}

#define FEW_BY_COLUMN 0                                           // how workgroups go through tiles and runs of blocks (see launch_routed_few);
#define FEW_BY_TILE -1                                            // more than 0: so many runs, of the tiles that there are
template <int KQ, bool GATED, bool CHOSEN>
__global__ __launch_bounds__(256, 2) void routed_product_few_kernel(const bf16* __restrict__ x, long ldx, const int* __restrict__ sorted_pair,
                                                                    const int* __restrict__ tile_expert, const uint4* __restrict__ w0,
                                                                    const uint4* __restrict__ w1, void* __restrict__ out_, int top, int n_out,
                                                                    int act, int blocks, float p0, float p1, int P, int E, int tiles, int order) {
    constexpr int K = KQ * 128, KB = K / 32, NS = 8;
    static_assert(KQ % NS == 0, "a step's place in the ring is known where it is written");
    constexpr int COLS = GATED ? 16 : 32;
    __shared__ __attribute__((aligned(16))) unsigned char ring[4][NS][2048];
    __shared__ float part[2][4][2][256];
    static_assert(sizeof(ring) >= (4 * ROUTE_MAX + 6) * sizeof(int), "the experts' counts fit the ring");
    // (CHOSEN: sorted_pair holds the choices; part's first half keeps the rows' pairs until its first sums)
    int* mine = reinterpret_cast<int*>(&part[0][0][0][0]);
    int tile = blockIdx.x, run = blockIdx.y;
    if (CHOSEN && order == FEW_BY_TILE) {                         // (what is left of the tiles lies in the last rows of the grid)
        const int left = (int)blockIdx.y - tiles;
        tile = left < 0 ? (int)blockIdx.y : left * (int)gridDim.x + (int)blockIdx.x;
        run = left < 0 ? (int)blockIdx.x : (int)gridDim.x;
    }
    const int e = CHOSEN ? few_tile(sorted_pair, P, E, tile, order > 0 ? order : 0, run, reinterpret_cast<int*>(&ring[0][0][0]), mine, 512) : tile_expert[tile];
    if (e < 0) return;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * 16, NBK = n_out / 16;           // (not CHOSEN)
    const int b0 = run * blocks, b1 = min(b0 + blocks, (n_out + COLS - 1) / COLS);
    if (b0 >= b1) return;
    long r = row0 + c;
    int out_row = row0 + 4 * g + w;                               // -1: not stored
    if (CHOSEN) {
        const int p = mine[w * 512 + c];
        out_row = mine[w * 512 + 4 * g + w];
        r = p >= 0 ? (GATED ? p / top : p) : 0;
    } else if (GATED) {
        const int p = sorted_pair[r];
        r = p >= 0 ? p / top : 0;                                 // (a padding row computes on row 0 and is never read)
    }
    const bf16* arow = x + (size_t)r * ldx + w * (K / 4) + 8 * g;
    frag16 a[KQ];
#pragma unroll
    for (int k = 0; k < KQ; ++k) a[k].u = *reinterpret_cast<const uint4*>(arow + 32 * k);
    // the two tiles of step k of block b
    auto fetch = [&](int b, int k, int slot) {
        b = b < b1 ? b : b1 - 1;                                  // (past the end: loaded, never used)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            int nb = GATED ? b : 2 * b + i;
            nb = nb < NBK ? nb : NBK - 1;                         // (columns past the end: never stored)
            const uint4* src = (GATED && i ? w1 : w0) + (((size_t)e * NBK + nb) * KB + w * KQ + k) * 64 + lane;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                             (__attribute__((address_space(3))) void*)&ring[w][slot][i * 1024], 16, 0, 0);
        }
    };
#pragma unroll
    for (int k = 0; k < NS - 1; ++k) fetch(b0, k, k);
    const unsigned at = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)&ring[w][0][0] + lane * 16;
    constexpr int IN_FLIGHT = 2 * (NS - 2);
    for (int b = b0; b < b1; ++b) {
        f32x4_t acc[2] = {};
        static_for<0, KQ>([&](auto kc) {
            constexpr int k = kc.value, slot = k % NS;
            __builtin_amdgcn_s_waitcnt(0x0F70 | (IN_FLIGHT & 15) | ((IN_FLIGHT >> 4) << 14));
            frag16 f0, f1;
            lds_read16<slot * 2048>(f0, at);
            lds_read16<slot * 2048 + 1024>(f1, at);
            lds_settle();
            lds_use(f0);
            lds_use(f1);
            // (the step before this one has been read: its place is free)
            fetch(k + NS - 1 < KQ ? b : b + 1, (k + NS - 1) % KQ, (slot + NS - 1) % NS);
            acc[0] = mfma_16x16x32(a[k], f0, acc[0]);
            acc[1] = mfma_16x16x32(a[k], f1, acc[1]);
        });
        // D: lane holds rows 4 g + e4, column c; wave w adds up and stores rows 4 g + w
        float (&sums)[4][2][256] = part[b & 1];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) sums[w][i][e4 * 64 + lane] = acc[i][e4];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                             // (a bare barrier: the next block's weights stay on their way)
        asm volatile("" ::: "memory");
        float v[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) v[i] = ((sums[0][i][w * 64 + lane] + sums[1][i][w * 64 + lane]) + sums[2][i][w * 64 + lane]) + sums[3][i][w * 64 + lane];
        if (CHOSEN && out_row < 0) continue;
        const size_t row = (size_t)out_row;
        if constexpr (GATED) {
            ((bf16*)out_)[row * n_out + b * 16 + c] = f32_to_bf16(expert_gated(v[0], v[1], act, p0, p1));
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int col = b * 32 + 16 * i + c;
                if (col < n_out) ((float*)out_)[row * n_out + col] = v[i];
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                           // loads past the last step land before the LDS goes to another workgroup
}

// The columns that the kernel above is built for (its rows take K / 32 registers a lane, and the ring's places have to come out even).
extern "C" int agave_routed_few_takes(int K) { return K == 1024 || K == 2048 || K == 4096; }

template <bool GATED, bool CHOSEN>
static bool launch_routed_few(const void* x, long ldx, const int* sorted_pair, const int* tile_expert, int max_tiles, const void* w0,
                              const void* w1, void* out, int top, int live, int n_out, int K, int act, float p0, float p1, int P, int E, hipStream_t stream) {
    if (!agave_routed_few_takes(K)) return false;
    const int all = (n_out + (GATED ? 15 : 31)) / (GATED ? 16 : 32);
    // Blocks a workgroup: the fewest with which all workgroups of the experts that are expected run at once, two to a compute unit, with a
    // few of the 512 places left.  Both products, 4 rows: 75.8, 63.0, 66.7 us with 2, 4, 5 blocks of the gate; 6 rows
    // 78.8, 68.3, 70.7; 16 rows 93.5, 93.0, 89.1; 1 row 32.5 and 42.3 with 2 and 4.  Whole feed-forwards: sixteen experts and a shared
    // one, 6 rows, 5 and 3 blocks of gate and down 78.3, 4 and 2 (480 workgroups) 73.5; 32 of 1,024 by 2,048 and a shared one, 16 rows, 5
    // blocks 98.9, 4 (496) 93.7; eight of 4,096 by 4,096, 12 rows, 5 and 3 (416) 178, 4 and 2 (512) 205.
    int blocks = (int)(((long)live * all + 499) / 500);
    blocks = blocks < 1 ? 1 : blocks > 16 ? 16 : blocks;
    // CHOSEN: column by column, as sorted tiles, where all places run at once.  Beyond, tile by tile, so that the workgroups with rows are
    // the first to start; those without look at the choices too and were among them, and with as many places for tiles as a multiple of
    // eight a tile's runs were all on one XCD.  What is less than `blocks` of a tile comes behind all of them and fills up a second
    // round if there is one.  With 4,096 columns, run by run of the tiles that there are.  us, sorted, column by
    // column, and so (means of six choices): eight of 96 of 1,024 by 2,048 a row, 8 rows 119, 122, 106; eight of 65 of 1,024 by 1,024, 6 rows 56.1,
    // 55.8, 47.9; eight of 129 of 1,024 by 2,048, 12 rows 175, 167, 155; two of 32 of 2,048 by 4,096, 16 rows 199, 193, 185.
    const int runs = (all + blocks - 1) / blocks, whole = all / blocks;
    if ((long)max_tiles * runs >= 1L << 31) return false;
    int order = FEW_BY_COLUMN;
    dim3 grid(max_tiles, runs);
    if (CHOSEN && (long)max_tiles * runs > 512) {
        if (K == 4096) order = runs, grid = dim3(max_tiles * runs);
        else order = FEW_BY_TILE, grid = dim3(whole, max_tiles + (runs > whole ? (max_tiles + whole - 1) / whole : 0));
    }
    if (grid.y > 65535) return false;
#define FEW_GO(KQ_) routed_product_few_kernel<KQ_, GATED, CHOSEN><<<grid, 256, 0, stream>>>((const bf16*)x, ldx, sorted_pair, tile_expert, (const uint4*)w0, \
                                                                                            (const uint4*)w1, out, top, n_out, act, blocks, p0, p1, P, E, max_tiles, order)
    if (K == 1024) FEW_GO(8);
    else if (K == 2048) FEW_GO(16);
    else FEW_GO(32);
#undef FEW_GO
    return true;
}

// experts that have rows, if the rows choose evenly
static int live_experts(int n_rows, int top, int E) { return top >= E ? E : (int)ceil(E * (1.0 - pow(1.0 - (double)top / E, (double)n_rows))); }

// Whether agave_routed_experts_chosen takes a feed-forward: few pairs, columns of both products that the kernel above streams.
extern "C" int agave_routed_chosen_takes(int P, int E, int ff, int hidden) {
    return P > 0 && P <= FEW_PAIRS && E > 0 && E <= ROUTE_MAX && agave_routed_few_takes(ff) && agave_routed_few_takes(hidden);
}

// The experts' products of few pairs, weights in tile order, without a sorted list: act_rows [n top, ff] bfloat16 and
// y [n top, hidden] float32 hold a row a pair (nothing for a pair whose choice is no expert).
extern "C" int agave_routed_experts_chosen(const void* x, long ldx, const int* choice, const void* wg, const void* wu, const void* wd, void* act_rows, float* y,
                                           int n_rows, int top, int E, int ff, int hidden, int act, float p0, float p1, hipStream_t stream) {
    AGAVE_CHECK(n_rows >= 0 && top > 0 && ldx >= hidden && ldx % 8 == 0, "routed_experts_chosen: bad sizes");
    if (n_rows == 0) return 0;
    AGAVE_CHECK((long)n_rows * top <= FEW_PAIRS && agave_routed_chosen_takes(n_rows * top, E, ff, hidden), "routed_experts_chosen: %d rows of %d pairs, %d experts of %d by %d",
                n_rows, top, E, ff, hidden);
    AGAVE_CHECK((act >= 0 && act < 4) || act == 6, "routed_experts_chosen: unknown activation %d", act);
    AGAVE_CHECK(x && choice && wg && wu && wd && act_rows && y, "routed_experts_chosen: null buffer");
    AGAVE_CHECK((((uintptr_t)x | (uintptr_t)wg | (uintptr_t)wu | (uintptr_t)wd | (uintptr_t)act_rows) & 15) == 0, "routed_experts_chosen: buffers must be aligned to 16 bytes");
    const int P = n_rows * top, live = live_experts(n_rows, top, E), tiles = min(P, (P + 15) / 16 + E);
    const bool done = launch_routed_few<true, true>(x, ldx, choice, nullptr, tiles, wg, wu, act_rows, top, live, ff, hidden, act, p0, p1, P, E, stream)
                   && launch_routed_few<false, true>(act_rows, ff, choice, nullptr, tiles, wd, nullptr, y, top, live, hidden, ff, act, p0, p1, P, E, stream);
    AGAVE_CHECK(done, "routed_experts_chosen: sizes the kernel is not built for");
    AGAVE_LAUNCH_CHECK("routed_experts_chosen");
    return 0;
}

// Many pairs an expert, weights in tile order: a workgroup takes a tile of TT sorted rows and 2 TT columns of weights
// (GATED: TT columns of the gate and the same of the up matrix), TT/16 waves of 64 weight columns by TT/2 rows each.
// Bound by the multiply-adds once both operands come through LDS: a wave that loads its own operands asks the compute
// unit's cache for 96 bytes a clock where it delivers 64.  Both operands go straight from memory into LDS (a kilobyte a
// load), stages of 32 columns in a ring of NS buffers, the loads of NS - 1 stages in flight while one is multiplied; 72 KB
// (TT 128), so that two workgroups share a compute unit and one multiplies while the other waits at its barrier.
// The rows' 16-byte pieces are permuted by the row so that the rows an operand reads lie in different banks.
// Workgroups go to the 8 XCDs in turn: each XCD takes an eighth of the tiles there are (neighbours, so mostly one expert's)
// and walks them column block by column block, which keeps an expert's block of weights in that XCD's L2 while its tiles
// pass over it.
// Measured, both products, 16 experts of 2,048 by 2,048: 12,004 pairs in tiles of 128 445 us (679 TFLOP/s), of 64 572 us;
// 3,200 pairs 138 and 209 us; 64 pairs in tiles of 64 84 us (4.8 TB/s of weights).  With every wave loading its own operands
// (as below, tiles of 64) 987 us, 334 us; tiles of 16 109 us at 64 pairs.
template <int TT, bool GATED>
__global__ __launch_bounds__(TT * 4, 4) void routed_product_tiled_kernel(const bf16* __restrict__ x, long ldx, const int* __restrict__ sorted_pair,
                                                                         const int* __restrict__ tile_expert, int max_tiles,
                                                                         const uint4* __restrict__ w0, const uint4* __restrict__ w1,
                                                                         void* __restrict__ out_, int top, int n_out, int K, int act, float p0,
                                                                         float p1) {
    constexpr int NWV = TT / 16, WSLOTS = TT / 8;                 // waves; weight tiles of 16 columns a stage
    constexpr int NS = TT == 128 ? 3 : 4;
    constexpr int X_BYTES = TT * 64, STAGE = X_BYTES + WSLOTS * 1024;
    constexpr int XB = TT / 32;                                   // 16-row tiles of a wave
    constexpr int COLS = GATED ? TT : 2 * TT;                     // columns of the result
    constexpr int LOADS = 3;                                      // a wave's loads per stage: 1 of rows, 2 of weights
    extern __shared__ __attribute__((aligned(16))) unsigned char rt_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wn = wave >> 1, wm = wave & 1;
    const int c = lane & 15, g = lane >> 4;
    // this XCD's share of the tiles that hold rows (they are the first ones of the table)
    int count = 0;
    for (int t0 = 0; t0 < max_tiles; t0 += 64) {
        const int t = t0 + lane;
        count += __popcll(__ballot(tile_expert[t < max_tiles ? t : max_tiles - 1] >= 0 && t < max_tiles));
    }
    const int share = (count + 7) / 8;
    if (share == 0) return;
    const int xcd = blockIdx.x & 7, turn = blockIdx.x >> 3;
    const int tile = xcd * share + turn % share, col0 = turn / share * COLS;
    if (tile >= count || col0 >= n_out) return;
    const int e = tile_expert[tile];
    const int row0 = tile * TT;
    const int KB = K / 32, NBK = n_out / 16;

    // staging: one 16-byte piece of a row and two weight tiles a wave and stage
    const unsigned char* xsrc;
    {
        const int o = wave * 64 + lane, row = o >> 2, piece = (o & 3) ^ ((row >> 2) & 3);
        long r = row0 + row;
        if (GATED) {
            const int p = sorted_pair[r];
            r = p >= 0 ? p / top : 0;                             // (a padding row computes on row 0 and is never read)
        }
        xsrc = (const unsigned char*)(x + (size_t)r * ldx) + piece * 16;
    }
    const unsigned char* wsrc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int slot = wave * 2 + i;
        const uint4* w = GATED && slot >= WSLOTS / 2 ? w1 : w0;
        int nb = col0 / 16 + (GATED ? slot % (WSLOTS / 2) : slot);
        if (nb >= NBK) nb = NBK - 1;                              // (columns past the end: never stored)
        wsrc[i] = (const unsigned char*)(w + ((size_t)e * NBK + nb) * KB * 64) + lane * 16;
    }
    auto fetch_one = [&](int st, int buf, int i) {                // load i of stage st (past the end: the last one again, never used)
        const size_t ste = st < KB ? st : KB - 1;
        unsigned char* dst = rt_lds + buf * STAGE + (i == 0 ? wave * 1024 : X_BYTES + (wave * 2 + i - 1) * 1024);
        const unsigned char* src = i == 0 ? xsrc + ste * 64 : wsrc[i - 1] + ste * 1024;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
    };
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)rt_lds;
    // operand a of a wave: 16 weight columns.  GATED: a = 0, 1 the gate's, 2, 3 the up matrix's of the same 32 columns
    const unsigned w_lane = lds0 + X_BYTES + (GATED ? wn * 2 : wn * 4) * 1024 + lane * 16;
    constexpr int UP_AT = GATED ? (WSLOTS / 2 - 2) * 1024 : 0;    // from slot a = 2 on: the up matrix's half
    const unsigned x_lane = lds0 + (wm * (TT / 2) + c) * 64 + ((g ^ ((c >> 2) & 3)) * 16);

    f32x4_t acc[4][XB];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < XB; ++b) acc[a][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int st = 0; st < NS - 1; ++st)
#pragma unroll
        for (int i = 0; i < LOADS; ++i) fetch_one(st, st, i);
    constexpr int IN_FLIGHT = LOADS * (NS - 2);
    int buf = 0, fill = NS - 1;
    for (int st = 0; st < KB; ++st) {
        __builtin_amdgcn_s_waitcnt(0x0F70 | (IN_FLIGHT & 15) | ((IN_FLIGHT >> 4) << 14));
        __builtin_amdgcn_s_barrier();                             // stage st has landed; stage st - 1 has been read by all
        frag16 fw[4], fx[XB];
        const unsigned wa = w_lane + buf * STAGE, xa = x_lane + buf * STAGE;
        static_for<0, 4>([&](auto a) { lds_read16<a.value * 1024 + (a.value >= 2 ? UP_AT : 0)>(fw[a.value], wa); });
        static_for<0, XB>([&](auto b) { lds_read16<b.value * 1024>(fx[b.value], xa); });
        lds_settle();
#pragma unroll
        for (int a = 0; a < 4; ++a) lds_use(fw[a]);
#pragma unroll
        for (int b = 0; b < XB; ++b) lds_use(fx[b]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < XB; ++b) {
#pragma unroll
            for (int a = 0; a < 4; ++a) acc[a][b] = mfma_16x16x32(fw[a], fx[b], acc[a][b]);
            __builtin_amdgcn_sched_barrier(0);
            if (b < LOADS) fetch_one(st + NS - 1, fill, b);       // a load at a time, between the multiplications
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int b = XB; b < LOADS; ++b) fetch_one(st + NS - 1, fill, b);
        buf = buf + 1 == NS ? 0 : buf + 1;
        fill = fill + 1 == NS ? 0 : fill + 1;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                           // loads past the last stage must have landed before LDS is used again

    // acc[a][b]: row 16 b + c of the wave's rows, columns 4 g .. 4 g + 3 of operand a.  Half of the tile's rows at a time go
    // through LDS and leave it row by row, 16 bytes a lane in whole lines (the 32-bit rows may begin at any element: in
    // single ones where that is off 16 bytes; the inner rows are aligned, the host has seen to it).
    const bool whole = ((uintptr_t)out_ & 15) == 0;
    constexpr int ES = GATED ? 2 : 4, ROW_BYTES = COLS * ES, CH = ROW_BYTES / 16, SWZ = (CH < 32 ? CH : 32) - 1;
    static_assert((TT / 2) * ROW_BYTES <= NS * STAGE, "half of the finished tile fits the LDS");
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        __syncthreads();
        if (wm == half) {
#pragma unroll
            for (int b = 0; b < XB; ++b) {
                const int t = 16 * b + c;
#pragma unroll
                for (int a = 0; a < (GATED ? 2 : 4); ++a) {
                    const int off = (GATED ? wn * 32 + a * 16 + 4 * g : wn * 64 + a * 16 + 4 * g) * ES;
                    unsigned char* dst = rt_lds + t * ROW_BYTES + (((off >> 4) ^ (t & SWZ)) << 4) + (off & 15);
                    if constexpr (GATED) {
                        float v[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) v[k] = expert_gated(acc[a][b][k], acc[a + 2][b][k], act, p0, p1);
                        *reinterpret_cast<uint2*>(dst) = make_uint2(f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3]));
                    } else {
                        *reinterpret_cast<f32x4_t*>(dst) = acc[a][b];
                    }
                }
            }
        }
        __syncthreads();
        constexpr int ROWS_PER = 64 / CH > 0 ? 64 / CH : 1;       // rows of one store
        const int piece = lane % CH;
        for (int t = wave * ROWS_PER + lane / CH; t < TT / 2; t += NWV * ROWS_PER) {
            const int col = col0 + piece * (16 / ES);
            if (col >= n_out) continue;                           // (n_out is a multiple of 16: a piece is inside or outside)
            const uint4 v = *reinterpret_cast<const uint4*>(rt_lds + t * ROW_BYTES + ((piece ^ (t & SWZ)) << 4));
            unsigned char* dst = (unsigned char*)out_ + ((size_t)(row0 + half * (TT / 2) + t) * n_out + col) * ES;
            if (GATED || whole) {
                *reinterpret_cast<uint4*>(dst) = v;
            } else {
                unsigned* one = reinterpret_cast<unsigned*>(dst);
                one[0] = v.x; one[1] = v.y; one[2] = v.z; one[3] = v.w;
            }
        }
    }
}

template <int TT, bool GATED>
static int launch_routed_tiled(const void* x, long ldx, const int* sorted_pair, const int* tile_expert, int max_tiles, const void* w0,
                               const void* w1, void* out, int top, int n_out, int K, int act, float p0, float p1, hipStream_t stream) {
    constexpr int COLS = GATED ? TT : 2 * TT;
    constexpr size_t lds = (size_t)(TT == 128 ? 3 : 4) * (TT * 64 + TT / 8 * 1024);
    const long wgs = 8L * ((max_tiles + 7) / 8) * ((n_out + COLS - 1) / COLS);
    AGAVE_CHECK(wgs < (1L << 31), "routed_experts_mfma: too many tiles for the grid");
    static bool raised = false;
    if (!raised) {
        hipError_t e = hipFuncSetAttribute((const void*)routed_product_tiled_kernel<TT, GATED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        AGAVE_CHECK(e == hipSuccess, "routed_experts_mfma: cannot raise the LDS allowance");
        raised = true;
    }
    routed_product_tiled_kernel<TT, GATED><<<(unsigned)wgs, TT * 4, lds, stream>>>((const bf16*)x, ldx, sorted_pair, tile_expert, max_tiles,
                                                                                   (const uint4*)w0, (const uint4*)w1, out, top, n_out, K, act, p0, p1);
    return 0;
}

// act_rows [cap, ff] bfloat16 and y [cap, hidden] float32 hold sorted rows (see route_sort)
extern "C" int agave_routed_experts_mfma(const void* x, long ldx, const int* sorted_pair, const int* tile_expert, const void* wg,
                                         const void* wu, const void* wd, void* act_rows, float* y, int TM, int max_tiles, int n_rows, int top,
                                         int E, int ff, int hidden, int act, int wpacked, float p0, float p1, hipStream_t stream) {
    AGAVE_CHECK(!wpacked || (ff % 32 == 0 && hidden % 32 == 0), "routed_experts_mfma: weights in tile order need sizes that are multiples of 32");
    AGAVE_CHECK(max_tiles > 0 && n_rows >= 0 && top > 0 && E > 0 && ff > 0 && hidden > 0 && (TM == 16 || TM == 64 || (TM == 128 && wpacked)), "routed_experts_mfma: bad sizes");
    AGAVE_CHECK((act >= 0 && act < 4) || act == 6, "routed_experts_mfma: unknown activation %d", act);
    AGAVE_CHECK(hidden % 8 == 0 && ff % 8 == 0 && ldx % 8 == 0, "routed_experts_mfma: sizes must be multiples of 8 (hidden %d, ff %d)", hidden, ff);
    AGAVE_CHECK(x && sorted_pair && tile_expert && wg && wu && wd && act_rows && y, "routed_experts_mfma: null buffer");
    AGAVE_CHECK(((uintptr_t)x % 16) == 0 && ((uintptr_t)wg % 16) == 0 && ((uintptr_t)wu % 16) == 0 && ((uintptr_t)wd % 16) == 0 &&
                ((uintptr_t)act_rows % 16) == 0, "routed_experts_mfma: buffers must be aligned to 16 bytes");
    if (wpacked && TM >= 64) {
        int rc;
        if (TM == 128) {
            rc = launch_routed_tiled<128, true>(x, ldx, sorted_pair, tile_expert, max_tiles, wg, wu, act_rows, top, ff, hidden, act, p0, p1, stream);
            if (rc == 0) rc = launch_routed_tiled<128, false>(act_rows, ff, sorted_pair, tile_expert, max_tiles, wd, nullptr, y, top, hidden, ff, act, p0, p1, stream);
        } else {
            rc = launch_routed_tiled<64, true>(x, ldx, sorted_pair, tile_expert, max_tiles, wg, wu, act_rows, top, ff, hidden, act, p0, p1, stream);
            if (rc == 0) rc = launch_routed_tiled<64, false>(act_rows, ff, sorted_pair, tile_expert, max_tiles, wd, nullptr, y, top, hidden, ff, act, p0, p1, stream);
        }
        if (rc != 0) return rc;
        AGAVE_LAUNCH_CHECK("routed_experts_mfma");
        return 0;
    }
    // tiles of 64 rows take 64 columns a wave (an operand that was loaded serves more multiplications); a tile of
    // 16 rows, which streams its weights once, takes 16 columns a workgroup, whose waves share K
    const int cols = TM == 64 ? 256 : 16;
    const dim3 g1(max_tiles, (ff + cols - 1) / cols), g2(max_tiles, (hidden + cols - 1) / cols);
    AGAVE_CHECK(g1.y <= 65535 && g2.y <= 65535, "routed_experts_mfma: too many columns for the grid");
    if (TM == 64) {
        routed_product_mfma_kernel<4, 4, true><<<g1, 256, 0, stream>>>((const bf16*)x, ldx, sorted_pair, tile_expert, (const bf16*)wg,
                                                                    (const bf16*)wu, act_rows, top, ff, hidden, act, wpacked, p0, p1);
        routed_product_mfma_kernel<4, 4, false><<<g2, 256, 0, stream>>>((const bf16*)act_rows, ff, sorted_pair, tile_expert, (const bf16*)wd,
                                                                     nullptr, y, top, hidden, ff, act, wpacked, p0, p1);
    } else {
        const int live = live_experts(n_rows, top, E);
        const bool few1 = wpacked && launch_routed_few<true, false>(x, ldx, sorted_pair, tile_expert, max_tiles, wg, wu, act_rows, top, live, ff, hidden, act, p0, p1, 0, 0, stream);
        if (!few1)
            routed_product_mfma_kernel<1, 1, true><<<g1, 256, 0, stream>>>((const bf16*)x, ldx, sorted_pair, tile_expert, (const bf16*)wg,
                                                                    (const bf16*)wu, act_rows, top, ff, hidden, act, wpacked, p0, p1);
        const bool few2 = wpacked && launch_routed_few<false, false>(act_rows, ff, nullptr, tile_expert, max_tiles, wd, nullptr, y, top, live, hidden, ff, act, p0, p1, 0, 0, stream);
        if (!few2)
            routed_product_mfma_kernel<1, 1, false><<<g2, 256, 0, stream>>>((const bf16*)act_rows, ff, sorted_pair, tile_expert, (const bf16*)wd,
                                                                     nullptr, y, top, hidden, ff, act, wpacked, p0, p1);
    }
    AGAVE_LAUNCH_CHECK("routed_experts_mfma");
    return 0;
}
