// The tile kernel of products of many tokens that are not taken in 256 x 256 tiles (gemm_mfma.hip chooses).
#pragma once
#include "common.h"
#include "mfma.h"

// A workgroup of eight waves (WN x WM) computes WN*RT*16 weight rows x WM*CT*16 tokens, a wave RT x CT tiles of 16 x 16
// (v_mfma_f32_16x16x32_bf16).  Both operands come into LDS straight from global memory, 64 columns a stage (whole cache lines of
// the token rows: with 32 a 160 x 256 tile took a seventh longer), in a ring of NS buffers, and go from there to registers a
// k-step of 32 columns ahead of their use.
//
// What bounds it.  A wave issues an instruction every four or five clocks, and with one barrier a stage the waves keep in
// step: in a 64 x 128 tile, whose stage multiplies for 256 clocks, some 130 instructions of addresses, conditions and waits a wave and
// stage cost more than the multiplications.  So the loop has none that can be worked out before it: scalar bases that move on,
// per-lane offsets that stay, the waits' counts as constants (the last NS stages, which ask for nothing any more, are a copy of
// their own), and 70 are left.  Past that it is the L2 and what lies behind it: 50 to 70 bytes a nanosecond and compute unit arrive
// with all 256 of them asking, and a tile of r x t needs (r + t) / (r t) of them an operation; hence the large tiles where they fill
// the chip.  The depth of the ring and a second k-step of operands ahead changed nothing.
// Tiles of 160 rows are there because the 4B sizes' row counts (20,480 and 2,560) make whole rounds of 256 workgroups with them.
// Measured, cold weights, microseconds, before (32 x 32 tiles of the matrix cores, loads and waits with their conditions) and now:
// gate and up (2 x 10,240 rows of 2,560) 256 tokens 40.4 -> 36, 384 65 -> 42, 512 75 -> 50, 1,024 111 -> 97, 2,048 210 -> 184;
// down (2,560 rows of 10,240) 512 in four slices 43.8 -> 35, 4,096 225 -> 164, 8,192 405 -> 328; o (2,560 of 2,048) 512 14.2 -> 12.7,
// 2,048 29.5 -> 24.1; q/k/v (4,096 of 2,560) 512 19.8 -> 19.3, 2,048 45 -> 41.
// No instantiation may spill: a register that the LDS still has to write must not be moved (RT * CT up to 24 is safe).
template <int RT, int CT, int WN, int WM, int NS, int EPI, typename TC>
__global__ __launch_bounds__(512, 2) void gemm_tile_kernel(const bf16* __restrict__ X, long ldx, const uint4* __restrict__ Wp,
                                                         TC* __restrict__ Y, long ldy, int M, int N, int K, int KB, int NB,
                                                         long part_stride, GateForm F) {
    static_assert(WN * WM == 8, "eight waves");
    static_assert(RT * CT <= 24, "the operands must stay in registers while they arrive");
    constexpr int TT = 16 * CT * WM, WTILES = RT * WN;               // tokens and packed 16-row weight tiles a workgroup
    constexpr int KT = 2;                                            // k-steps a stage: whole cache lines of the token rows
    constexpr int CPR = KT * 4;                                      // 16-byte pieces per staged token row
    constexpr int RP = 16 / CPR;                                     // token rows per 256 bytes of LDS
    constexpr int X_BYTES = TT * KT * 64, W_BYTES = WTILES * KT * 1024, STAGE_BYTES = X_BYTES + W_BYTES;
    constexpr int X_LOADS = X_BYTES / 1024, W_LOADS = W_BYTES / 1024, TL = X_LOADS + W_LOADS;   // of a kilobyte, a workgroup and stage
    constexpr int LMAX = (TL + 7) / 8, FULL = TL % 8;                // the first FULL waves (0: all) have LMAX of them, the others one less
    static_assert(NS >= 2 && LMAX * (NS - 1) < 64, "the load counter holds 6 bits");
    extern __shared__ __attribute__((aligned(16))) unsigned char gt_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wn = wave % WN, wm = wave / WN;
    const int j = lane & 15, g = lane >> 4;
    const int nbw = blockIdx.x * WTILES;                             // first packed weight tile of this workgroup
    const int m0 = blockIdx.y * TT;                                  // first token of this workgroup
    // gridDim.z workgroups share a tile's columns: each takes a run of stages and leaves its sum in its own slice of Y
    const int n_stage_all = (KB + KT - 1) / KT;
    const int st0 = (int)((long)blockIdx.z * n_stage_all / gridDim.z);
    const int st_end = (int)((long)(blockIdx.z + 1) * n_stage_all / gridDim.z);       // one past this workgroup's last stage
    Y += (size_t)blockIdx.z * part_stride;

    f32x4_t acc[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[r][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // Load l of a stage (its kilobyte of LDS): token rows first, weight tiles behind them; wave w takes l = w, w + 8, ...  An
    // address is one of two scalar bases, moved from stage to stage, plus a per-lane offset that stays: the loop is bound by the
    // instructions a wave issues where the tile is small (see below), so none is spent on what can be worked out before it.
    constexpr int XI = X_LOADS / 8, WI = LMAX - XI;                  // of them loads of token rows and of weights
    static_assert(X_LOADS % 8 == 0, "token tiles of whole multiples of 64");
    const int st_last = n_stage_all - 1;                             // the stage that may hold columns past K
    const unsigned char* xp = (const unsigned char*)(X + (size_t)m0 * ldx) + (size_t)st0 * (KT * 64);
    const unsigned char* wp = (const unsigned char*)(Wp + w_tile(nbw, st0 * KT + (wave % KT), NB, KB) * 64);
    const size_t wstep = (size_t)(w_tile(0, KT, NB, KB) - w_tile(0, 0, NB, KB)) * 1024;
    unsigned xoff[XI], woff[WI];
    const int xrow = lane / CPR + wave * (64 / CPR), xpos = lane % CPR;        // (load i: 512 / CPR rows further)
    auto x_piece = [&](int i) { return xpos ^ (((xrow + i * (512 / CPR)) / RP) % CPR); };      // the 8 columns a lane's piece holds
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int row = xrow + i * (512 / CPR);
        const int mrow = m0 + row < M ? row : M - 1 - m0;            // rows past the end repeat the last one (never stored)
        xoff[i] = (unsigned)(((size_t)mrow * ldx + x_piece(i) * 8) * 2);
    }
#pragma unroll
    for (int i = 0; i < WI; ++i) {
        const int t = wave / KT + i * (8 / KT);                      // row tile of the workgroup's
        woff[i] = lane * 16 + (nbw + t < NB ? t : NB - 1 - nbw) * 1024;        // (rows past the end: never stored)
    }
    auto fetch_one = [&](unsigned buf, auto ic) {
        constexpr int i = decltype(ic)::value;
        if ((i + 1) * 8 > TL && i * 8 + wave >= TL) return;
        __attribute__((address_space(3))) void* dst = (__attribute__((address_space(3))) void*)(gt_lds + buf + wave * 1024 + i * 8192);
        const unsigned char* src = i < XI ? xp + xoff[i < XI ? i : 0] : wp + woff[i < XI ? 0 : i - XI];
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, dst, 16, 0, 0);
    };
    auto next_stage = [&]() { xp += KT * 64; wp += wstep; };
    // Before the loads of the last stage where columns or k-steps are missing from it: a piece past the last column reads the
    // stage's first columns instead (the weights are zero there), a k-step past the last one the last one (zeroed before it is used).
    const int ragged = K % (KT * 32) != 0 ? st_last : -1;
    auto mend_last = [&]() {
#pragma unroll
        for (int i = 0; i < XI; ++i)
            if (st_last * (KT * 32) + x_piece(i) * 8 >= K) xoff[i] -= x_piece(i) * 16;
        if (st_last * KT + wave % KT >= KB) wp -= (size_t)NB * 1024;
    };

    // This lane's operands of a k-step.  The token rows' pieces are permuted by (row / RP) % CPR, the same for rows 16 apart.
    struct Operands { frag16 w[RT]; frag16 x[CT]; };
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)gt_lds;
    const unsigned w_lane = lds0 + X_BYTES + wn * RT * KT * 1024 + lane * 16;
    unsigned x_lane[KT];
#pragma unroll
    for (int ks = 0; ks < KT; ++ks)
        x_lane[ks] = lds0 + (wm * CT * 16 + j) * (CPR * 16) + (((ks * 4 + g) ^ ((j / RP) % CPR)) * 16);
    constexpr int READS = RT + CT;
    auto read_one = [&](Operands& f, unsigned buf, auto kc, auto nc) {        // the n-th read of a k-step
        constexpr int n = decltype(nc)::value, ks = decltype(kc)::value;
        if constexpr (n < CT) lds_read16<n * 16 * CPR * 16>(f.x[n], x_lane[ks] + buf);
        else lds_read16<((n - CT) * KT + ks) * 1024>(f.w[n - CT], w_lane + buf);
    };
    auto use = [&](Operands& f) {
#pragma unroll
        for (int r = 0; r < RT; ++r) lds_use(f.w[r]);
#pragma unroll
        for (int c = 0; c < CT; ++c) lds_use(f.x[c]);
    };
    // In a stage that columns are missing from, what was read in their place counts nothing, whatever it was.
    auto clear_tail = [&](Operands& f, int ks) {
        const int kb = st_last * KT + ks;
        if (kb >= KB) {
#pragma unroll
            for (int r = 0; r < RT; ++r) f.w[r].u = uint4{0, 0, 0, 0};
        }
        if (kb * 32 + g * 8 >= K) {
#pragma unroll
            for (int c = 0; c < CT; ++c) f.x[c].u = uint4{0, 0, 0, 0};
        }
    };
    // Until the loads of at most S stages of this wave's are in flight, and every wave's are as far.
    auto landed = [&](auto sc) {
        constexpr int S = decltype(sc)::value, n = S * LMAX, n1 = S * (LMAX - 1);
        if (FULL == 0 || wave < FULL) __builtin_amdgcn_s_waitcnt(0x0F70 | (n & 15) | ((n >> 4) << 14));
        else __builtin_amdgcn_s_waitcnt(0x0F70 | (n1 & 15) | ((n1 >> 4) << 14));
        __builtin_amdgcn_s_barrier();                                // (bare: __syncthreads() would wait for all loads)
    };

    // The stage loop.  Stage st lies in buffer (st - st0) % NS.  While a k-step multiplies, the next one's operands are read.
    // Every wave has its operands of a stage's second k-step in registers before it comes to the barrier in the middle of the
    // stage; from there on the stage's buffer takes stage st + NS.
    constexpr int MF = RT * CT;                                      // multiplications of a wave and k-step
    const int n = st_end - st0;
    static_for<0, NS>([&](auto s) {
        if (s.value < n) {
            if (st0 + s.value == ragged) mend_last();
            static_for<0, LMAX>([&](auto i) { fetch_one(s.value * STAGE_BYTES, i); });
            next_stage();
        }
    });
    // one k-step's multiplications, with the reads of the next one and LOADS loads into buffer buf between them
    auto multiply = [&](Operands& now, Operands& next, unsigned next_buf, auto next_ks, auto loads, unsigned buf) {
        constexpr int LD = decltype(loads)::value;
        static_for<0, MF>([&](auto mc) {
            constexpr int m = decltype(mc)::value;
            constexpr int r_lo = READS * 3 * m / (2 * MF), r_hi = READS * 3 * (m + 1) / (2 * MF);
            __builtin_amdgcn_sched_barrier(0);
            static_for<(r_lo < READS ? r_lo : READS), (m + 1 == MF ? READS : (r_hi < READS ? r_hi : READS))>(
                [&](auto n) { read_one(next, next_buf, next_ks, n); });
            __builtin_amdgcn_sched_barrier(0);
            constexpr int c = m / RT, r = m % RT;
            acc[r][c] = mfma_16x16x32(now.w[r], now.x[c], acc[r][c]);
            constexpr int l_lo = LD * m / MF, l_hi = LD * (m + 1) / MF;
            if constexpr (l_hi > l_lo) {
                __builtin_amdgcn_sched_barrier(0);
                static_for<l_lo, l_hi>([&](auto i) { fetch_one(buf, i); });
            }
        });
        __builtin_amdgcn_sched_barrier(0);
        lds_settle();
        use(next);
    };
    Operands a, b;
    unsigned buf = 0;                                                // of the stage that is being multiplied
    // a stage, with the loads of another (LMAX or none) and the loads of S stages in flight behind the next one's
    auto step = [&](int st, auto loads, auto flight) {
        constexpr bool last = decltype(loads)::value == 0;           // (one of the last NS stages)
        multiply(a, b, buf, IntC<1>{}, IntC<0>{}, 0);
        if (last && st == ragged) clear_tail(b, 1);
        const unsigned buf_next = buf == (NS - 1) * STAGE_BYTES ? 0 : buf + STAGE_BYTES;
        landed(flight);
        multiply(b, a, buf_next, IntC<0>{}, loads, buf);
        if (last && st + 1 == ragged) clear_tail(a, 0);
        buf = buf_next;
    };
    static_for<0, NS>([&](auto s) {                                  // the first stage has landed
        if (s.value + 1 == (n < NS ? n : NS)) landed(s);
    });
    static_for<0, READS>([&](auto n) { read_one(a, 0, IntC<0>{}, n); });
    lds_settle();
    use(a);
    if (st0 == ragged) clear_tail(a, 0);
    int st = st0;
    for (; st + NS < st_end; ++st) {
        if (st + NS == ragged) mend_last();
        step(st, IntC<LMAX>{}, IntC<NS - 2>{});
        next_stage();
    }
    static_for<0, NS>([&](auto s) {                                  // the last NS stages, with no loads left to ask for
        constexpr int flight = NS - 2 - s.value > 0 ? NS - 2 - s.value : 0;
        if (n >= NS - s.value) {
            step(st, IntC<0>{}, IntC<flight>{});
            ++st;
        }
    });

    // A lane holds token j of its 16 and rows 4g .. 4g+3: four consecutive outputs of one token.  The finished tile goes through
    // LDS, which is free now, and leaves it row by row in whole lines.  A row is padded by 16 bytes so that the 16 tokens of a
    // store into LDS fall into different banks.
    constexpr int ES = (int)sizeof(TC);
    constexpr int OUT_COLS = EPI == 0 ? WTILES * 16 : WTILES * 8, ROW_BYTES = OUT_COLS * ES, PITCH = ROW_BYTES + 16;
    constexpr int CH = ROW_BYTES / 16, EPC = 16 / ES;                // 16-byte pieces per row, elements per piece
    static_assert(TT * PITCH <= 160 * 1024, "the finished tile must fit the LDS");
    const int n_base = EPI == 0 ? nbw * 16 : nbw * 8;
    __builtin_amdgcn_s_barrier();                                    // every wave has read its last operands
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        unsigned char* dst = gt_lds + ((wm * CT + c) * 16 + j) * PITCH;
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const f32x4_t s = acc[r][c];
            const int tile = wn * RT + r;
            if (EPI == 0) {
                store4(reinterpret_cast<TC*>(dst) + tile * 16 + g * 4, float4{s[0], s[1], s[2], s[3]});
            } else {
                const int n = n_base + tile * 8 + g * 2;
                const float v0 = gated_at(s[0], s[2], F, n, N), v1 = gated_at(s[1], s[3], F, n + 1, N);
                *reinterpret_cast<uint32_t*>(dst + (tile * 8 + g * 2) * ES) = f32x2_to_bf16x2(v0, v1);
            }
        }
    }
    __syncthreads();
    const bool whole = (((uintptr_t)Y | (uintptr_t)(ldy * ES)) & 15) == 0;           // pieces are aligned in memory
#pragma unroll 4
    for (int i = threadIdx.x; i < TT * CH; i += 512) {
        const int t = i / CH, piece = i % CH;
        const int m = m0 + t, n = n_base + piece * EPC;
        if (m >= M || n >= N) continue;
        const uint4 v = *reinterpret_cast<const uint4*>(gt_lds + t * PITCH + piece * 16);
        TC* dst = Y + (size_t)m * ldy + n;
        if (whole && n + EPC <= N) {
            *reinterpret_cast<uint4*>(dst) = v;
        } else {
            const TC* e = reinterpret_cast<const TC*>(&v);
#pragma unroll
            for (int x = 0; x < EPC; ++x)
                if (n + x < N) dst[x] = e[x];
        }
    }
}

template <int RT, int CT, int WN, int WM, int NS, int EPI, typename TC>
static int launch_tile(const void* X, long ldx, const void* Wp, void* Y, long ldy, int M, int N, int K, int KB, int NB,
                       const GateForm& F, hipStream_t stream, int splits = 1, long part_stride = 0) {
    constexpr int TT = 16 * CT * WM, WTILES = RT * WN, KT = 2;
    constexpr size_t ring = (size_t)NS * (TT * KT * 64 + WTILES * KT * 1024);
    constexpr size_t out = (size_t)TT * ((EPI == 0 ? WTILES * 16 : WTILES * 8) * sizeof(TC) + 16);
    constexpr size_t lds = ring > out ? ring : out;
    static_assert(lds <= 160 * 1024, "the ring must fit the LDS");
    const dim3 grid((NB + WTILES - 1) / WTILES, (M + TT - 1) / TT, splits);
    AGAVE_CHECK(grid.y <= 65535, "gemm_tile: M=%d exceeds the grid limit", M);
    static bool raised = false;
    if (!raised) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_tile_kernel<RT, CT, WN, WM, NS, EPI, TC>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        AGAVE_CHECK(e == hipSuccess, "gemm_tile: cannot raise the LDS allowance");
        raised = true;
    }
    gemm_tile_kernel<RT, CT, WN, WM, NS, EPI, TC><<<grid, 512, lds, stream>>>(
        (const bf16*)X, ldx, (const uint4*)Wp, (TC*)Y, ldy, M, N, K, KB, NB, part_stride, F);
    return 0;
}
