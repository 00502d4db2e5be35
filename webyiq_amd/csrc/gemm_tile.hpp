// The 128-token tile kernel of the prefill GEMM (gemm_q4q8.hip describes it)
// and its launch, shared by the two translation units that instantiate it:
// gemm_q4q8.hip (KS = 2) and gemm_q4q8_shared.hip (KS = 1).
#pragma once

#include "common.hpp"
#include "gemm_common.hpp"
#include "launch.hpp"

#pragma clang fp contract(off)

namespace wq {
namespace {

constexpr int kBM = 128;          // tokens per tile
constexpr int kWaveGroup = 256;   // 4 waves: 2 along M x 2 along N

// Spin limit of a split-K partner's wait for the first half's partial sums
// (each poll one device-coherent load plus a short sleep; ~0.5 s, far beyond
// any launch).
constexpr unsigned kSplitSpinLimit = 1u << 22;
// s_getreg operand of HW_REG_XCC_ID (hardware register 20 on gfx940 and
// later), bits 3:0: the XCD the wave runs on
constexpr int kHwRegXccId = 20 | (0 << 6) | ((4 - 1) << 11);

// KS = 2: two groups of 4 waves run alternate K steps of the tile on a ring of
// four stages, one workgroup per CU (two waves per SIMD, so that one wave's
// fold overlaps the other's MFMAs), for grids of few tiles.  KS = 1: one group
// on two stages, two workgroups per CU, so that one tile's start (operands'
// first landing, min term), barriers and epilogue run beside the other's
// K steps, for grids of two tiles per CU and more.
template <int BN, int G, int MODE, int KS, bool DUMP>
__global__ __launch_bounds__(KS * kWaveGroup, KS == 1 ? 2 : 1) void gemm_kernel(GemmParams p) {
    constexpr int kThreads = KS * kWaveGroup;
    constexpr int BM = kBM;
    constexpr bool G32 = G == 32;            // one MFMA and one fold per group
    constexpr int NGS = kBK / G;             // groups per step
    constexpr int TM = 2;                    // 32-token subtiles per wave
    constexpr int TN = BN / 64;              // 32-row subtiles per wave
    constexpr int NST = KS == 2 ? 4 : 2;     // LDS stages
    // direct-to-LDS instructions per wave and step (4 waves share each tile)
    constexpr int A_PW = BM * kBK / 1024 / 4;          // 1 KiB activation blocks
    constexpr int B_PW = BN * (kBK / 2) / 1024 / 4;    // 1 KiB packed weight blocks
    constexpr int S_W = BN * NGS;                      // scale words per step
    constexpr int S_PW = (S_W + 255) / 256;            // 64-word blocks
    constexpr int VM = A_PW + B_PW + S_PW;
    static_assert(BN % 64 == 0 && B_PW == TN && VM < 64, "tile width");
    static_assert(TN <= 3 || (KS == 2 && !G32), "four columns: two wave groups, group 128");

    // LDS: NST stages of (activations, scale words), then the packed weights;
    // the partial sums of the second wave group reuse it at the end.  With two
    // wave groups (PAIRB) the packed weights of a round's two steps share one
    // buffer of BN rows x 128 bytes: a row's two 64-byte halves are one cache
    // line, fetched by one load, half of the rows by each group.
    constexpr bool PAIRB = KS == 2;
    constexpr int A_SZ = BM * kBK, B_SZ = BN * kBK / 2, S_SZ = S_PW * 1024;
    constexpr int OFF_S = A_SZ;
    constexpr int ST_SZ = OFF_S + S_SZ;
    constexpr int PB_BASE = NST * ST_SZ;  // pair buffers
    constexpr int RING_SZ = PB_BASE + NST * B_SZ;
    constexpr int RED_SZ = KS == 2 ? kWaveGroup * TM * TN * 16 * 4 : 0;
    constexpr int NWAVES = kThreads / 64;
    constexpr int TR_STRIDE = 36;  // floats per row of a wave's 32 x 32 output transpose (16-byte rows)
    // floats of a wave's transpose: gate/up subtiles go in pairs, the second 16
    // banks on from the first
    constexpr bool PAIRS = MODE == 2 && TN >= 2;
    constexpr int TR_SUB = 32 * TR_STRIDE + 16, TR_WAVE = PAIRS ? 2 * TR_SUB : TR_SUB;
    constexpr int TR_SZ = NWAVES * TR_WAVE * 4;
    constexpr int BODY_SZ = RING_SZ > RED_SZ ? RING_SZ : RED_SZ;
    // + the tile's per-token scales; then (per-token group-128 format) the
    // tile's scale words for the whole K range, loaded once: BN rows of NGP
    // words (NGP = NG rounded up to odd, so that 32 consecutive rows read
    // distinct banks), in what is left of the 160 KiB
    constexpr int SP_BASE = (BODY_SZ > TR_SZ ? BODY_SZ : TR_SZ) + BM * 4;
    constexpr int SP_NGP = (kLdsBytes * KS / 2 - 16 - SP_BASE) / (BN * 4);  // row words that fit (beside `ready`)
    constexpr int LDS_SZ = SP_BASE + BN * SP_NGP * 4;
    static_assert(LDS_SZ <= kLdsBytes * KS / 2 - 16, "LDS");
    __shared__ __align__(1024) unsigned char lds[LDS_SZ];
    float* dx_tile = reinterpret_cast<float*>(lds + SP_BASE - BM * 4);
    auto As = [&](int st) -> int8_t* { return reinterpret_cast<int8_t*>(lds + st * ST_SZ); };
    // packed weights of stage st: its own buffer, or (PAIRB) the pair buffer of
    // its round, the step's half selected when reading
    auto Bs = [&](int st) -> uint32_t* {
        return reinterpret_cast<uint32_t*>(lds + PB_BASE + (PAIRB ? (st >> 1) * 2 : st) * B_SZ);
    };
    auto Ss = [&](int st) -> uint32_t* { return reinterpret_cast<uint32_t*>(lds + st * ST_SZ + OFF_S); };

    const LinearArgs& a = p.a;
    pin_arg(a.wq); pin_arg(a.ws); pin_arg(a.xq); pin_arg(a.dx); pin_arg(a.xs); pin_arg(a.y);
    pin_arg(a.N); pin_arg(a.K); pin_arg(a.M); pin_arg(a.params);
    pin_arg(p.tilesM); pin_arg(p.tilesN); pin_arg(p.NG);
    if (DUMP) pin_arg(a.acc_dump);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    // wave group (K steps s with s % KS == wk) and wave within its group;
    // wave-uniform, so that every step and stage index derived from them
    // stays scalar
    const int wk = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid / kWaveGroup);
    const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
    // tokens of this call: M, or (device Params) min(p.m, M) read when the
    // kernel runs; the grid is sized for M
    int64_t M = a.M;
    if (a.params) {
        const int64_t pm = (int64_t)a.params[kParamM];
        M = pm < M ? pm : M;
    }
    const int64_t N = a.N;
    const int K = (int)a.K;
    const int NG = p.NG;  // groups per row of the weights and of the activations

    // XCD-aware tile order: consecutive tiles (same weight rows) on one XCD.
    // Only token tiles of this step are numbered, the workgroups past them
    // leave: with the empty ones interleaved, two working ones met on every
    // eighth CU while the others stood idle (102 of 1,024 tokens, K = 2048,
    // gate/up pairs N = 6144: 36.9 -> 28.3 us, group 32 72.5 -> 49.5 us; 512 of
    // 1,024 tokens 39.3 -> 31.4 and 77.3 -> 53.8 us).
    int bid = blockIdx.x, tilesM = p.tilesM;
    if (a.params) {
        tilesM = (int)((M + BM - 1) / BM);
        if (bid >= tilesM * p.tilesN * (p.split ? 2 : 1)) return;  // (uniform: nothing issued yet)
    }
    const int T = tilesM * p.tilesN;
    // Split K: workgroups T.. 2T-1 take the second half of the
    // K steps of tile bid - T; with T a multiple of 8 the pair shares an XCD.
    // (Widths up to 128 only: the exchange's registers do not fit beside the
    // wider tiles' accumulators.)
    constexpr bool SPLITOK = KS == 2 && BN <= 128;
    const bool split = SPLITOK && p.split;
    const int half = split && bid >= T ? 1 : 0;
    bid -= half * T;
    const int nsteps = split ? K / kBK / 2 : K / kBK;  // this workgroup's K steps
    const int s_begin = half * nsteps;
    const int NGL = split ? NG / 2 : NG;               // its weight groups
    const int g_begin = half * NGL;
    const int xcd = bid % kXcds, li = bid / kXcds;
    const int per = T / kXcds, rem = T % kXcds;
    const int lt = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + li;
    // tiles in groups of GM token tiles: the run of consecutive tiles one
    // XCD takes spans GM token tiles x (run / GM) row tiles, so that for long
    // rows (K >= 4096, 128 tokens x K bytes per token tile) or long prompts
    // its L2 holds the activations of 4 token tiles rather than of all of them
    // (M = 4096, K = 2048, gate/up pairs N = 6144: 172.8 -> 165.7 us); others
    // keep every token tile of a row tile together (GM = tilesM)
    const int GM = K >= 4096 || tilesM > 8 ? 4 : tilesM;
    const int grp = lt / (GM * p.tilesN);
    const int gm = tilesM - grp * GM < GM ? tilesM - grp * GM : GM;
    const int off = lt - grp * GM * p.tilesN;
    const int tile_m = grp * GM + off % gm, tile_n = off / gm;
    const int64_t m0 = (int64_t)tile_m * BM;
    constexpr int OUTW = MODE == 2 ? BN / 2 : BN;  // output columns per tile
    const int64_t n0 = (int64_t)tile_n * OUTW;

    // weight row of tile row r (mode 2: each subtile of 32 holds 16 gate rows,
    // then the same outputs' 16 up rows)
    auto wrow = [&](int r) -> int64_t {
        int64_t n = n0 + (MODE == 2 ? 16 * (r >> 5) + (r & 15) : r);
        n = n < N ? n : N - 1;
        return MODE == 2 && (r & 16) ? n + N : n;
    };
    auto trow = [&](int r) -> int64_t {
        int64_t t = m0 + r;
        return t < M ? t : M - 1;
    };

    // ---------------- staging: per-lane source offsets ----------------
    // A direct-to-LDS instruction writes 64 consecutive 16-byte (or 4-byte)
    // slots, lane l the l-th; each lane fetches whatever belongs in its slot.
    uint32_t a_off[A_PW], b_off[B_PW], s_off[S_PW];
#pragma unroll
    for (int i = 0; i < A_PW; ++i) {  // block = 8 rows of 128 B
        const int r = 8 * (A_PW * wave + i) + lane / 8;
        a_off[i] = (uint32_t)(trow(r) * K + 16 * ((lane % 8) ^ swz_a(r)));
    }
#pragma unroll
    for (int i = 0; i < B_PW; ++i) {
        if constexpr (PAIRB) {  // block = 8 rows of 128 B; the 8 waves cover BN rows
            const int r = 8 * ((4 * wk + wave) * B_PW + i) + lane / 8;
            b_off[i] = (uint32_t)(wrow(r) * (K / 2) + 16 * ((lane % 8) ^ swz_p(r)));
        } else {  // block = 16 rows of 64 B
            const int r = 16 * (B_PW * wave + i) + lane / 4;
            b_off[i] = (uint32_t)(wrow(r) * (K / 2) + 16 * ((lane % 4) ^ swz_b(r)));
        }
    }
#pragma unroll
    for (int i = 0; i < S_PW; ++i) {  // block = 64 scale words, [row][group]
        int w = 64 * (S_PW * wave + i) + lane;
        w = w < S_W ? w : 0;  // padding slots re-read word 0
        s_off[i] = (uint32_t)(wrow(w / NGS) * NG + w % NGS);
    }
    // The scale words of every K step at once when they fit (the per-token
    // group-128 format) and the row has 32 steps or more: each step
    // otherwise fetches BN scattered 4-byte words, one cache-line request
    // each.  Measured: K = 6144, N = 2048 27.08 -> 25.49 us; at K = 2048 (16
    // steps) the preload's start-up cost outweighs it, 22.31 -> 22.65 us, where
    // no second workgroup covers it.
    const int NGPs = NGL + 1 - (NGL & 1);  // odd row stride
    // (the last 64-word instruction may run up to 63 words past BN rows)
    const bool spre = !G32 && (KS == 1 || nsteps >= 32) && BN * NGPs + 64 <= BN * SP_NGP;  // uniform
    const uint32_t* sp_lds = reinterpret_cast<const uint32_t*>(lds + SP_BASE);
    // Every load is unconditional (steps past the end re-read the last one),
    // so each call issues the same vector-memory instructions per wave.
    // LDS byte address of the ring (scalar); stage st, part at byte b of it
    const uint32_t lds0 = lds_addr(lds);
    auto stage_at = [&](int st, int b) -> uint32_t { return lds0 + (uint32_t)(st * ST_SZ + b); };
    auto dma = [&](int step, const int st) {
        step = step < nsteps ? step : nsteps - 1;
        const int8_t* xq = a.xq + (s_begin + step) * kBK;
        const uint32_t* ws = a.ws + (s_begin + step) * NGS;
#pragma unroll
        for (int i = 0; i < A_PW; ++i) dma16_at(xq, a_off[i], stage_at(st, 1024 * (A_PW * wave + i)));
        if constexpr (PAIRB) {
            // steps s0 and s0 + 1 into the pair buffer of stage st; with an
            // odd step count the last round has no second step, and the lanes
            // of the second halves re-read the first (a row's end is not
            // passed): the half of a lane's chunk is bit 2 of
            // (lane % 8) ^ swz_p(r), = ((lane >> 2) ^ block) & 1
            const int s0 = step & ~1;
            const uint8_t* wq = reinterpret_cast<const uint8_t*>(a.wq) + (s_begin + s0) * (kBK / 2);
            const bool tail = s0 + 1 >= nsteps;  // uniform
#pragma unroll
            for (int i = 0; i < B_PW; ++i) {
                const int blk = (4 * wk + wave) * B_PW + i;
                const uint32_t off = tail ? b_off[i] - 64u * (uint32_t)(((lane >> 2) ^ blk) & 1) : b_off[i];
                dma16_at(wq, off, lds0 + (uint32_t)(PB_BASE + (st >> 1) * 2 * B_SZ + 1024 * blk));
            }
        } else {
            const uint8_t* wq = reinterpret_cast<const uint8_t*>(a.wq) + (s_begin + step) * (kBK / 2);
#pragma unroll
            for (int i = 0; i < B_PW; ++i)
                dma16_at(wq, b_off[i], lds0 + (uint32_t)(PB_BASE + st * B_SZ + 1024 * (B_PW * wave + i)));
        }
        if (!spre) {
#pragma unroll
            for (int i = 0; i < S_PW; ++i)
                dma4_at(ws, 4 * s_off[i], stage_at(st, OFF_S + 256 * (S_PW * wave + i)));
        }
    };

    // ---------------- compute layout ----------------
    const int wm = wave >> 1, wn = wave & 1;
    const int l32 = lane & 31, h = lane >> 5;
    // tile row (of W) of this lane's column in subtile j
    auto bcol = [&](int j) -> int { return wn * (BN / 2) + 32 * j + l32; };
    // token row (within the tile) of accumulator element r of subtile i
    auto arow = [&](int i, int r) -> int { return wm * 64 + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3); };

    // min term operands: blocks of 8 groups, wave group wk taking blocks
    // wk, wk + KS, ... (the groups' partial sums are added at the end like
    // their K steps'), with NSL blocks in flight per wave in registers: two
    // up to 2 columns per wave, one at 3.  The first NSL are requested
    // before any tile load: loads return in issue order, so operands
    // requested after the tiles would land after them.  With 4 columns the
    // registers are short: wave group 0 loads each block after the tiles,
    // when it is used.
    constexpr int NSL = TN <= 2 ? 2 : TN == 3 ? 1 : 0;
    constexpr int NSA = NSL > 0 ? NSL : 1;  // register slots
    // (with split K, this workgroup's groups g_begin .. g_begin + NGL - 1)
    const int nfull = NGL % 8 == 0 ? NGL / 8 : 0;  // full blocks (32-byte aligned rows: K a multiple of 1024)
    const int nblk = (NGL + 7) / 8;
    const int32_t* xr[TM];
    const uint32_t* sr[TN];
    int32_t xv[NSA][TM][8];
    uint32_t wv[NSA][TN][8];
    auto mt_full = [&](int32_t (&x)[TM][8], uint32_t (&w)[TN][8], int blk) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int4 lo = *reinterpret_cast<const int4*>(xr[i] + 8 * blk);
            const int4 hi = *reinterpret_cast<const int4*>(xr[i] + 8 * blk + 4);
            x[i][0] = lo.x; x[i][1] = lo.y; x[i][2] = lo.z; x[i][3] = lo.w;
            x[i][4] = hi.x; x[i][5] = hi.y; x[i][6] = hi.z; x[i][7] = hi.w;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const uint4 lo = *reinterpret_cast<const uint4*>(sr[j] + 8 * blk);
            const uint4 hi = *reinterpret_cast<const uint4*>(sr[j] + 8 * blk + 4);
            w[j][0] = lo.x; w[j][1] = lo.y; w[j][2] = lo.z; w[j][3] = lo.w;
            w[j][4] = hi.x; w[j][5] = hi.y; w[j][6] = hi.z; w[j][7] = hi.w;
        }
    };
    // word by word, indices past the last group clamped (their values are zeroed)
    auto mt_words = [&](int32_t (&x)[TM][8], uint32_t (&w)[TN][8], int blk) {
        const int b = 8 * blk;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int u = 0; u < 8; ++u) x[i][u] = xr[i][b + u < NGL ? b + u : NGL - 1];
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int u = 0; u < 8; ++u) w[j][u] = sr[j][b + u < NGL ? b + u : NGL - 1];
    };
    auto mt_load = [&](auto slot, int blk) {
        constexpr int S = decltype(slot)::value;
        if (blk < nfull) mt_full(xv[S], wv[S], blk);
        else mt_words(xv[S], wv[S], blk);
    };
    using ic0 = std::integral_constant<int, 0>;
    using ic1 = std::integral_constant<int, NSA - 1>;
    auto mt_rows = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i) xr[i] = a.xs + trow(wm * 64 + 32 * i + l32) * NG + g_begin;
#pragma unroll
        for (int j = 0; j < TN; ++j) sr[j] = a.ws + wrow(bcol(j)) * NG + g_begin;
    };
    if constexpr (NSL >= 1) {
        mt_rows();
        if (wk < nblk) mt_load(ic0{}, wk);
        if constexpr (NSL == 2)
            if (wk + KS < nblk) mt_load(ic1{}, wk + KS);
    }

    if (spre) {  // 64 words per instruction, the workgroup's waves in turn
        const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int nins = (BN * NGPs + 63) / 64;
        for (int i = wid; i < nins; i += NWAVES) {
            const int pw = 64 * i + lane;
            const int r = pw / NGPs, gg = pw - r * NGPs;
            const uint32_t src = r < BN && gg < NGL ? (uint32_t)(wrow(r) * NG + g_begin + gg) : 0u;  // padding: word 0
            dma4_at(a.ws, 4 * src, lds0 + (uint32_t)(SP_BASE + 256 * i));
        }
    }
    // the tile's per-token scales for the epilogue, ahead of the ring loads
    // (every wait below also covers them)
    if (wave < BM / 64 && wk == 0)
        dma4(a.dx, 4 * (uint32_t)trow(64 * wave + lane), dx_tile + 64 * wave);

    dma(wk, wk);  // each group's first step
    if (KS == 1 && nsteps > 1) dma(1, 1);

    v16f facc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) facc[i][j] = v16f{};

    // min term: facc += sum_g m[n,g] * X[t,g] (per-token group-128 format
    // only) on v_mfma_f32_32x32x16_f16.  One MFMA covers 8 groups: lane half
    // h = 0 holds (64 X_hi, m), h = 1 (X_lo, m) of groups b .. b+7, both
    // halves of a row reading the same 32 bytes.
    auto min_term_block = [&](const int32_t (&xv)[TM][8], const uint32_t (&wv)[TN][8], int b) {
        v8h xa[TM], mb[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int32_t v = b + u < NGL ? xv[i][u] : 0;
                xa[i][u] = (_Float16)(h == 0 ? (float)((v >> 6) * 64) : (float)(v & 63));
            }
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int u = 0; u < 8; ++u)
                mb[j][u] = b + u < NGL ? __builtin_bit_cast(_Float16, (unsigned short)(wv[j][u] >> 16))
                                      : (_Float16)0.0f;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                facc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xa[i], mb[j], facc[i][j], 0, 0, 0);
    };
    // this wave group's min term blocks, the two register slots in turn
    if constexpr (NSL == 0) {  // wave group 0 alone, block by block
        if (wk == 0) {
            mt_rows();
            for (int blk = 0; blk < nfull; ++blk) {
                int32_t x[TM][8];
                uint32_t w[TN][8];
                mt_full(x, w, blk);
                min_term_block(x, w, 8 * blk);
            }
            for (int blk = nfull; blk < nblk; ++blk) {
                int32_t x[TM][8];
                uint32_t w[TN][8];
                mt_words(x, w, blk);
                min_term_block(x, w, 8 * blk);
            }
        }
    } else if constexpr (NSL == 1) {
        for (int blk = wk; blk < nblk; blk += KS) {
            min_term_block(xv[0], wv[0], 8 * blk);
            if (blk + KS < nblk) mt_load(ic0{}, blk + KS);
        }
    } else {
        for (int blk = wk; blk < nblk; blk += 2 * KS) {
            min_term_block(xv[0], wv[0], 8 * blk);
            if (blk + 2 * KS < nblk) mt_load(ic0{}, blk + 2 * KS);
            if (blk + KS >= nblk) break;
            min_term_block(xv[NSA - 1], wv[NSA - 1], 8 * (blk + KS));
            if (blk + 3 * KS < nblk) mt_load(ic1{}, blk + 3 * KS);
        }
    }

    if (KS == 2) step_barrier<0>();  // the first step of each group has landed

    const int rows_total = MODE == 2 ? 2 * (int)N : (int)N;
    auto dump = [&](int step, int e_local, int i, int br, const v16i& acc) {
        const int64_t e = (int64_t)(s_begin + step) * NGS + e_local;
        const int64_t nn = n0 + (MODE == 2 ? 16 * (br >> 5) + (br & 15) : br);
        const int64_t wr = MODE == 2 && (br & 16) ? nn + N : nn;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t t = m0 + arow(i, r);
            if (t < M && nn < N) a.acc_dump[(t * rows_total + wr) * NG + e] = acc[r];
        }
    };

    // release() is called when this wave has read all it needs of the stage
    // into registers (KS = 1)
    auto compute = [&](const int step, const int st, auto release) __attribute__((always_inline)) {
        const int8_t* Ab = As(st);
        const uint8_t* Bb = reinterpret_cast<const uint8_t*>(Bs(st));
        // 16-byte chunk c (of 4) of this step's packed weights in tile row br
        auto bfrag = [&](int br, int c) -> uint4 {
            if constexpr (PAIRB)
                return *reinterpret_cast<const uint4*>(Bb + br * 128 + 16 * ((4 * (st & 1) + c) ^ swz_p(br)));
            else
                return *reinterpret_cast<const uint4*>(Bb + br * 64 + 16 * (c ^ swz_b(br)));
        };
        const uint32_t* Sb = Ss(st);
        // scale word of tile row br for this step: Sx[br * sst]
        const uint32_t* Sx = spre ? sp_lds + step : Sb;
        const int sst = spre ? NGPs : 1;
        // k-slice ks of lane half h = codes 64 h + 16 ks .. +15 of the
        // group (any assignment shared by both operands gives the same
        // sums): 32 contiguous packed bytes per lane and weight row.
        // Group 32: k-slice ks = group ks, lane half h its codes
        // 32 ks + 16 h .. +15, so that each MFMA sums one group.
        v4i af[4][TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int ra = wm * 64 + 32 * i + l32;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                af[ks][i] = *reinterpret_cast<const v4i*>(
                    Ab + ra * kBK + 16 * ((G32 ? 2 * ks + h : 4 * h + ks) ^ swz_a(ra)));
        }
        // (group 32) the 8 packed bytes of group c, lane half h, in tile row br
        auto bhalf = [&](int br, int c) -> uint2 {
            if constexpr (PAIRB)
                return *reinterpret_cast<const uint2*>(Bb + br * 128 + 16 * ((4 * (st & 1) + c) ^ swz_p(br)) + 8 * h);
            else
                return *reinterpret_cast<const uint2*>(Bb + br * 64 + 16 * (c ^ swz_b(br)) + 8 * h);
        };
        auto bload = [&](int br, uint4& p0, uint4& p1) {
            if constexpr (G32) {
                const uint2 q0 = bhalf(br, 0), q1 = bhalf(br, 1), q2 = bhalf(br, 2), q3 = bhalf(br, 3);
                p0 = uint4{q0.x, q0.y, q1.x, q1.y};
                p1 = uint4{q2.x, q2.y, q3.x, q3.y};
            } else {
                p0 = bfrag(br, 2 * h);
                p1 = bfrag(br, 2 * h + 1);
            }
        };
        // up to 3 columns: every column's packed weight fragment is read up
        // front (one LDS latency per step instead of one per column), with
        // one wave group the scale words too: the stage is then free for the
        // next loads
        constexpr bool PRE = TN <= 3;
        uint4 pb[PRE ? TN : 1][2];
        float sv[PRE ? TN : 1];
        if constexpr (PRE) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int br = bcol(j);
                bload(br, pb[j][0], pb[j][1]);
                if constexpr (KS == 2 && !G32) sv[j] = f16lo(Sx[br * sst]);
            }
        }
        constexpr bool SUP = KS == 1;
        uint32_t su[SUP ? TN : 1][NGS];
        if constexpr (SUP) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if constexpr (G32) {
                    const uint4 v = *reinterpret_cast<const uint4*>(Sb + bcol(j) * NGS);
                    su[j][0] = v.x; su[j][1] = v.y; su[j][2] = v.z; su[j][3] = v.w;
                } else {
                    su[j][0] = Sx[bcol(j) * sst];
                }
            }
            release();
        }
        // 16 of column j's codes per lane: k-slice ks (group 32: group ks)
        auto expand = [&](int j, int ks) -> v4i {
            const uint4& q = pb[PRE ? j : 0][ks >> 1];
            return (ks & 1) ? expand8(q.z, q.w) : expand8(q.x, q.y);
        };
        // A scale as an f32 register: from its f16 form the compiler makes the
        // fold a v_fma_mix_f32, which issues at half the rate of v_fmac_f32
        // when two waves share the SIMD (4.6 against 2.5-3.3 clocks).  (The
        // group-128 loop of two wave groups, whose waves meet at every
        // barrier, measured the same or slower with it: K = 6144, N = 2048 at
        // M = 2048 40.7 -> 42.0 us.)
        auto scale = [](uint32_t w) {
            float v = f16lo(w);
            asm volatile("" : "+v"(v));
            return v;
        };
        if constexpr (G32) {
            // Units of one MFMA (column j, group g, subtile row i), each
            // followed by the fold of the unit before it, so that the VALU
            // never waits for the MFMA just issued.  (Units as compile-time
            // indices: a run-time index would put the arrays in scratch.)
            constexpr int NU = TN * 4 * TM;
            v16i acc[2];
            uint32_t sw = SUP ? su[0][0] : Sb[bcol(0) * NGS];  // the next group's scale word
            float sc[2];
            v4i bf;
            auto fold = [&](auto uc) __attribute__((always_inline)) {
                constexpr int u = decltype(uc)::value, j = u / (4 * TM), g = u / TM % 4, i = u % TM;
                if (DUMP) dump(step, g, i, bcol(j), acc[u & 1]);
#pragma unroll
                for (int r = 0; r < 16; ++r) facc[i][j][r] = fmaf(sc[u / TM & 1], (float)acc[u & 1][r], facc[i][j][r]);
            };
            static_for<0, NU>([&](auto uc) __attribute__((always_inline)) {
                constexpr int u = decltype(uc)::value, j = u / (4 * TM), g = u / TM % 4, i = u % TM;
                if constexpr (i == 0) {
                    bf = expand(j, g);
                    sc[u / TM & 1] = scale(sw);
                    if constexpr (g < 3) sw = SUP ? su[SUP ? j : 0][g + 1] : Sb[bcol(j) * NGS + g + 1];
                    else if constexpr (j + 1 < TN) sw = SUP ? su[SUP ? j + 1 : 0][0] : Sb[bcol(j + 1) * NGS];
                }
                acc[u & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[g][i], bf, v16i{}, 0, 0, 0);
                if constexpr (u > 0) fold(std::integral_constant<int, u - 1>{});
            });
            fold(std::integral_constant<int, NU - 1>{});
        } else if constexpr (KS == 2) {
            // a column's MFMAs, then its fold (columns as compile-time
            // indices: a run-time index would put the arrays in scratch)
            static_for<0, TN>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                const int br = bcol(j);
                uint4 p0, p1;
                if constexpr (PRE) {
                    p0 = pb[j][0];
                    p1 = pb[j][1];
                } else {
                    bload(br, p0, p1);
                }
                v16i ac[TM];
                const v4i bf[4] = {expand8(p0.x, p0.y), expand8(p0.z, p0.w), expand8(p1.x, p1.y),
                                   expand8(p1.z, p1.w)};
#pragma unroll
                for (int ks = 0; ks < 4; ++ks)
#pragma unroll
                    for (int i = 0; i < TM; ++i)
                        ac[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[ks][i], bf[ks], ks == 0 ? v16i{} : ac[i], 0, 0, 0);
                const float s = PRE ? sv[PRE ? j : 0] : f16lo(Sx[br * sst]);
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    if (DUMP) dump(step, 0, i, br, ac[i]);
#pragma unroll
                    for (int r = 0; r < 16; ++r) facc[i][j][r] = fmaf(s, (float)ac[i][r], facc[i][j][r]);
                }
            });
        } else {
            // Units of four chained MFMAs (column j, subtile row i); between
            // them the fold of the unit before and, beside a column's last
            // unit, the next column's expansion.  The two subtile rows share
            // no registers, so one folds while the other multiplies (M = 4096,
            // K = 2048, N = 6144 pairs: 159 us, column by column 164 us).
            constexpr int NU = TN * TM;
            v16i acc[2];
            v4i bf[2][4];
            float sc[2];
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) bf[0][ks] = expand(0, ks);
            uint32_t sw = su[0][0];
            sc[0] = scale(sw);
            auto fold4 = [&](auto uc, int ks) __attribute__((always_inline)) {
                constexpr int u = decltype(uc)::value, j = u / TM, i = u % TM;
                if (DUMP && ks == 0) dump(step, 0, i, bcol(j), acc[u & 1]);
#pragma unroll
                for (int r = 4 * ks; r < 4 * ks + 4; ++r)
                    facc[i][j][r] = fmaf(sc[j & 1], (float)acc[u & 1][r], facc[i][j][r]);
            };
            static_for<0, NU>([&](auto uc) __attribute__((always_inline)) {
                constexpr int u = decltype(uc)::value, j = u / TM, i = u % TM;
                if constexpr (i == 0 && j + 1 < TN) {
                    sw = su[j + 1][0];
                }
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    acc[u & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[ks][i], bf[j & 1][ks],
                                                                      ks == 0 ? v16i{} : acc[u & 1], 0, 0, 0);
                    if constexpr (u > 0) fold4(std::integral_constant<int, u - 1>{}, ks);
                    if constexpr (i == TM - 1 && j + 1 < TN) bf[(j + 1) & 1][ks] = expand(j + 1, ks);
                }
                if constexpr (i == TM - 1 && j + 1 < TN) sc[(j + 1) & 1] = scale(sw);
            });
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) fold4(std::integral_constant<int, NU - 1>{}, ks);
        }
    };

    if constexpr (KS == 1) {
        // step s: its loads have landed (those of step s + 1 stay in flight);
        // every wave reads its fragments, then the loads of step s + 2 go
        // into the stage they leave
        auto one = [&](auto stage, const int s) __attribute__((always_inline)) {
            if (s + 1 < nsteps) {
                if (spre) step_barrier<VM - S_PW>();
                else step_barrier<VM>();
            } else {
                step_barrier<0>();
            }
            compute(s, stage, [&]() __attribute__((always_inline)) {
                step_barrier<63>();
                if (s + 2 < nsteps) dma(s + 2, stage);
            });
        };
        for (int s = 0; s < nsteps; s += 2) {
            one(std::integral_constant<int, 0>{}, s);
            if (s + 1 >= nsteps) break;
            one(std::integral_constant<int, 1>{}, s + 1);
        }
    } else {
        // round r: group wk loads step 2r + 2 + wk into the stage that its
        // step 2r - 2 + wk left and computes step 2r + wk; both steps of the
        // next round land before the barrier.  A group only ever uses stages
        // wk and wk + 2, so (up to 3 columns per wave) rounds run in pairs
        // with the stage parity fixed at compile time: each fragment address
        // is then a loop-invariant lane address plus a constant (the
        // instruction's offset field), not a per-step addition.
        if constexpr (TN <= 3) {
            auto round = [&](auto parity, int r) __attribute__((always_inline)) {
                constexpr int P = decltype(parity)::value;
                const int sl = 2 * r + 2 + wk, sc = 2 * r + wk;
                dma(sl, wk + 2 * (1 - P));
                if (sc < nsteps) compute(sc, wk + 2 * P, [] {});
                step_barrier<0>();
            };
            for (int r = 0; 2 * r < nsteps; r += 2) {
                round(std::integral_constant<int, 0>{}, r);
                if (2 * (r + 1) >= nsteps) break;
                round(std::integral_constant<int, 1>{}, r + 1);
            }
        } else {  // wider tiles: no registers for the extra lane addresses
            for (int r = 0; KS * r < nsteps; ++r) {
                const int sl = KS * r + KS + wk, sc = KS * r + wk;
                dma(sl, sl % NST);
                if (sc < nsteps) compute(sc, sc % NST, [] {});
                step_barrier<0>();
            }
        }
    }
    // no direct-to-LDS load may outlive the workgroup
    step_barrier<0>();

    if constexpr (KS == 2) {
        // group g stores subtile row i = g after adding the other group's partial
        // sums (exchanged through LDS, 16 bytes per lane and instruction,
        // lane-major; the fp32 addition of two partials is the same in either
        // order)
        static_assert(TM == 2, "one subtile row per wave group");
        v4f* red = reinterpret_cast<v4f*>(lds);
        const int give = 1 - wk;  // the subtile row the other group stores
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                v4f v;
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = wk == 0 ? facc[1][j][4 * q + u] : facc[0][j][4 * q + u];
                red[(((give * 4 + wave) * TN + j) * 4 + q) * 64 + lane] = v;
            }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const v4f o = red[(((wk * 4 + wave) * TN + j) * 4 + q) * 64 + lane];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int r = 4 * q + u;
                    if (wk == 0) facc[0][j][r] = facc[0][j][r] + o[u];
                    else facc[1][j][r] = o[u] + facc[1][j][r];
                }
            }
    }

    // Split K: the first half's workgroup hands its partial sums (this
    // thread's subtile row wk, every column) to its partner through the
    // workspace and ends; the partner adds them to its own, first half
    // first (one fixed order), and runs the epilogue.  The partial stores
    // and loads are agent-scope atomics (sc1: performed at the device's
    // coherence point, past a non-coherent L2), so the same argument as the
    // lm_head argmax combine orders them without a release fence: the
    // stores are complete (vmcnt 0) in every wave before the barrier, the
    // flag is set after it, and the partner's loads are issued after its
    // poll has seen the flag.  The partner waits only for a workgroup of
    // lower index (dispatched before it, waiting for nothing), and the wait
    // is bounded: if it ran out, the tile's outputs are written as NaN.
    if constexpr (SPLITOK) {
        if (split) {
            // this thread's values, subtile row wk, as 4 x TN 16-byte chunks
            // (compile-time indices only: a run-time index would put facc in
            // scratch memory); chunk c of this thread at slot[c * 64]
            static_assert(TN <= 2, "the exchange holds 8 chunks in flight");
            v4f* slot = reinterpret_cast<v4f*>(p.part) + (size_t)lt * (BM * BN / 4) +
                        (size_t)(tid >> 6) * (TN * 4 * 64) + lane;
            unsigned int* flag = p.flags + (size_t)lt * 16;
            // the XCD this workgroup runs on (gfx950 XCC_ID, bits 3:0)
            const unsigned xcc = __builtin_amdgcn_s_getreg(kHwRegXccId) & 15u;
            if (half == 0) {
                // written through to the device's coherence point (sc1, the
                // agent-scope store), each 64 lanes' chunks 1 KiB contiguous
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        v4f v;
#pragma unroll
                        for (int u = 0; u < 4; ++u) v[u] = wk == 0 ? facc[0][j][4 * q + u] : facc[1][j][4 * q + u];
                        asm volatile("global_store_dwordx4 %0, %1, off sc1" ::"v"(slot + (j * 4 + q) * 64), "v"(v)
                                     : "memory");
                    }
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every partial store of this wave has completed
                __syncthreads();
                // the flag tells the partner where the sums were written from
                if (tid == 0)
                    __hip_atomic_store(flag, 1u + xcc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return;
            }
            __shared__ unsigned int ready;
            if (tid == 0) {
                unsigned spins = 0;
                unsigned v = 0;
                while ((v = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0 &&
                       ++spins < kSplitSpinLimit)
                    __builtin_amdgcn_s_sleep(1);
                ready = v;
                if (v) __hip_atomic_store(flag, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
            const unsigned rv = ready;
            // All 4 TN chunks in flight at once.  From the partner's own XCD
            // the sums are in this L2 (a write-through store updates it):
            // loads that skip only the CU's cache (sc0); from another XCD,
            // loads at the coherence point (sc1, the agent-scope load).
            // (One statement issues the loads and waits for them, so that no
            // destination register is read or moved before its data landed.)
            v4f buf[8];
            const v4f* s0 = slot;
            const v4f* s1 = slot + 4 * 64;  // chunks 4..7: 4 KiB on (immediate offsets stop at 4095)
#define WQ_LOAD4(CP, O0, O1, O2, O3, B)                               \
    "global_load_dwordx4 %" #O0 ", %" #B ", off " CP "\n\t"           \
    "global_load_dwordx4 %" #O1 ", %" #B ", off offset:1024 " CP "\n\t" \
    "global_load_dwordx4 %" #O2 ", %" #B ", off offset:2048 " CP "\n\t" \
    "global_load_dwordx4 %" #O3 ", %" #B ", off offset:3072 " CP "\n\t"
            if constexpr (TN == 1) {
                if (rv == 1u + xcc)
                    asm volatile(WQ_LOAD4("sc0", 0, 1, 2, 3, 4) "s_waitcnt vmcnt(0)"
                                 : "=&v"(buf[0]), "=&v"(buf[1]), "=&v"(buf[2]), "=&v"(buf[3])
                                 : "v"(s0)
                                 : "memory");
                else
                    asm volatile(WQ_LOAD4("sc1", 0, 1, 2, 3, 4) "s_waitcnt vmcnt(0)"
                                 : "=&v"(buf[0]), "=&v"(buf[1]), "=&v"(buf[2]), "=&v"(buf[3])
                                 : "v"(s0)
                                 : "memory");
            } else {
                if (rv == 1u + xcc)
                    asm volatile(WQ_LOAD4("sc0", 0, 1, 2, 3, 8) WQ_LOAD4("sc0", 4, 5, 6, 7, 9) "s_waitcnt vmcnt(0)"
                                 : "=&v"(buf[0]), "=&v"(buf[1]), "=&v"(buf[2]), "=&v"(buf[3]), "=&v"(buf[4]),
                                   "=&v"(buf[5]), "=&v"(buf[6]), "=&v"(buf[7])
                                 : "v"(s0), "v"(s1)
                                 : "memory");
                else
                    asm volatile(WQ_LOAD4("sc1", 0, 1, 2, 3, 8) WQ_LOAD4("sc1", 4, 5, 6, 7, 9) "s_waitcnt vmcnt(0)"
                                 : "=&v"(buf[0]), "=&v"(buf[1]), "=&v"(buf[2]), "=&v"(buf[3]), "=&v"(buf[4]),
                                   "=&v"(buf[5]), "=&v"(buf[6]), "=&v"(buf[7])
                                 : "v"(s0), "v"(s1)
                                 : "memory");
            }
#undef WQ_LOAD4
            const bool timed_out = rv == 0;
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int r = 4 * q + u;
                        const float v = timed_out ? __builtin_nanf("") : buf[j * 4 + q][u];
                        if (wk == 0) facc[0][j][r] = v + facc[0][j][r];
                        else facc[1][j][r] = v + facc[1][j][r];
                    }
        }
    }

    // epilogue: per-token scale and output mode in registers, then each
    // 32 x 32 subtile goes through a per-wave LDS transpose so that every lane
    // stores 16 consecutive bytes of a row (8 lanes cover a 128-byte row
    // segment) instead of single words down a column.  In mode 2 a subtile
    // gives 16 outputs per row, half a segment: two adjacent ones are stored
    // together, since half lines written one after the other cost the memory
    // more (gate/up pairs, M = 8192, K = 768, N = 1000 41.9 -> 37.8 us, K = 256
    // 29.8 -> 27.0, M = 4096, K = 1024, N = 3074 68.2 -> 64.3, M = 4096,
    // K = 2048, N = 6144 154.1 -> 151.3).
    __syncthreads();  // the ring and the exchange area are free again
    float* tr = reinterpret_cast<float*>(lds) + (tid >> 6) * TR_WAVE;
    const bool vec_ok = (reinterpret_cast<uintptr_t>(a.y) & 15) == 0 && (N & 3) == 0;  // 16-byte rows chunks
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        if (KS == 2 && i != wk) continue;
        float dtok[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) dtok[r] = dx_tile[arow(i, r)];
        // subtiles j .. j + n - 1
        auto store = [&](auto jc, auto nc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value, n = decltype(nc)::value;
#pragma unroll
            for (int s = 0; s < n; ++s)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    tr[s * TR_SUB + (8 * (r >> 2) + 4 * h + (r & 3)) * TR_STRIDE + l32] = facc[i][j + s][r] * dtok[r];
            __builtin_amdgcn_wave_barrier();  // LDS operations of a wave complete in order
            // a lane's four outputs of a row: 8 lanes cover a row's 32 columns,
            // in mode 2 4 lanes the 16 gate/up pairs of a subtile
            constexpr int LPR = MODE == 2 ? 4 * n : 8, RPP = 64 / LPR, NP = 32 / RPP;
            const int lc = lane % LPR;
            const float* own = MODE == 2 ? tr + (lc >> 2) * TR_SUB + 4 * (lc & 3) : tr + 4 * lc;
            // first output column (formed from bcol: the other form of the same
            // value left the 256-wide loop's MFMAs in one clump, 72 -> 76 us
            // at M = 4096, K = 6144, N = 2048)
            int64_t c0 = n0 + bcol(j) - l32 + 4 * lc;
            if (MODE == 2) c0 = n0 + ((bcol(j) - l32) >> 1) + 4 * lc;
            float4 o[NP], yo4[NP];
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                const float* row = own + (RPP * q + lane / LPR) * TR_STRIDE;
                o[q] = *reinterpret_cast<const float4*>(row);
                if (MODE == 2) {
                    const float4 u = *reinterpret_cast<const float4*>(row + 16);
                    o[q].x = silu_mul(o[q].x, u.x);
                    o[q].y = silu_mul(o[q].y, u.y);
                    o[q].z = silu_mul(o[q].z, u.z);
                    o[q].w = silu_mul(o[q].w, u.w);
                }
            }
            if (MODE == 1) {
#pragma unroll
                for (int q = 0; q < NP; ++q) {
                    const int64_t t = m0 + wm * 64 + 32 * i + RPP * q + lane / LPR;
                    yo4[q] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (t < M && vec_ok && c0 + 3 < N) yo4[q] = *reinterpret_cast<const float4*>(a.y + t * N + c0);
                }
            }
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                const int64_t t = m0 + wm * 64 + 32 * i + RPP * q + lane / LPR;
                if (t >= M) continue;
                float* yp = a.y + t * N + c0;
                if (vec_ok && c0 + 3 < N) {
                    float4 v = o[q];
                    if (MODE == 1) {
                        v.x = yo4[q].x + v.x;
                        v.y = yo4[q].y + v.y;
                        v.z = yo4[q].z + v.z;
                        v.w = yo4[q].w + v.w;
                    }
                    // streamed: the output is not re-read here, and lines left
                    // dirty in L2 would be written back at the end of the kernel
                    __builtin_nontemporal_store(v4f{v.x, v.y, v.z, v.w}, reinterpret_cast<v4f*>(yp));
                } else {
                    const float vv[4] = {o[q].x, o[q].y, o[q].z, o[q].w};
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (c0 + u < N) yp[u] = MODE == 1 ? yp[u] + vv[u] : vv[u];
                }
            }
            __builtin_amdgcn_wave_barrier();
        };
        constexpr int JS = PAIRS ? 2 : 1;
        static_for<0, TN / JS>([&](auto b) __attribute__((always_inline)) {
            store(std::integral_constant<int, JS * decltype(b)::value>{}, std::integral_constant<int, JS>{});
        });
        if constexpr (TN % JS != 0) store(std::integral_constant<int, TN - 1>{}, std::integral_constant<int, 1>{});
    }
}

template <int BN, int G, int KS, bool DUMP>
hipError_t launch_mode(const GemmParams& gp, hipStream_t s) {
    dim3 grid((unsigned)(gp.tilesM * gp.tilesN * (gp.split ? 2 : 1))), block(KS * kWaveGroup);
    switch (gp.a.mode) {
        case 0: hipLaunchKernelGGL((gemm_kernel<BN, G, 0, KS, DUMP>), grid, block, 0, s, gp); break;
        case 1: hipLaunchKernelGGL((gemm_kernel<BN, G, 1, KS, DUMP>), grid, block, 0, s, gp); break;
        default: hipLaunchKernelGGL((gemm_kernel<BN, G, 2, KS, DUMP>), grid, block, 0, s, gp); break;
    }
    return hipGetLastError();
}

// Workspace of a split launch: one 64-byte flag line per tile, then (256-byte
// aligned) each tile's 128 x bn partial sums.
size_t split_flag_bytes(int64_t tiles) { return (((size_t)tiles * 64) + 255) / 256 * 256; }

template <int BN, int KS, bool DUMP>
hipError_t launch_tile(const LinearArgs& a, hipStream_t s, bool split = false) {
    GemmParams gp{};
    gp.a = a;
    const int outw = a.mode == 2 ? BN / 2 : BN;
    gp.tilesM = (int)((a.M + kBM - 1) / kBM);
    gp.tilesN = (int)((a.N + outw - 1) / outw);
    gp.NG = (int)(a.K / a.G);
    if (split) {
        gp.split = 1;
        gp.flags = static_cast<unsigned int*>(a.workspace);
        gp.part = reinterpret_cast<float*>(static_cast<unsigned char*>(a.workspace) +
                                           split_flag_bytes((int64_t)gp.tilesM * gp.tilesN));
    }
    if (a.G == 128) return launch_mode<BN, 128, KS, DUMP>(gp, s);
    if constexpr (KS == 2 && BN > 128) return hipErrorInvalidConfiguration;  // (group 32 there: never planned)
    else return launch_mode<BN, 32, KS, DUMP>(gp, s);
}

}  // namespace
}  // namespace wq
