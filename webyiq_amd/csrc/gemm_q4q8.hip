// Prefill GEMM Y[M, N] = X W^T on int8 MFMA (webyIQ
// crates/engine/src/shaders/gemm_q4q8.wgsl, host side Builder::gemm in
// crates/engine/src/graph.rs:200-205; the reference runs it on ALU
// dot4I8Packed in 32x32 tiles).
//
// y[t,n] = dx[t] * sum_g (s[n,g] * A[t,n,g] + m[n,g] * X[t,g]),
// A = exact int32 sum of q * xq over group g, X = sum of xq over g.  This file
// serves per-token activations; per-32 scales, and calls of few tokens, run
// the kernel of gemm_wave.hip.
//
// MI355X design.  A group of 4 waves (2 along M x 2 along N, one per SIMD)
// owns a 128-token x BN-row tile, and each wave a 64 x BN/2 block of 32 x 32
// subtiles computed with v_mfma_i32_32x32x32_i8.  Every tile of a K step (128
// codes) travels global -> LDS directly (global_load_lds, no registers): the
// int8 activations, the packed int4 weights, the scale words.  Two forms keep
// two waves on each SIMD, so that one's folds run beside the other's products:
// - two wave groups on one tile, one workgroup per CU: they take alternate K
//   steps on a ring of 4 LDS stages, the loads of the next two steps in flight
//   while two are computed, one barrier per round, and add their sums at the
//   end (gemm_tile.hpp, KS = 2);
// - one wave group on 2 stages, two workgroups per CU: a step's fragments move
//   to registers, a barrier, and the loads of the step after next go into the
//   stage they leave (KS = 1).
// Each wave expands its weight fragments from nibbles to int8 in registers.
// Tiles are stored in rows whose 16-byte chunks are XOR-swizzled by the row
// index, so that the 16-byte fragment reads of consecutive rows hit distinct
// banks.
//
// Folding the exact group sums into fp32 is VALU work per output element per
// group, as much issue time as the MFMAs themselves.  Group 128, and group 32
// with one MFMA pair and one fold per group, keep it at two instructions,
// acc = fma(s, float(A), acc), and compute the min term sum_g m * X up front
// on the f16 MFMA: X = 64 * X_hi + X_lo with 64 * X_hi and X_lo exact in f16
// (|X| <= 128 * 127), so each product with the f16 m is exact.  Tiles are
// assigned XCD by XCD so that the workgroups sharing a weight tile share
// one L2.
#include "gemm_tile.hpp"

namespace wq {
namespace {

int64_t tiles_of(const LinearArgs& a, int bn) {
    const int64_t outw = a.mode == 2 ? bn / 2 : bn;
    return ((a.M + kBM - 1) / kBM) * ((a.N + outw - 1) / outw);
}

// Tile width, and how the grid fills the chip: the cheapest of these by costs
// (us) fitted to measured launches, `steps` K steps of 128 codes.
//   ks = 2: rounds of 256 workgroups, each c0 + steps x (ca + cb x width);
//     split (K across a workgroup pair: widths up to 128, K a multiple of 512
//     with 32 steps or more, a workspace): half the steps plus ~3 us for the
//     exchange.  It splits where the unsplit grid leaves CUs idle (K = 6144,
//     N = 2048 at width 64: M = 512 20.4 us against 25.2 unsplit, M = 300 17.9
//     against 24.5).
//   ks = 1: two workgroups per CU side by side, c0 + steps x (ca + cb x width)
//     for a pair and for a workgroup alone.
// With ks = 1 a tile's first loads, min term, barriers and epilogue run beside
// another tile's products.  Measured, us, best width of ks = 2 / ks = 1 (back
// to back in a graph): M = 2048, K = 2048, N = 6144 44.7 / 40.3 (both 192),
// M = 4096 in pairs 165 / 144 (192), K = 6144, N = 2048 71.4 (256) / 73.0 (128);
// group 32, whose fold takes most of the time, 94.6 (128) / 78.0 (192) and, in
// pairs, 371 / 270.  With one tile per CU the two wave groups of ks = 2 stay
// ahead at group 128: M = 1024, K = 2048, N = 6144 24.5 / 29.6, group 32 63.4 /
// 52.2.
struct Plan {
    int bn, ks;
    bool split;
    double us;
};

Plan pick_plan(const LinearArgs& a, bool allow_split) {
    constexpr int64_t kCu = 256;
    constexpr double kExchange = 3.0;
    const bool g32 = a.G == 32;
    const double steps = (double)(a.K / kBK);
    Plan best{64, 2, false, -1.0};
    auto offer = [&](int bn, int ks, bool split, double us) {
        if (best.us < 0 || us < best.us) best = Plan{bn, ks, split, us};
    };
    for (int bn : {256, 192, 128, 64}) {
        const int64_t tiles = tiles_of(a, bn);
        if (!(g32 && bn > 128)) {
            const double step = g32 ? 0.35 + 0.0105 * bn : 0.131 + 0.00525 * bn;
            for (int sp = 0; sp < (allow_split && bn <= 128 ? 2 : 1); ++sp) {
                const int64_t rounds = (tiles * (sp ? 2 : 1) + kCu - 1) / kCu;
                offer(bn, 2, sp != 0, (double)rounds * (3.2 + (sp ? kExchange : 0.0) + steps / (sp ? 2 : 1) * step));
            }
        }
        if (bn > 192) continue;
        const int64_t per_cu = (tiles + kCu - 1) / kCu;
        const double pair = 4.0 + steps * (g32 ? 0.5 + 0.0197 * bn : 0.17 + 0.0102 * bn);
        const double one = 4.0 + steps * (g32 ? 0.37 + 0.0124 * bn : 0.15 + 0.0065 * bn);
        offer(bn, 1, false, (double)(per_cu / 2) * pair + (double)(per_cu % 2) * one);
    }
    return best;
}

// flag lines, then each tile's partial sums
size_t split_bytes(const LinearArgs& a, int bn) {
    const int64_t t = tiles_of(a, bn);
    return split_flag_bytes(t) + (size_t)t * kBM * bn * 4;
}

// the shapes whose K the pair can split: per-token activations at group 128
// or 32 (the formats with two wave groups), an even number of steps per half
bool split_shape(const LinearArgs& a) {
    return a.GA == a.K && (a.G == 128 || a.G == 32) && a.K % 512 == 0 && a.K / kBK >= 32;
}

template <bool DUMP>
hipError_t launch_bn(const LinearArgs& a, const Plan& pl, hipStream_t s) {
    if (pl.ks == 1) return launch_gemm_shared(a, pl.bn, s);
    switch (pl.bn) {
        case 256: return launch_tile<256, 2, DUMP>(a, s);
        case 192: return launch_tile<192, 2, DUMP>(a, s);
        case 128: return launch_tile<128, 2, DUMP>(a, s, pl.split);
        default: return launch_tile<64, 2, DUMP>(a, s, pl.split);
    }
}

// The kernel of a call: the tile plan, and whether the wave-split kernel takes
// the call instead (the plan then splits nothing).
struct Choice {
    Plan tiles;
    bool wave;
};

Choice choose(const LinearArgs& a, bool may_split) {
    Choice c{pick_plan(a, may_split && split_shape(a)), false};
    c.wave = gemm_wave_fits(a, c.tiles.us);
    if (c.wave) c.tiles.split = false;
    return c;
}

// the same for a call's own workspace
Choice choose_for(const LinearArgs& a) {
    const Choice c = choose(a, !a.acc_dump);
    if (c.tiles.split && !(a.workspace && a.workspace_bytes >= split_bytes(a, c.tiles.bn))) return choose(a, false);
    return c;
}

}  // namespace

size_t gemm_workspace_bytes(const LinearArgs& a) {
    const Choice c = choose(a, true);
    return c.tiles.split ? split_bytes(a, c.tiles.bn) : 0;
}

GemmForm gemm_form(const LinearArgs& a) {
    const Choice c = choose_for(a);
    if (c.wave) return gemm_wave_form(a);
    return GemmForm{kFormTiles, c.tiles.bn, 4 * c.tiles.ks, c.tiles.split};
}

// The group-sum dump (a test hook) runs the tile width the production launch
// without a workspace picks for the same shape, so the sums it stores are
// those of the kernel instance that serves the call.
hipError_t launch_gemm(const LinearArgs& a, hipStream_t s) {
    const Choice c = choose_for(a);
    if (c.wave) return launch_gemm_wave(a, s);
    return a.acc_dump ? launch_bn<true>(a, c.tiles, s) : launch_bn<false>(a, c.tiles, s);
}

}  // namespace wq
