// Prefill GEMM with K split between the waves of a workgroup (webyIQ
// crates/engine/src/shaders/gemm_q4q8.wgsl), for the calls that the 128-token
// tiles of gemm_q4q8.hip serve badly: few tokens, whose tiles leave most CUs
// idle, and activations with one scale per 32 elements.
//
// y[t,n] = sum_g dx[t,g] * (s[n,g] * A[t,n,g] + m[n,g] * X[t,g])
// (per-token activations: dx[t] applied to the total).
//
// A workgroup of W waves owns 32 tokens x 32 TN weight rows; wave w takes the
// K steps (128 codes) S w / W .. S (w + 1) / W - 1 of all of them.  Each wave
// fills its own LDS stage by direct global -> LDS loads and waits for its own
// loads only, so the main loop has no barrier: a step's fragments move to
// registers, the next step's loads are issued into the stage, and the step is
// computed meanwhile (a second stage per wave halves the workgroups that share
// a CU, and was slower where several do).  The waves' fp32 sums meet in LDS at the end,
// added in wave order.
//
// Few tokens are bound by the chain of one workgroup (launch, loads, a few
// steps, the exchange: back to back in a graph 4.6-5.0 us at one step per wave,
// 0.7 us for each further step, 1.1 us with per-32 activations), many by the
// fold.  With groups of 32 each output takes a
// conversion and an fma per group on the VALU; per-32 activations need the
// factor dx[t,g] * s[n,g] besides.  That factor, an outer product, comes out
// of one f32 MFMA in the accumulator layout, rounded once like the product it
// replaces, and the min term sum_g m[n,g] (dx[t,g] X[t,g]) of two groups out
// of another: both ran on the VALU with LDS reads per element in the kernel
// before it (M = 19, K = 6144, N = 2048: 120 -> 10.6 us; M = 1024, K = 2048,
// N = 6144 in pairs: 223 -> 117 us).
#include "common.hpp"
#include "gemm_common.hpp"
#include "launch.hpp"

#pragma clang fp contract(off)

namespace wq {
namespace {

// wait until at most n vector-memory operations of this wave are in flight
template <int n>
__device__ __forceinline__ void wait_vm() {
    static_assert(n >= 0 && n < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
    asm volatile("" ::: "memory");
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// direct global -> LDS load of 16 bytes per lane from per-lane addresses
__device__ __forceinline__ void dma16_lane(const void* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop

template <int TN, int G, bool PT>
struct WaveTile {
    static constexpr int GE = PT ? G : 32;   // accumulation group
    static constexpr int NES = kBK / GE;     // accumulation groups per step
    static constexpr int NGS = kBK / G;      // weight groups per step
    // LDS of one stage: activations, packed weights, scale words (one or four
    // per row), group sums (one or four per token), per-32 scales
    static constexpr int A_SZ = 32 * kBK;
    static constexpr int B_SZ = TN * 32 * kBK / 2;
    static constexpr int S_SZ = NGS == 1 ? 256 : 1024;
    static constexpr int X_SZ = NES == 1 ? 256 : 1024;
    static constexpr int OFF_S = A_SZ + B_SZ, OFF_X = OFF_S + S_SZ;
    static constexpr int OFF_D = OFF_X + 512;  // per-32 scales: the upper lanes' half of the group sums' load
    static constexpr int STAGE = OFF_X + X_SZ;
    static constexpr int NA = A_SZ / 1024, NB = B_SZ / 1024;  // direct-to-LDS instructions of 1 KiB
};

// LATE (mode 1): the outputs' old values are read after the last step instead
// of before the first (see launch_mode)
template <int TN, int W, int G, bool PT, int MODE, bool LATE, bool DUMP>
__global__ __launch_bounds__(64 * W) void wave_gemm_kernel(GemmParams p) {
    using T = WaveTile<TN, G, PT>;
    constexpr int NES = T::NES, NGS = T::NGS;
    static_assert(MODE != 2 || TN == 2, "mode 2 pairs a gate and an up subtile");
    static_assert(TN == 1 || TN == 2, "tile");
    constexpr int RED_SZ = W == 1 ? 0 : W * TN * 4096;  // the waves' sums
    constexpr int LDS_SZ = W * T::STAGE > RED_SZ ? W * T::STAGE : RED_SZ;
    static_assert(LDS_SZ <= kLdsBytes, "LDS");
    __shared__ __align__(1024) unsigned char lds[LDS_SZ];

    const LinearArgs& a = p.a;
    pin_arg(a.wq); pin_arg(a.ws); pin_arg(a.xq); pin_arg(a.dx); pin_arg(a.xs); pin_arg(a.y);
    pin_arg(a.N); pin_arg(a.K); pin_arg(a.M); pin_arg(a.params);
    pin_arg(p.tilesM); pin_arg(p.tilesN); pin_arg(p.NE); pin_arg(p.NG); pin_arg(p.first); pin_arg(p.count); pin_arg(p.wide);
    if (DUMP) pin_arg(a.acc_dump);

    const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int64_t M = a.M;  // tokens of this call: M, or (device Params) min(p.m, M)
    if (a.params) {
        const int64_t pm = (int64_t)a.params[kParamM];
        M = pm < M ? pm : M;
    }
    const int64_t N = a.N;
    const int K = (int)a.K, NG = p.NG, NE = p.NE;

    // XCD-aware tile order: the token tiles of one set of weight rows on one
    // XCD.  Only tiles with tokens of this step are numbered, the workgroups
    // past them leave: with the token tiles past M interleaved, the working
    // ones landed on every second or fourth CU of the dispatch order and shared
    // it (19 tokens of a 128-token chunk, per-32, K = 2048, gate/up pairs
    // N = 6144 19.5 -> 10.1 us; the whole block's chunk 55 -> 43.6 us).
    const int tilesM = a.params ? (int)((M + 31) / 32) : p.tilesM;
    const int64_t left = (int64_t)tilesM * p.tilesN - p.first;
    const int tiles = left < p.count ? (int)left : p.count, bid = blockIdx.x;
    if (bid >= tiles) return;  // (uniform: nothing issued yet)
    const int xcd = bid % kXcds, li = bid / kXcds;
    const int per = tiles / kXcds, rem = tiles % kXcds;
    const int lt = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + li + p.first;
    const int tile_n = lt / tilesM, tile_m = lt - tile_n * tilesM;
    const int64_t m0 = (int64_t)tile_m * 32;
    constexpr int OUTW = MODE == 2 ? 32 : 32 * TN;  // output columns per tile
    const int64_t n0 = (int64_t)tile_n * OUTW;

    // weight row of tile row r (mode 2: a gate subtile, then its up subtile), token of tile token r
    auto wrow = [&](int r) -> int64_t {
        int64_t n = n0 + (MODE == 2 ? r & 31 : r);
        n = n < N ? n : N - 1;
        return MODE == 2 && r >= 32 ? n + N : n;
    };
    auto trow = [&](int r) -> int64_t {
        const int64_t t = m0 + r;
        return t < M ? t : M - 1;
    };

    // ---------------- staging ----------------
    const int S = K / kBK;
    const int s_begin = S * wave / W, s_end = S * (wave + 1) / W;
    const uint32_t lds0 = lds_addr(lds) + (uint32_t)(wave * T::STAGE);
    uint32_t a_off[T::NA], b_off[T::NB];
#pragma unroll
    for (int i = 0; i < T::NA; ++i) {  // 8 rows of 128 bytes
        const int r = 8 * i + lane / 8;
        a_off[i] = (uint32_t)(trow(r) * K + 16 * ((lane % 8) ^ swz_a(r)));
    }
#pragma unroll
    for (int i = 0; i < T::NB; ++i) {  // 16 rows of 64 bytes
        const int r = 16 * i + lane / 4;
        b_off[i] = (uint32_t)(wrow(r) * (K / 2) + 16 * ((lane % 4) ^ swz_b(r)));
    }
    const int64_t srow = wrow(lane & (32 * TN - 1));
    const int64_t xrow = trow(l32);
    const bool wide = p.wide;  // the four-word pieces as one load
    auto issue = [&](int step) {
        const int8_t* xq = a.xq + step * kBK;
        const uint8_t* wq = reinterpret_cast<const uint8_t*>(a.wq) + step * (kBK / 2);
#pragma unroll
        for (int i = 0; i < T::NA; ++i) dma16_at(xq, a_off[i], lds0 + 1024 * i);
#pragma unroll
        for (int i = 0; i < T::NB; ++i) dma16_at(wq, b_off[i], lds0 + T::A_SZ + 1024 * i);
        if constexpr (NGS == 1) dma4_at(a.ws + step, (uint32_t)(4 * srow * NG), lds0 + T::OFF_S);
        if constexpr (NES == 1) dma4_at(a.xs + step, (uint32_t)(4 * xrow * NE), lds0 + T::OFF_X);
        if constexpr (NGS == 4 || NES == 4) {
            // lane's piece: the four words of its row (lanes past the rows repeat them)
            const uint32_t* sp = a.ws + srow * NG + 4 * step;
            const int32_t* xp = a.xs + xrow * NE + 4 * step;
            const float* dp = a.dx + (PT ? 0 : xrow * NE + 4 * step);
            const void* xd = !PT && h ? static_cast<const void*>(dp) : static_cast<const void*>(xp);
            if (wide) {
                if constexpr (NGS == 4) dma16_lane(sp, lds0 + T::OFF_S);
                if constexpr (NES == 4) dma16_lane(xd, lds0 + T::OFF_X);
            } else {
                unsigned char* l = lds + wave * T::STAGE + 16 * lane;
                auto copy4 = [&](const void* src, int off) {
                    const uint32_t* q = static_cast<const uint32_t*>(src);
                    *reinterpret_cast<uint4*>(l + off) = make_uint4(q[0], q[1], q[2], q[3]);
                };
                if constexpr (NGS == 4) copy4(sp, T::OFF_S);
                if constexpr (NES == 4) copy4(xd, T::OFF_X);
            }
        }
    };

    v16f facc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) facc[j] = v16f{};

    const int rows_total = MODE == 2 ? 2 * (int)N : (int)N;
    auto dump = [&](int e, int j, const v16i& acc) {  // test hook: the exact group sums
        const int64_t nn = n0 + (MODE == 2 ? l32 : 32 * j + l32);
        const int64_t wr = MODE == 2 && j == 1 ? nn + N : nn;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t t = m0 + 8 * (r >> 2) + 4 * h + (r & 3);
            if (t < M && nn < N) a.acc_dump[(t * rows_total + wr) * NE + e] = acc[r];
        }
    };

    // outputs this wave finishes: UPW units (j, r) of 64 (32 columns of two
    // tokens); their token scales and (mode 1) old values, requested first
    constexpr int UNITS = (MODE == 2 ? 1 : TN) * 16, UPW = UNITS / W;
    static_assert(UNITS % W == 0, "the waves share the outputs evenly");
    auto out_t = [&](int q) -> int64_t {
        const int r = (wave * UPW + q) & 15;
        return m0 + 8 * (r >> 2) + 4 * h + (r & 3);
    };
    auto out_n = [&](int q) -> int64_t { return n0 + 32 * ((wave * UPW + q) >> 4) + l32; };
    auto out_ok = [&](int q) { return out_t(q) < M && out_n(q) < N; };
    auto out_at = [&](int q) -> int64_t { return out_t(q) * N + out_n(q); };
    float dtok[UPW], yold[UPW];
#pragma unroll
    for (int q = 0; q < UPW; ++q) {
        if (PT) dtok[q] = a.dx[out_t(q) < M ? out_t(q) : M - 1];
        if (MODE == 1 && !LATE) yold[q] = out_ok(q) ? a.y[out_at(q)] : 0.0f;
    }

    const unsigned char* st = lds + wave * T::STAGE;
    if (s_begin < s_end) issue(s_begin);
    for (int s = s_begin; s < s_end; ++s) {
        wait_vm<0>();
        // this step's fragments and scales into registers, then the next
        // step's loads into the stage they leave
        v4i af[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)  // group 128: codes 64 h + 16 ks ..; groups of 32: 32 ks + 16 h ..
            af[ks] = *reinterpret_cast<const v4i*>(st + l32 * kBK + 16 * ((NES == 4 ? 2 * ks + h : 4 * h + ks) ^ swz_a(l32)));
        uint4 pb[TN][2];
        uint32_t sw[TN][NGS];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int br = 32 * j + l32;
            const unsigned char* Bb = st + T::A_SZ + br * 64;
            if constexpr (NES == 4) {
                uint2 q[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) q[c] = *reinterpret_cast<const uint2*>(Bb + 16 * (c ^ swz_b(br)) + 8 * h);
                pb[j][0] = make_uint4(q[0].x, q[0].y, q[1].x, q[1].y);
                pb[j][1] = make_uint4(q[2].x, q[2].y, q[3].x, q[3].y);
            } else {
                pb[j][0] = *reinterpret_cast<const uint4*>(Bb + 16 * ((2 * h) ^ swz_b(br)));
                pb[j][1] = *reinterpret_cast<const uint4*>(Bb + 16 * ((2 * h + 1) ^ swz_b(br)));
            }
            if constexpr (NGS == 4) {
                const uint4 v = *reinterpret_cast<const uint4*>(st + T::OFF_S + 16 * br);
                sw[j][0] = v.x; sw[j][1] = v.y; sw[j][2] = v.z; sw[j][3] = v.w;
            } else {
                sw[j][0] = *reinterpret_cast<const uint32_t*>(st + T::OFF_S + 4 * br);
            }
        }
        int32_t xv[NES];
        float dv[NES];
        if constexpr (NES == 4) {
            const int4 v = *reinterpret_cast<const int4*>(st + T::OFF_X + 16 * l32);
            xv[0] = v.x; xv[1] = v.y; xv[2] = v.z; xv[3] = v.w;
        } else {
            xv[0] = *reinterpret_cast<const int32_t*>(st + T::OFF_X + 4 * l32);
        }
        if constexpr (!PT) {
            const float4 v = *reinterpret_cast<const float4*>(st + T::OFF_D + 16 * l32);
            dv[0] = v.x; dv[1] = v.y; dv[2] = v.z; dv[3] = v.w;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (s + 1 < s_end) issue(s + 1);

        // min term: facc += sum_g m[n,g] X[t,g] on the matrix cores
        if constexpr (PT) {
            // f16: X = 64 X_hi + X_lo, exact products; lane half 0 holds
            // (64 X_hi, m) of the step's groups, half 1 (X_lo, m)
            v8h xa = {};
#pragma unroll
            for (int u = 0; u < NES; ++u) xa[u] = (_Float16)(h == 0 ? (float)((xv[u] >> 6) * 64) : (float)(xv[u] & 63));
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                v8h mb = {};
#pragma unroll
                for (int u = 0; u < NGS; ++u) mb[u] = __builtin_bit_cast(_Float16, (unsigned short)(sw[j][u] >> 16));
                facc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xa, mb, facc[j], 0, 0, 0);
            }
        } else {
            // f32: two groups per instruction, lane half h group u + h
#pragma unroll
            for (int u = 0; u < 4; u += 2) {
                const float xm = h ? dv[u + 1] * (float)xv[u + 1] : dv[u] * (float)xv[u];
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const float mm = f16hi(NGS == 1 ? sw[j][0] : h ? sw[j][(u + 1) % NGS] : sw[j][u % NGS]);
                    facc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xm, mm, facc[j], 0, 0, 0);
                }
            }
        }

        if constexpr (NES == 1) {  // one group of 128 per step
            v16i acc[TN];
            float sv[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const v4i bf[4] = {expand8(pb[j][0].x, pb[j][0].y), expand8(pb[j][0].z, pb[j][0].w),
                                   expand8(pb[j][1].x, pb[j][1].y), expand8(pb[j][1].z, pb[j][1].w)};
                sv[j] = f16lo(sw[j][0]);
                asm volatile("" : "+v"(sv[j]));  // an f32 operand: v_fmac_f32 instead of the slower v_fma_mix_f32
#pragma unroll
                for (int ks = 0; ks < 4; ++ks)
                    acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[ks], bf[ks], ks == 0 ? v16i{} : acc[j], 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if (DUMP) dump(s, j, acc[j]);
#pragma unroll
                for (int r = 0; r < 16; ++r) facc[j][r] = fmaf(sv[j], (float)acc[j][r], facc[j][r]);
            }
        } else {
            // four groups of 32: the MFMAs of group u + 1 are issued before
            // the fold of group u
            v16i acc[2][TN];
            v16f sc[2][TN];  // per-32 activations: dx[t,g] * s[n,g], an outer product on the f32 MFMA
            float sv[2][TN];
            auto mfmas = [&](auto uc) __attribute__((always_inline)) {
                constexpr int u = decltype(uc)::value, q = u & 1;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const uint4& w4 = pb[j][u >> 1];
                    const v4i bf = (u & 1) ? expand8(w4.z, w4.w) : expand8(w4.x, w4.y);
                    sv[q][j] = f16lo(sw[j][u % NGS]);
                    asm volatile("" : "+v"(sv[q][j]));
                    acc[q][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[u], bf, v16i{}, 0, 0, 0);
                    if constexpr (!PT)
                        sc[q][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(h ? 0.0f : dv[u], h ? 0.0f : sv[q][j], v16f{}, 0, 0, 0);
                }
            };
            auto fold = [&](auto uc) __attribute__((always_inline)) {
                constexpr int u = decltype(uc)::value, q = u & 1;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if (DUMP) dump(4 * s + u, j, acc[q][j]);
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        facc[j][r] = fmaf(PT ? sv[q][j] : sc[q][j][r], (float)acc[q][j][r], facc[j][r]);
                }
            };
            mfmas(std::integral_constant<int, 0>{});
            static_for<1, 4>([&](auto uc) __attribute__((always_inline)) {
                mfmas(uc);
                fold(std::integral_constant<int, decltype(uc)::value - 1>{});
            });
            fold(std::integral_constant<int, 3>{});
        }
    }

    // ---------------- the waves' sums, epilogue ----------------
    float* red = reinterpret_cast<float*>(lds);  // [wave][j][r][lane]
    constexpr int WS = TN * 16 * 64;
    if constexpr (W > 1) {
        __syncthreads();  // every wave has left its stage
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) red[wave * WS + (j * 16 + r) * 64 + lane] = facc[j][r];
        __syncthreads();
    }
    if (MODE == 1 && LATE) {
#pragma unroll
        for (int q = 0; q < UPW; ++q) yold[q] = out_ok(q) ? a.y[out_at(q)] : 0.0f;
    }
    auto total = [&](int j, int r) {  // the waves' sums in wave order
        if constexpr (W == 1) return facc[j][r];
        const float* q = red + (j * 16 + r) * 64 + lane;
        float v = q[0];
#pragma unroll
        for (int w = 1; w < W; ++w) v = v + q[w * WS];
        return v;
    };
#pragma unroll
    for (int q = 0; q < UPW; ++q) {
        const int unit = W == 1 ? q : wave * UPW + q, r = unit & 15, j = unit >> 4;
        float v = total(j, r);
        float u = MODE == 2 ? total(1, r) : 0.0f;
        if (PT) {
            v = v * dtok[q];
            if (MODE == 2) u = u * dtok[q];
        }
        if (MODE == 2) v = silu_mul(v, u);
        if (out_ok(q)) a.y[out_at(q)] = MODE == 1 ? yold[q] + v : v;
    }
}

// Mode 1 with four waves: early reads of the old values overlap the steps, but
// their addresses take some 60 registers, and with them a third of the waves
// of a SIMD.  Per-32 calls of many tiles read them late (us, early / late, 2,048
// tiles M = 2048, K = 1536, N = 2048 40.7 / 36.3, K = 6144 124 / 120; 24,576
// tiles M = 8192, K = 256, N = 6144 201 / 166; 1,504 tiles 17.4 / 16.0 and 96 /
// 95; below, and per token, early ones are ahead: M = 600, K = 768, N = 1000
// 5.9 / 7.2).  One wave per tile always does.
template <int TN, int W, int G, bool PT, bool DUMP>
hipError_t launch_mode(GemmParams gp, hipStream_t s) {
    constexpr bool MAY = !PT && !DUMP && W <= 4;
    // groups of 32 keep narrow tiles up to 768 of them and run wide ones with
    // eight waves up to 256 only, that is in mode 2 alone
    constexpr bool PAIRS_ONLY = TN == 2 && W == 8 && !DUMP && (G == 32 || !PT);
    const bool late = W == 1 || (int64_t)gp.tilesM * gp.tilesN >= 2048;
    // a grid holds fewer than 2^32 threads: larger ones as several launches
    const int64_t tiles = (int64_t)gp.tilesM * gp.tilesN, most = (int64_t(1) << 31) / (64 * W);
    for (int64_t first = 0; first < tiles; first += most) {
        gp.first = (int)first;
        gp.count = (int)(tiles - first < most ? tiles - first : most);
        dim3 grid((unsigned)gp.count), block(64 * W);
        switch (gp.a.mode) {
            case 0:
                if constexpr (PAIRS_ONLY) return hipErrorInvalidConfiguration;
                else hipLaunchKernelGGL((wave_gemm_kernel<TN, W, G, PT, 0, false, DUMP>), grid, block, 0, s, gp);
                break;
            case 1:
                if constexpr (PAIRS_ONLY) return hipErrorInvalidConfiguration;
                else if (MAY && late)
                    hipLaunchKernelGGL((wave_gemm_kernel<TN, W, G, PT, 1, MAY, DUMP>), grid, block, 0, s, gp);
                else if constexpr (W > 1)
                    hipLaunchKernelGGL((wave_gemm_kernel<TN, W, G, PT, 1, false, DUMP>), grid, block, 0, s, gp);
                break;
            default:
                if constexpr (TN == 2)
                    hipLaunchKernelGGL((wave_gemm_kernel<TN, W, G, PT, 2, false, DUMP>), grid, block, 0, s, gp);
                else
                    return hipErrorInvalidConfiguration;  // the host pairs mode 2 with two columns
                break;
        }
    }
    return hipGetLastError();
}

template <int TN, int W, bool DUMP>
hipError_t launch_tile(const LinearArgs& a, hipStream_t s) {
    GemmParams gp{};
    gp.a = a;
    const bool pt = a.GA == a.K;
    const int outw = a.mode == 2 ? 32 : 32 * TN;
    gp.tilesM = (int)((a.M + 31) / 32);
    gp.tilesN = (int)((a.N + outw - 1) / outw);
    gp.NE = (int)(a.K / (pt ? a.G : 32));
    gp.NG = (int)(a.K / a.G);
    auto al = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    gp.wide = al(a.ws) && al(a.xs) && (pt || al(a.dx));
    if (pt) {
        if constexpr (W == 1) return hipErrorInvalidConfiguration;  // (never planned: per-32 activations only)
        else return a.G == 128 ? launch_mode<TN, W, 128, true, DUMP>(gp, s) : launch_mode<TN, W, 32, true, DUMP>(gp, s);
    }
    return a.G == 128 ? launch_mode<TN, W, 128, false, DUMP>(gp, s) : launch_mode<TN, W, 32, false, DUMP>(gp, s);
}

int64_t tiles_of(const LinearArgs& a, int tn) {
    const int64_t outw = a.mode == 2 ? 32 : 32 * tn;
    return ((a.M + 31) / 32) * ((a.N + outw - 1) / outw);
}

// Tile width and waves.  While the grid leaves CUs idle, narrow tiles put
// more of them to work and eight waves shorten each wave's chain of K steps;
// past one workgroup per CU, wider tiles read the activations half as often
// and four waves leave room for more workgroups on a CU.  Measured, us, 64
// rows x 8 waves / 64 x 4 / 32 x 8: M = 60, K = 2048, N = 3072 (192 tiles of
// 32 rows) 6.1 / 6.2 / 5.4, M = 130, N = 2048 (320) 6.3 / 6.4 / 7.1, M = 700,
// K = 1024, N = 2048 (704 tiles of 64 rows) 9.6 / 8.6 / 10.5; with groups of
// 32 the fold outweighs the loads and narrow tiles, whose waves hold fewer
// registers, stay ahead longer: per-32 at M = 333, K = 4096, N = 2048 (704)
// 25.4 / 23.4 / 20.8, at M = 512, K = 2048, N = 3072 (1,536) 23.9 / 19.6 / 22.0.
// A row of one step (K = 128) leaves all waves but one without work; past a few
// tiles per CU the call waits for their exchange and their place on the CU:
// per-32 calls run one wave per tile there (us, one / four waves, 512 tiles
// M = 512, N = 2048 6.8 / 6.0, 1,024 tiles 7.6 / 9.4, 24,576 tiles M = 8192,
// N = 6144 67 / 114; mode 1 at 1,024 tiles 11.1 / 10.4, 1,824 tiles 14 / 18).
// One step's sum is the same bits either way.
struct Plan {
    int tn, w;
};
Plan pick_plan(const LinearArgs& a) {
    const bool groups32 = a.G == 32 || a.GA != a.K;
    if (a.mode != 2 && tiles_of(a, 1) <= (groups32 ? 768 : 256)) return Plan{1, 8};
    const int64_t tiles = tiles_of(a, 2);
    if (a.K == kBK && a.GA != a.K && tiles >= (a.mode == 1 ? 1280 : 1024)) return Plan{2, 1};
    return Plan{2, tiles <= 256 ? 8 : 4};
}

}  // namespace

// Per-32 activations always; per-token activations when the 128-token tiles
// would leave most CUs idle: the grid fits one workgroup per CU, or the
// fitted cost (4 us + tile-steps per CU x 0.18 us, 0.197 us from 48 steps on,
// 0.25 us with groups of 32) is clearly below that of the other kernel's best
// plan, `tiled_us`.  Measured, us, here / there (its best width; back to back
// in a graph): K = 2048, N = 3072 at M = 97 6.4 / 11.3, M = 200 8.9 / 11.6,
// M = 333 11.5 / 11.7; gate/up pairs N = 6144 12.0 / 12.4, 18.3 / 17.9 and
// 26.5 / 23.0; groups of 32 at M = 333 15.3 / 20.4 and 34.7 / 51.0; K = 6144,
// N = 2048 at M = 256 12.4 / 17.4, M = 300 18.9 / 17.9 (K split in pairs there).
bool gemm_wave_fits(const LinearArgs& a, double tiled_us) {
    if (a.GA != a.K) return true;
    const int64_t tiles = tiles_of(a, 2);
    if (tiles <= 256) return true;
    // one step (K = 128) of many tiles: the waves mostly exchange zeros (us, here /
    // there, gate/up pairs N = 6144 at M = 300, 1,920 tiles, 9.4 / 10.2, M = 1500
    // 36 / 22, group 32 at M = 8192, mode 0 143 / 51)
    if (a.K == kBK && tiles > 2048) return false;
    const int64_t steps = a.K / kBK;
    const double us = 4.0 + (a.G == 32 ? 0.25 : steps < 48 ? 0.18 : 0.197) * (double)(tiles * steps) / 256.0;
    return us < 0.9 * tiled_us;
}

GemmForm gemm_wave_form(const LinearArgs& a) {
    const Plan pl = pick_plan(a);
    return GemmForm{kFormWaves, 32 * pl.tn, pl.w, false};
}

// The group-sum dump (a test hook) runs the plan's waves, and with them its
// fp32 order, on the wide tile; the width does not enter an output's order.
hipError_t launch_gemm_wave(const LinearArgs& a, hipStream_t s) {
    const Plan pl = pick_plan(a);
    if (a.acc_dump) return pl.w == 8 ? launch_tile<2, 8, true>(a, s) : launch_tile<2, 4, true>(a, s);
    if (pl.tn == 1) return launch_tile<1, 8, false>(a, s);
    if (pl.w == 1) return launch_tile<2, 1, false>(a, s);
    return pl.w == 8 ? launch_tile<2, 8, false>(a, s) : launch_tile<2, 4, false>(a, s);
}

}  // namespace wq
