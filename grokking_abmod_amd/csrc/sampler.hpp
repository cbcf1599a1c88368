// The reference's token choice made by one wave (gpu.rs:2028-2049), shared by
// the kernel files: greedy, or one SplitMix64 draw against the softmax's
// cumulative sums with the reference's f32 result.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

#include "dpp.hpp"

namespace meshgpt::kern {

__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, dpp_move<0xB1>(v, v));
    v = fmaxf(v, dpp_move<0x4E>(v, v));
    v = fmaxf(v, dpp_move<0x141>(v, v));
    v = fmaxf(v, dpp_move<0x140>(v, v));
    v = fmaxf(v, dpp_move<0x142, 0xa>(v, v));
    v = fmaxf(v, dpp_move<0x143, 0xc>(v, v));
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// The lane's value moved by a DPP pattern, 0 where the pattern has no source.
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ double dpp_move_f64(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const int lo = __builtin_amdgcn_update_dpp(0, int(uint32_t(b)), CTRL, ROW_MASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, int(uint32_t(b >> 32)), CTRL, ROW_MASK, 0xf, false);
    return __builtin_bit_cast(double, (uint64_t(uint32_t(hi)) << 32) | uint32_t(lo));
}

// Inclusive prefix sum over the wave's lanes: row shifts inside each 16-lane
// row, then the row broadcasts carry row totals forward.
__device__ __forceinline__ double wave_inclusive_sum(double x) {
    x += dpp_move_f64<0x111>(x);       // row_shr:1
    x += dpp_move_f64<0x112>(x);       // row_shr:2
    x += dpp_move_f64<0x114>(x);       // row_shr:4
    x += dpp_move_f64<0x118>(x);       // row_shr:8
    x += dpp_move_f64<0x142, 0xa>(x);  // row_bcast:15
    x += dpp_move_f64<0x143, 0xc>(x);  // row_bcast:31
    return x;
}

__device__ __forceinline__ uint64_t splitmix_next(uint64_t &state) {
    state += 0x9e3779b97f4a7c15ULL;
    uint64_t bits = state;
    bits = (bits ^ (bits >> 30)) * 0xbf58476d1ce4e5b9ULL;
    bits = (bits ^ (bits >> 27)) * 0x94d049bb133111ebULL;
    return bits ^ (bits >> 31);
}

// exp(x) rounded once to f32 from an f64 evaluation: the correctly rounded
// value except within about 2^-29 ulp of a rounding midpoint, which is what
// host libm expf returns (the reference's f32::exp).  The device's f32 expf
// can differ by an ulp, and a near-tie draw then picks another token.
// Table of 2^(i/32) in the form the method below uses: the bits of the
// correctly rounded double 2^(i/32) minus i << 47.
static __constant__ uint64_t kExp2Tab[32] = {
    0x3ff0000000000000, 0x3fefd9b0d3158574, 0x3fefb5586cf9890f, 0x3fef9301d0125b51, 0x3fef72b83c7d517b,
    0x3fef54873168b9aa, 0x3fef387a6e756238, 0x3fef1e9df51fdee1, 0x3fef06fe0a31b715, 0x3feef1a7373aa9cb,
    0x3feedea64c123422, 0x3feece086061892d, 0x3feebfdad5362a27, 0x3feeb42b569d4f82, 0x3feeab07dd485429,
    0x3feea47eb03a5585, 0x3feea09e667f3bcd, 0x3fee9f75e8ec5f74, 0x3feea11473eb0187, 0x3feea589994cce13,
    0x3feeace5422aa0db, 0x3feeb737b0cdc5e5, 0x3feec49182a3f090, 0x3feed503b23e255d, 0x3feee89f995ad3ad,
    0x3feeff76f2fb5e47, 0x3fef199bdd85529c, 0x3fef3720dcef9069, 0x3fef5818dcfba487, 0x3fef7c97337b9b5f,
    0x3fefa4afa2a490da, 0x3fefd0765b6e4540};

// The reference's f32 exp: Rust's f32::exp is the C library's expf, which in
// glibc >= 2.28 is the exp2f-table method of ARM's optimized-routines
// (published; e_expf.c): x * 32/ln2 = k + r with |r| <= 1/2, exp(x) =
// 2^(k/32) * p(r) with a cubic p, all in double, then one rounding to float.
// This is that method in the operation order of glibc's FMA build (the one
// x86-64 hosts with FMA run): it equals that expf on every one of the 2^32
// float inputs (checked on the host against glibc 2.35); glibc's build for
// hosts without FMA rounds 2 of them differently.
// `tab` is kExp2Tab staged in LDS (a per-lane lookup in constant memory costs
// a memory round trip per call).  Branch-free, so that several calls
// interleave: the cases outside the method's range (x > 0x1.62e42ep6 gives
// +inf, x < -0x1.9fe368p6 and -inf give 0, NaN gives NaN) are selected after
// it runs on x clamped to [-104, 89].
__device__ __forceinline__ float expf_rounded(float x, const uint64_t *tab) {
    constexpr double N = 32.0, InvLn2N = 0x1.71547652b82fep+0 * N, Shift = 0x1.8p+52;
    constexpr double C0 = 0x1.c6af84b912394p-5 / (N * N * N), C1 = 0x1.ebfce50fac4f3p-3 / (N * N),
                     C2 = 0x1.62e42ff0c52d6p-1 / N;
    const double xd = double(fminf(fmaxf(x, -104.0f), 89.0f));
    double kd = InvLn2N * xd + Shift;  // rounds k to the nearest integer
    const uint64_t ki = uint64_t(__double_as_longlong(kd));
    kd -= Shift;
    const double r = fma(InvLn2N, xd, -kd);
    const double sc = __longlong_as_double(int64_t(tab[ki & 31] + (ki << 47)));
    const double z = fma(C0, r, C1), r2 = r * r;
    double y = fma(C2, r, 1.0);
    y = fma(z, r2, y);
    float e = float(y * sc);
    e = x > 0x1.62e42ep6f ? INFINITY : e;
    e = x < -0x1.9fe368p6f ? 0.0f : e;
    return x != x ? x + x : e;
}

// Copies kExp2Tab to `tab` (32 words of LDS); a barrier must follow before use.
__device__ __forceinline__ void stage_exp_table(uint64_t *tab) {
    for (int i = threadIdx.x; i < 32; i += blockDim.x) tab[i] = kExp2Tab[i];
}

// The lowest lane's value of v among the lanes where `has` holds, else `none`
// (a ballot and a lane read instead of a reduction).
__device__ __forceinline__ int first_lane_value(bool has, int v, int none) {
    const uint64_t mask = __ballot(has);
    return mask ? __builtin_amdgcn_readlane(v, int(__builtin_ctzll(mask))) : none;
}

// The reference's sequential f32 process (sequential_pick) run by a whole
// wave on p_i held in its registers: token t = j*R + k is pc[k] of lane j.
// Each p_i reaches every lane by a lane read (an exact copy), so all lanes
// compute the same sum and remainder; no memory is touched.
template <int RMAX>
__device__ __forceinline__ int wave_sequential_pick(const float (&pc)[RMAX], int R, int V, float u) {
#pragma clang fp contract(off)
    auto at = [&](int k, int j) {
        return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, pc[k]), j));
    };
    float sum = 0.0f;
    for (int j = 0; j < 64; ++j) {
#pragma unroll
        for (int k = 0; k < RMAX; ++k)
            if (k < R && j * R + k < V) sum = sum + at(k, j);
    }
    float sample = u * sum;
    for (int j = 0; j < 64; ++j) {
#pragma unroll
        for (int k = 0; k < RMAX; ++k) {
            if (k < R && j * R + k < V) {
                sample = sample - at(k, j);
                if (sample < 0.0f) return j * R + k;
            }
        }
    }
    return V - 1;
}

// choose_token's decision made by one wave on its own: lane l holds the
// logits of the contiguous run [l*R, l*R + R) of tokens in lg[0..R),
// R = ceil(V / 64) <= RMAX, and u is the generator's draw (made by the
// caller, so that it is ready before the logits are).  Every lane returns the
// token.  Nothing touches memory but the non-finite flag: a near-tie runs the
// sequential f32 process on the wave's registers (wave_sequential_pick), so
// waves of one workgroup never share scratch and need no barrier.  VC > 0
// compiles the choice for the vocabulary V = VC: the run length and every
// token mask are then constants, and the uniform branches on them vanish.
template <int RMAX, int VC = 0>
__device__ __forceinline__ int wave_choose_token(const float (&lg)[RMAX], int V, float temperature, float u,
                                                 const uint64_t *exp_tab, int *flags) {
    static_assert(RMAX == 1 || RMAX % 4 == 0, "runs are handled one or four tokens at a time");
    static_assert(VC >= 0 && (VC + 63) / 64 <= RMAX, "a fixed vocabulary fits the runs");
    if constexpr (VC > 0) {
        V = VC;
    } else {
        // V is hidden from the optimiser so that the f64 constants derived
        // from it are formed here, not hoisted out of a caller's step loop
        // and spilled.
        V = __builtin_amdgcn_readfirstlane(V);
        asm volatile("" : "+s"(V));
    }
    // Every per-token step below is straight-line code in blocks of four
    // tokens (a lane's tokens past V are masked by selects), so the f64
    // evaluations of neighbouring tokens overlap; only `k < R` branches, and
    // it is wave-uniform.  Since the runs ascend with the lane, the first
    // token with a property lies in the lowest lane that has one.
    const int R = (V + 63) / 64, i0 = int(threadIdx.x & 63) * R;
    float mx = -INFINITY;
    bool bad = false;
#pragma unroll
    for (int k = 0; k < RMAX; ++k) {
        if (k < R) {
            const bool v = i0 + k < V;
            bad = bad || (v && !isfinite(lg[k]));
            mx = v ? fmaxf(mx, lg[k]) : mx;
        }
    }
    mx = wave_max(mx);
    if (__ballot(bad) && threadIdx.x == 0) atomicOr(flags, 1);
    if (temperature == 0.0f) {
        int best = INT_MAX;
#pragma unroll
        for (int k = RMAX - 1; k >= 0; --k)
            if (k < R && i0 + k < V && lg[k] == mx) best = i0 + k;
        return first_lane_value(best != INT_MAX, best, 0);
    }
    float pc[RMAX];
    auto exps = [&](auto scaled) {
#pragma unroll
        for (int c = 0; c < (RMAX + 3) / 4; ++c) {
            if (4 * c < R) {
#pragma unroll
                for (int q = 0; q < (RMAX < 4 ? RMAX : 4); ++q) {
                    const int k = 4 * c + q;
                    const float p = expf_rounded(scaled(lg[k]), exp_tab);
                    pc[k] = k < R && i0 + k < V ? p : 0.0f;
                }
            }
        }
    };
    // (l - max) / T in f32 (gpu.rs:2037); division by 1 is exact, so T = 1
    // skips it.
    if (temperature == 1.0f)
        exps([&](float l) { return l - mx; });
    else
        exps([&](float l) { return (l - mx) / temperature; });
    double mine = 0.0;  // the masked tokens add exact zeros
#pragma unroll
    for (int k = 0; k < RMAX; ++k)
        if (k < R) mine += double(pc[k]);
    const double incl = wave_inclusive_sum(mine);
    const uint64_t sb = __builtin_bit_cast(uint64_t, incl);
    const double S = __builtin_bit_cast(
        double, (uint64_t(uint32_t(__builtin_amdgcn_readlane(int(uint32_t(sb >> 32)), 63))) << 32) |
                    uint32_t(__builtin_amdgcn_readlane(int(uint32_t(sb)), 63)));
    const double e = 0x1p-24, slack = 1e-12 * S;
    const double g = double(V + 2) * e * 1.01;
    const double s_lo = S * (1.0 - g) - slack, s_hi = S * (1.0 + g) + slack;
    const double beta = double(V + 2) * e * s_hi * 1.01 + slack;
    const double lo = double(u) * s_lo - beta, hi = double(u) * s_hi + beta;
    double prefix = incl - mine;
    int key = INT_MAX;
#pragma unroll
    for (int k = 0; k < RMAX; ++k) {
        if (k < R) {
            prefix += double(pc[k]);
            const bool first = key == INT_MAX && i0 + k < V && !(prefix < lo);
            key = first ? 2 * (i0 + k) + (prefix > hi ? 0 : 1) : key;
        }
    }
    key = first_lane_value(key != INT_MAX, key, INT_MAX);
    if (key == INT_MAX) return V - 1;
    if (!(key & 1)) return key >> 1;
    return wave_sequential_pick(pc, R, V, u);
}

// Random::unit (src/mesh.rs:263-265): one SplitMix64 draw per sampled token.
__device__ __forceinline__ float rng_unit(uint64_t &state) {
    return float(uint32_t(splitmix_next(state) >> 40)) / 16777216.0f;
}

}  // namespace meshgpt::kern
