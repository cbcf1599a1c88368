// Generation by recomputing a short window, every token of it in one launch
// (gpu.rs:2006-2053: past the context the window slides, positions restart at
// 0 and each token needs the whole window again).
//
// What bounds it is the chain of dependent steps of one token, not work: the
// default model's window (32 rows of 32 channels, two blocks) is 0.2 MFLOP.  As
// one launch per operator a token took seven launches of 3-9 us (48 us); in one
// launch it takes 7.1 us, about half of it the mesh layers (a wave issues some
// 40 dependent instructions for a layer of q, k and v).  A workgroup keeps a
// sequence's window to itself from token to token:
//  - a row lies in 16 lanes, channel CPL l + j in register j of lane l (CPL =
//    W / 16), four rows a wave: a mesh layer's partner is another register, or
//    one DPP move inside the 16 lanes, for every stride of both connectivities;
//    row and head sums are DPP sums; nothing of a row leaves its lanes but q, k,
//    v and the attention output;
//  - these meet in LDS, and each wave takes (head, 16 queries) units of the
//    attention on the FP32 matrix cores in the two products of train_attn.hip;
//  - the last block works for the window's last row only, but for its k and v;
//  - every wave makes the same draw from the logits in LDS, so the new token
//    needs no hand-off.
// Two barriers a block and two for the head remain.  240 tokens from a prompt of
// 17 (W32, context 32, two blocks), one sequence: 11.7 ms before, 1.70 now; W64,
// context 32: 13.1 and 2.3; W128, context 64: 17.5 and 8.0.  The last family's
// sixteen waves leave 128 registers a lane, and five of its six forms spill four to
// eight of them (20-36 bytes of scratch a lane).
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "dpp.hpp"
#include "kernels.hpp"
#include "sampler.hpp"

namespace meshgpt::kern {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr float kRmsEps = 1e-5f;  // src/gpt/mod.rs:38
// (f64(1e-12f))^2 rounded to f32: the XSA norm floor of reference.rs:591
constexpr float kXsaFloor = float(double(1e-12f) * double(1e-12f));
constexpr float kLog2e = 1.4426950408889634f, kLn2 = 0.6931471805599453f;
constexpr int kRing = 2 * kWindowRows;  // tokens kept in LDS
constexpr size_t kWindowLds = 160 * 1024;  // a CU's

// What a value is multiplied by on its way into the meshes and out of them:
// SCALED ones are carried times log2(e), which the ELU's exponential would
// otherwise multiply in (Shape::wide: their own units).
template <bool SCALED>
struct Units {
    static constexpr float in = SCALED ? kLog2e : 1.0f, out = SCALED ? kLn2 : 1.0f;
};

// The ELU in these units, of t = z or z log2(e): z, or e^z - 1 where z is not
// positive, NaN included.  A select on t, which does not wait for the
// exponential, keeps the dependent chain one step shorter than a maximum.
template <bool SCALED>
__device__ __forceinline__ float elu_units(float t) {
    const float p = __builtin_amdgcn_exp2f(SCALED ? t : t * kLog2e);
    return t > 0.0f ? t : SCALED ? __builtin_fmaf(p, kLog2e, -kLog2e) : p - 1.0f;
}

// v of the lane 16 (32) away combined with the lane's own: register swaps
// between rows of 16 lanes, no LDS round trip.
template <class F>
__device__ __forceinline__ float across_groups(float v, F f) {
    const auto s = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), false, false);
    v = f(__builtin_bit_cast(float, int(s[0])), __builtin_bit_cast(float, int(s[1])));
    const auto t = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), false, false);
    return f(__builtin_bit_cast(float, int(t[0])), __builtin_bit_cast(float, int(t[1])));
}
__device__ __forceinline__ float sum_groups(float v) {
    return across_groups(v, [](float a, float b) { return a + b; });
}

// v of lane l ^ M inside 16 lanes.
template <int M>
__device__ __forceinline__ float lane_xor(float v, int l16) {
    static_assert(M == 1 || M == 2 || M == 4, "half the lanes of a head: two, four or eight heads in 16");
    if constexpr (M == 1)
        return dpp_move<0xB1>(v, v);  // quad_perm [1,0,3,2]
    else if constexpr (M == 2)
        return dpp_move<0x4E>(v, v);  // quad_perm [2,3,0,1]
    const float down = dpp_move<0x124>(v, v), up = dpp_move<0x12C>(v, v);  // row_ror:4, :12
    return (l16 & 4) ? down : up;
}

// Lane l of each 16 gets v of lane (l + K) mod 16.
template <int K>
__device__ __forceinline__ float lanes_up(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x120 + (16 - K), 0xf, 0xf, true));
}

// p[j] = the value ST channels on (mod W) from x[j]'s channel.
template <int CPL, int ST>
__device__ __forceinline__ void partner(const float (&x)[CPL], float (&p)[CPL]) {
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
        if constexpr (ST >= CPL)
            p[j] = lanes_up<ST / CPL>(x[j]);
        else
            p[j] = j + ST < CPL ? x[(j + ST) % CPL] : lanes_up<1>(x[(j + ST) % CPL]);
    }
}

// N mesh stacks of one depth (reference.rs:422-453) on x, in place, in the
// meshes' units; stack i's weights at w[i].  Strides are 1, or
// 2^(layer mod log2 W) (W = 16 CPL).  Two layers' weights are in registers or
// on their way while a third is computed.
template <bool BF, bool SCALED, int N, int CPL>
struct Stacks {
    static constexpr int W = 16 * CPL, LEVELS = CPL == 2 ? 5 : (CPL == 4 ? 6 : 7);
    float2 buf[2][N][CPL];
    const float *const (&w)[N];
    const int depth, l16;
    __device__ __forceinline__ void load(int l, int to) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float4 *src =
                reinterpret_cast<const float4 *>(w[i] + size_t(min(l, depth - 1)) * 2 * W + 2 * CPL * l16);
#pragma unroll
            for (int j = 0; j < CPL / 2; ++j) {
                const float4 t = src[j];
                buf[to][i][2 * j] = make_float2(t.x, t.y);
                buf[to][i][2 * j + 1] = make_float2(t.z, t.w);
            }
        }
    }
    // Layer l on buffer B; true at the last.
    template <int B>
    __device__ __forceinline__ bool step(float (&x)[N][CPL], int l) {
        float p[N][CPL];
        if constexpr (BF) {
            switch (l % LEVELS) {
                case 0: partners<1>(x, p); break;
                case 1: partners<2>(x, p); break;
                case 2: partners<4>(x, p); break;
                case 3: partners<8>(x, p); break;
                case 4: partners<16>(x, p); break;
                case 5: partners<W == 32 ? 1 : 32>(x, p); break;
                default: partners<W == 128 ? 64 : 1>(x, p); break;
            }
        } else {
            partners<1>(x, p);
        }
        const bool last = l + 1 == depth;
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const float z = x[i][j] * buf[B][i][j].x + p[i][j] * buf[B][i][j].y;
                x[i][j] = last ? z : elu_units<SCALED>(z);
            }
        if (!last) load(l + 2, B);
        return last;
    }
    template <int ST>
    static __device__ __forceinline__ void partners(const float (&x)[N][CPL], float (&p)[N][CPL]) {
#pragma unroll
        for (int i = 0; i < N; ++i) partner<CPL, ST>(x[i], p[i]);
    }
    __device__ __forceinline__ void all(float (&x)[N][CPL]) {
        load(0, 0);
        load(1, 1);
#pragma nounroll
        for (int l = 0;; l += 2)
            if (step<0>(x, l) || step<1>(x, l + 1)) return;
    }
};

template <bool BF, bool SCALED, int N, int CPL>
__device__ __forceinline__ void stacks(float (&x)[N][CPL], const float *const (&w)[N], int depth, int l16) {
    Stacks<BF, SCALED, N, CPL> s{{}, w, depth, l16};
    s.all(x);
}

// n = RMSNorm(x) times `unit` (reference.rs:392-409).
template <int CPL>
__device__ __forceinline__ void norm(const float (&x)[CPL], float (&n)[CPL], float unit) {
    float sq = 0.0f;
#pragma unroll
    for (int j = 0; j < CPL; ++j) sq = fmaf(x[j], x[j], sq);
    const float inv = rsqrtf(group_sum<16>(sq) * (1.0f / float(16 * CPL)) + kRmsEps) * unit;
#pragma unroll
    for (int j = 0; j < CPL; ++j) n[j] = x[j] * inv;
}

template <int CPL>
__device__ __forceinline__ void put_row(float *row, const float (&x)[CPL]) {
    if constexpr (CPL == 2) {
        *reinterpret_cast<float2 *>(row) = make_float2(x[0], x[1]);
    } else {
#pragma unroll
        for (int j = 0; j < CPL; j += 4)
            *reinterpret_cast<float4 *>(row + j) = make_float4(x[j], x[j + 1], x[j + 2], x[j + 3]);
    }
}

__device__ __forceinline__ v4f mfma(float a, float b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <int N>
__device__ __forceinline__ void take(const float *from, float (&to)[N]) {
    if constexpr (N == 2) {
        const float2 t = *reinterpret_cast<const float2 *>(from);
        to[0] = t.x, to[1] = t.y;
    } else {
#pragma unroll
        for (int i = 0; i < N; i += 4) {
            const float4 t = *reinterpret_cast<const float4 *>(from + i);
            to[i] = t.x, to[i + 1] = t.y, to[i + 2] = t.z, to[i + 3] = t.w;
        }
    }
}

// to[0..n) = from[0..n) by the whole workgroup, n a multiple of four.
__device__ __forceinline__ void copy4(const float *from, float *to, int n) {
    for (int i = 4 * int(threadIdx.x); i < n; i += 4 * int(blockDim.x))
        *reinterpret_cast<float4 *>(to + i) = *reinterpret_cast<const float4 *>(from + i);
}

// Causal attention of queries [16 qt, 16 qt + 16) of one head whose columns
// start at Q, K and V, then XSA against each query's own value row; the result
// replaces the queries.  The operand layouts are those of train_attn.hip.
template <int HD, int KB, int STRIDE>
__device__ __forceinline__ void attend(float *Q, const float *K, const float *V, int qt, int lane, float scale_log2,
                                       bool xsa) {
    constexpr int KS = HD / 4, DB = (HD + 15) / 16;
    const int jq = lane & 15, g = lane >> 4, qi = 16 * qt + jq;
    float q[KS];
    take(Q + qi * STRIDE + KS * g, q);
#pragma unroll
    for (int i = 0; i < KS; ++i) q[i] *= scale_log2;
    v4f sc[KB];
    float mx = -INFINITY;
#pragma unroll
    for (int b = 0; b < KB; ++b) {
        if (b > qt) continue;
        float k[KS];
        take(K + (16 * b + jq) * STRIDE + KS * g, k);
        sc[b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < KS; ++i) sc[b] = mfma(k[i], q[i], sc[b]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (16 * b + 4 * g + r > qi) sc[b][r] = -INFINITY;
            mx = fmaxf(mx, sc[b][r]);
        }
    }
    mx = across_groups(mx, [](float a, float b) { return fmaxf(a, b); });
    float sum = 0.0f;
    v4f acc[DB], odd[DB];  // two chains: a narrow head has one product a key
#pragma unroll
    for (int d = 0; d < DB; ++d) acc[d] = odd[d] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < KB; ++b) {
        if (b > qt) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float p = __builtin_amdgcn_exp2f(sc[b][r] - mx);
            sum += p;
            const float *row = V + (16 * b + 4 * g + r) * STRIDE + jq;
#pragma unroll
            for (int d = 0; d < DB; ++d) (r & 1 ? odd : acc)[d] = mfma(row[16 * d], p, (r & 1 ? odd : acc)[d]);
        }
    }
    const float inv = 1.0f / sum_groups(sum);
    float dot = 0.0f, vsq = 0.0f;
    float4 own[DB];
#pragma unroll
    for (int d = 0; d < DB; ++d) {
        // Lanes past the head's dims (head width 8: the upper groups, whose
        // columns are the next head's or padding) add zeros.
        const bool live = 16 * d + 4 * g < HD;
        own[d] = live ? *reinterpret_cast<const float4 *>(V + qi * STRIDE + 16 * d + 4 * g) : make_float4(0, 0, 0, 0);
        acc[d] = live ? (acc[d] + odd[d]) * inv : v4f{0.0f, 0.0f, 0.0f, 0.0f};
        dot += acc[d][0] * own[d].x + acc[d][1] * own[d].y + acc[d][2] * own[d].z + acc[d][3] * own[d].w;
        vsq += own[d].x * own[d].x + own[d].y * own[d].y + own[d].z * own[d].z + own[d].w * own[d].w;
    }
    const float iv = rsqrtf(fmaxf(sum_groups(vsq), kXsaFloor)), c = xsa ? sum_groups(dot) * iv : 0.0f;
#pragma unroll
    for (int d = 0; d < DB; ++d)
        if (16 * d + 4 * g < HD)
            *reinterpret_cast<float4 *>(Q + qi * STRIDE + 16 * d + 4 * g) =
                make_float4(acc[d][0] - c * (own[d].x * iv), acc[d][1] - c * (own[d].y * iv),
                            acc[d][2] - c * (own[d].z * iv), acc[d][3] - c * (own[d].w * iv));
}

// A workgroup of NW waves per sequence: windows of up to 4 NW rows.  STAGED: the
// blocks' weights and the token vectors are copied to LDS first.
template <int CPL, int HD, int NW, bool STAGED, bool BF, bool SCALED>
__global__ void __launch_bounds__(64 * NW) window_kernel(WindowArgs a) {
    constexpr int W = 16 * CPL, H = W / HD, LPH = 16 / H, ROWS = 4 * NW, KB = ROWS / 16, STRIDE = W + 4;
    using U = Units<SCALED>;
    constexpr int GROUP = CPL * NW <= 32 ? 3 : 1;  // stacks side by side, as registers allow
    static_assert(H == 2 || H == 4 || H == 8, "a head is two, four or eight whole lanes");
    extern __shared__ __align__(16) float lds[];
    // The matrix products read whole 16-dim blocks, past a narrow last head.
    float *Q = lds, *K = Q + ROWS * STRIDE, *V = K + ROWS * STRIDE, *xn = V + ROWS * STRIDE + 16, *logits = xn + W;
    uint32_t *ring = reinterpret_cast<uint32_t *>(logits + 256);
    uint64_t *tab = reinterpret_cast<uint64_t *>(ring + kRing);
    float *staged = reinterpret_cast<float *>(tab + 32);  // weights, then token vectors
    const int b = int(blockIdx.x), lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
    const int l16 = lane & 15, row = 4 * wave + (lane >> 4), half = HD / 2, V_ = a.V;
    uint32_t *tokens = a.tokens + size_t(b) * a.tok_stride;
    const int len0 = a.len[b];
    for (int i = max(0, len0 - kWindowRows) + int(threadIdx.x); i < len0; i += 64 * NW) ring[i & (kRing - 1)] = tokens[i];
    stage_exp_table(tab);
    uint64_t rng = a.rng[b];
    // The rotation of this lane's channels at its row's position.
    float2 turn[CPL];
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
        const int d = (CPL * l16 + j) % HD;
        turn[j] = a.rotate && row < a.context ? a.rope[size_t(row) * half + d % half] : make_float2(1.0f, 0.0f);
        if (d < half) turn[j].y = -turn[j].y;
    }
    const size_t gA = size_t(2) * W * a.A, gF = size_t(2) * W * a.F;
    const float *weights = a.w, *E = a.E;
    if constexpr (STAGED) {
        const int nw = a.L * int(4 * gA + gF);
        copy4(a.w, staged, nw);
        copy4(a.E, staged + nw, a.V * W);
        weights = staged;
        E = staged + nw;
    }
    __syncthreads();

    for (int s = 0; s < a.steps; ++s) {
        const int length = len0 + s, win = min(length, a.context), start = length - win;
        const int last = win - 1, last_wave = last >> 2;
        float x[CPL];
        {
            const uint32_t tok = ring[(start + min(row, last)) & (kRing - 1)];
            const float *e = E + size_t(tok) * W + CPL * l16;
            take(e, x);
        }
        for (int l = 0; l < a.L; ++l) {
            const float *w = weights + size_t(l) * (4 * gA + gF);
            const bool tail = l + 1 == a.L;  // only the last row goes on, past its keys and values
            const bool goes_on = !tail || wave == last_wave;
            float qkv[3][CPL];
            norm(x, qkv[0], U::in);
#pragma unroll
            for (int j = 0; j < CPL; ++j) qkv[1][j] = qkv[2][j] = qkv[0][j];
            if constexpr (GROUP == 3) {
                const float *const ws[3] = {w, w + gA, w + 2 * gA};
                stacks<BF, SCALED>(qkv, ws, a.A, l16);
            } else {
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    if (i == 0 && !goes_on) continue;
                    float (&one)[1][CPL] = reinterpret_cast<float(&)[1][CPL]>(qkv[i]);
                    const float *const ws[1] = {w + i * gA};
                    stacks<BF, SCALED>(one, ws, a.A, l16);
                }
            }
            // QK-Norm, then slice RoPE (reference.rs:174-193), each when on.
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                float inv = U::out;
                if (a.qk_norm) {
                    float sq = 0.0f;
#pragma unroll
                    for (int j = 0; j < CPL; ++j) sq = fmaf(qkv[i][j], qkv[i][j], sq);
                    inv = rsqrtf(group_sum<LPH>(sq) * (1.0f / float(HD)) + kRmsEps * U::in * U::in);
                }
#pragma unroll
                for (int j = 0; j < CPL; ++j) qkv[i][j] *= inv;
                if (a.rotate) {
                    float o[CPL];
#pragma unroll
                    for (int j = 0; j < CPL; ++j) o[j] = lane_xor<LPH / 2>(qkv[i][j], l16);
#pragma unroll
                    for (int j = 0; j < CPL; ++j) qkv[i][j] = qkv[i][j] * turn[j].x + o[j] * turn[j].y;
                }
            }
            float *at = Q + row * STRIDE + CPL * l16;
#pragma unroll
            for (int j = 0; j < CPL; ++j) qkv[2][j] *= U::out;
            put_row(at, qkv[0]);
            put_row(at + ROWS * STRIDE, qkv[1]);
            put_row(at + 2 * ROWS * STRIDE, qkv[2]);
            if (a.kc && s + 1 == a.steps && row <= last) {
                // The cache as the decode of this length leaves it: every row of the window.
                const int c0 = CPL * l16;
#pragma unroll
                for (int j = 0; j < CPL; ++j) {
                    const int c = c0 + j;
                    const size_t to = size_t(l) * a.layer_elems +
                                      (size_t(b * H + c / HD) * a.cap + row) * HD + c % HD;
                    a.kc[to] = qkv[1][j];
                    a.vc[to] = qkv[2][j];
                }
            }
            __syncthreads();
            for (int u = wave; u < H * KB; u += NW) {
                const int qt = u / H, h = u % H;
                if (16 * qt > last || (tail && qt != last >> 4)) continue;
                attend<HD, KB, STRIDE>(Q + h * HD, K + h * HD, V + h * HD, qt, lane, a.scale_log2, a.xsa);
            }
            __syncthreads();
            if (goes_on) {
                float z[1][CPL];
                take(Q + row * STRIDE + CPL * l16, z[0]);
#pragma unroll
                for (int j = 0; j < CPL; ++j) z[0][j] *= U::in;
                const float *const wp[1] = {w + 3 * gA}, *const wf[1] = {w + 4 * gA};
                stacks<BF, SCALED>(z, wp, a.A, l16);
#pragma unroll
                for (int j = 0; j < CPL; ++j) x[j] = fmaf(z[0][j], U::out, x[j]);
                norm(x, z[0], U::in);
                stacks<BF, SCALED>(z, wf, a.F, l16);
#pragma unroll
                for (int j = 0; j < CPL; ++j) x[j] = fmaf(z[0][j], U::out, x[j]);
            }
        }
        if (row == last) {
            float n[CPL];
            norm(x, n, 1.0f);
            put_row(xn + CPL * l16, n);
        }
        __syncthreads();
        // The tied head: 16 lanes a token.
        {
            float n[CPL];
            take(xn + CPL * l16, n);
            for (int t = row; t < V_; t += ROWS) {
                float e[CPL], dot = 0.0f;
                take(E + size_t(t) * W + CPL * l16, e);
#pragma unroll
                for (int j = 0; j < CPL; ++j) dot = fmaf(n[j], e[j], dot);
                dot = group_sum<16>(dot);
                if (l16 == 0) logits[t] = dot;
            }
        }
        const float u = a.temperature == 0.0f ? 0.0f : rng_unit(rng);  // greedy draws nothing
        __syncthreads();
        uint32_t token;
        if (V_ <= 64) {
            const float lg[1] = {lane < V_ ? logits[lane] : 0.0f};
            token = uint32_t(wave_choose_token(lg, V_, a.temperature, u, tab, a.flags));
        } else {
            float lg[4];
            const int run = (V_ + 63) / 64;
#pragma unroll
            for (int k = 0; k < 4; ++k) lg[k] = k < run && run * lane + k < V_ ? logits[run * lane + k] : 0.0f;
            token = uint32_t(wave_choose_token(lg, V_, a.temperature, u, tab, a.flags));
        }
        // Every wave writes the same word and reads its own write.
        if (lane == 0) ring[length & (kRing - 1)] = token;
        if (threadIdx.x == 0) tokens[length] = token;
        __builtin_amdgcn_wave_barrier();
    }
    for (int t = int(threadIdx.x); t < V_; t += 64 * NW) a.logits[size_t(b) * V_ + t] = logits[t];
    if (threadIdx.x == 0) {
        a.len[b] = len0 + a.steps;
        a.rng[b] = rng;
    }
}

// Bytes of LDS of a workgroup of `waves` waves, and of the weights and token
// vectors that it may hold beside them.
size_t window_lds(int W, int waves) { return (3 * 4 * size_t(waves) * (W + 4) + 16 + W + 256 + kRing) * 4 + 32 * 8; }
size_t window_weights(const Shape &s, size_t layers, size_t vocab) {
    return (layers * 2 * s.W * (4 * s.A + s.F) + vocab * s.W) * 4;
}

template <int CPL, int HD, int NW>
void launch_window(const Shape &s, const WindowArgs &a, int batch, hipStream_t stream) {
    const size_t lds = window_lds(16 * CPL, NW), staged = window_weights(s, size_t(a.L), size_t(a.V));
    auto launch = [&](auto kernel, size_t bytes) {
        // A refusal is the thread's last error, which the model's next wait reports.
        if (bytes > 65536 && hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)) != hipSuccess)
            return;
        hipLaunchKernelGGL(kernel, dim3(batch), dim3(64 * NW), bytes, stream, a);
    };
    if (s.wide) {
        a.butterfly ? launch(window_kernel<CPL, HD, NW, false, true, false>, lds)
                    : launch(window_kernel<CPL, HD, NW, false, false, false>, lds);
        return;
    }
    if constexpr (NW == 8) {
        if (lds + staged <= kWindowLds) {
            a.butterfly ? launch(window_kernel<CPL, HD, NW, true, true, true>, lds + staged)
                        : launch(window_kernel<CPL, HD, NW, true, false, true>, lds + staged);
            return;
        }
    }
    a.butterfly ? launch(window_kernel<CPL, HD, NW, false, true, true>, lds)
                : launch(window_kernel<CPL, HD, NW, false, false, true>, lds);
}

// f(CPL, HD) for the widths and head widths that have a kernel (2 to 8 heads);
// false without one.
template <class F>
bool by_window_shape(const Shape &s, F &&f) {
    auto width = [&](auto cpl) {
        constexpr int C = decltype(cpl)::value;
        switch (s.hd) {
            case 8:
                if constexpr (C < 8) return f(cpl, std::integral_constant<int, 8>{}), true;
                return false;
            case 16: return f(cpl, std::integral_constant<int, 16>{}), true;
            case 32:
                if constexpr (C > 2) return f(cpl, std::integral_constant<int, 32>{}), true;
                return false;
            case 64:
                if constexpr (C > 4) return f(cpl, std::integral_constant<int, 64>{}), true;
                return false;
            default: return false;
        }
    };
    switch (s.W) {
        case 32: return width(std::integral_constant<int, 2>{});
        case 64: return width(std::integral_constant<int, 4>{});
        case 128: return width(std::integral_constant<int, 8>{});
        default: return false;
    }
}

}  // namespace

bool window_supported(const Shape &s, size_t context) {
    return context <= size_t(kWindowRows) && s.V <= 256 && s.hd == s.hdp && by_window_shape(s, [](auto, auto) {});
}

// Workgroups run 256 at a time, a CU's LDS or wave slots each (windows of up to
// 32 narrow rows overlap somewhat), and a layer of a stack takes the time below;
// the last block works for one row past its keys.  Measured between one and
// twelve blocks, stacks of 4 to 9 layers and 16 to 4096 sequences: within 15 %
// wherever another route comes near.
double window_us(const Shape &s, size_t context, size_t layers, size_t batch, size_t vocab) {
    const bool wide = context > kWindowRows / 2, staged = !wide && window_lds(s.W, 8) + window_weights(s, layers, vocab) <= kWindowLds;
    const double layer = s.W == 32 ? (wide ? 0.22 : 0.15) : s.W == 64 ? (wide ? 0.335 : 0.22) : wide ? 1.03 : staged ? 0.33 : 0.53;
    return double((batch + 255) / 256) * (double(layers) - 0.33) * double(4 * s.A + s.F) * layer;
}

void window_generate(const Shape &s, WindowArgs a, int batch, hipStream_t stream) {
    a.scale_log2 = float(1.4426950408889634 / std::sqrt(double(s.hd)));
    by_window_shape(s, [&](auto cpl, auto hd) {
        constexpr int C = decltype(cpl)::value, D = decltype(hd)::value;
        a.context <= kWindowRows / 2 ? launch_window<C, D, 8>(s, a, batch, stream)
                                     : launch_window<C, D, 16>(s, a, batch, stream);
    });
}

}  // namespace meshgpt::kern
