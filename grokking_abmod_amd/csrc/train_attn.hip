// Training attention for gfx950 on the FP32 matrix cores: the causal softmax
// forward with its log-sum-exp and the XSA epilogue (reference.rs:510-554,
// 577-603), and its backward (dq, dk, dv) from the saved log-sum-exp.
//
// A workgroup of four waves owns 64 rows of one (sequence, head), 16 a wave:
// query rows in the forward and for dq, key rows for dk and dv.  The other
// side streams through LDS in tiles of 64 rows (32 at head width 128), the
// next tile's loads in flight in registers while this one is multiplied.
// Every product runs on v_mfma_f32_16x16x4f32 in one of two operand forms, so
// nothing leaves registers in between: a tile's rows against the wave's own
// rows (contracted over the head's dims, four rows of ONE own row left in
// each lane), then the tile's columns against that result (contracted over
// the tile's rows), whose B operand layout is exactly what the first product
// left.
//
// What bounds it: the matrix cores' FP32 rate.  Eight sequences of 512 rows,
// 8 heads of 64 dims: 33.8k 16 x 16 blocks of 32 (forward), 48 (dq) and 64
// (dk, dv) instructions of 32 cycles, 14 and 49 us at full rate on 1024 SIMDs.
// Measured 60 us forward and 166 us backward (512 workgroups, two a CU, so a
// wave waits on its own LDS reads and softmax); one thread per (row, head),
// each reading its rows from memory by itself, took 5.4 and 20.9 ms.
// Head widths that are no power of two are padded with zeros in LDS to 16,
// 32, 64 or 128 dims.  Rows of W + 4 floats in LDS keep the 16-byte reads of
// eight neighbouring rows and the 4-byte reads of four rows, 16 dims each,
// on distinct banks.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "train.hpp"

namespace meshgpt::kern::train {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr float kXsaFloor = float(double(1e-12f) * double(1e-12f));  // XSA_EPSILON^2
constexpr int kWaves = 4;
constexpr int kOwn = 16 * kWaves;  // rows of a workgroup

template <int HDP>
struct Tiling {
    static constexpr int KS = HDP / 4;               // k-steps of a row product: dim = KS * (lane / 16) + step
    static constexpr int DB = HDP / 16;              // 16-dim blocks of an output row
    static constexpr int T = HDP == 128 ? 32 : 64;   // rows of an LDS tile
    static constexpr int KB = T / 16;                // 16-row blocks of a tile
    static constexpr int STRIDE = HDP + 4;           // floats between LDS rows
    static constexpr int NV = T * HDP / 4 / (64 * kWaves);  // 16-byte pieces of a tile per thread
};

struct AttnShape {
    int sequence, W, H, hd, tiles, pairs, xsa;
    float scale, scale_log2;
};

// D = A B + C of one 16x16x4 block: lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16] and holds D[4 (l / 16) + r][l % 16] in element r.
__device__ __forceinline__ v4f mfma(float a, float b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float across_groups(float v) {
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

// Four floats of a head's row from dim d on; dims past hd are zero.  Rows are
// 16-byte aligned when hd is a multiple of four (the row stride W = H hd then
// is one as well).
__device__ __forceinline__ float4 row4(const float *row, int d, int hd) {
    if ((hd & 3) == 0) return d < hd ? *reinterpret_cast<const float4 *>(row + d) : make_float4(0, 0, 0, 0);
    return make_float4(d < hd ? row[d] : 0.0f, d + 1 < hd ? row[d + 1] : 0.0f, d + 2 < hd ? row[d + 2] : 0.0f,
                       d + 3 < hd ? row[d + 3] : 0.0f);
}

__device__ __forceinline__ void store4(float *row, int d, int hd, float4 v) {
    if ((hd & 3) == 0) {
        if (d < hd) *reinterpret_cast<float4 *>(row + d) = v;
        return;
    }
    const float t[4] = {v.x, v.y, v.z, v.w};
    for (int e = 0; e < 4; ++e)
        if (d + e < hd) row[d + e] = t[e];
}

// A tile of one array in flight: this thread's 16-byte pieces of rows
// [t0, t0 + T) (rows past the sequence are zero).
template <int HDP>
struct Piece {
    using C = Tiling<HDP>;
    float4 v[C::NV];
    __device__ __forceinline__ void load(const float *base, int t0, const AttnShape &s) {
#pragma unroll
        for (int i = 0; i < C::NV; ++i) {
            const int at = i * 64 * kWaves + int(threadIdx.x), row = t0 + at / (HDP / 4), d = at % (HDP / 4) * 4;
            v[i] = row < s.sequence ? row4(base + size_t(row) * s.W, d, s.hd) : make_float4(0, 0, 0, 0);
        }
    }
    __device__ __forceinline__ void store(float *lds) const {
#pragma unroll
        for (int i = 0; i < C::NV; ++i) {
            const int at = i * 64 * kWaves + int(threadIdx.x);
            *reinterpret_cast<float4 *>(lds + at / (HDP / 4) * C::STRIDE + at % (HDP / 4) * 4) = v[i];
        }
    }
};

// The wave's own rows as the B operand of a row product: lane holds
// row[lane % 16][KS (lane / 16) + step] times `scale`.
template <int HDP>
__device__ __forceinline__ void own_rows(const float *base, int row, const AttnShape &s, int g, float scale,
                                         float (&op)[HDP / 4]) {
#pragma unroll
    for (int t = 0; t < HDP / 16; ++t) {
        const float4 v = row < s.sequence ? row4(base + size_t(row) * s.W, HDP / 4 * g + 4 * t, s.hd)
                                          : make_float4(0, 0, 0, 0);
        op[4 * t] = v.x * scale;
        op[4 * t + 1] = v.y * scale;
        op[4 * t + 2] = v.z * scale;
        op[4 * t + 3] = v.w * scale;
    }
}

// out[b][r] += tile row 16 b + 4 (lane / 16) + r . own row lane % 16
template <int HDP>
__device__ __forceinline__ void row_product(const float *tile, const float (&own)[HDP / 4], int jq, int g,
                                            v4f (&out)[Tiling<HDP>::KB]) {
    using C = Tiling<HDP>;
#pragma unroll
    for (int t = 0; t < C::KS / 4; ++t) {
        float4 a[C::KB];
#pragma unroll
        for (int b = 0; b < C::KB; ++b)
            a[b] = *reinterpret_cast<const float4 *>(tile + (16 * b + jq) * C::STRIDE + C::KS * g + 4 * t);
#pragma unroll
        for (int b = 0; b < C::KB; ++b) out[b] = mfma(a[b].x, own[4 * t], out[b]);
#pragma unroll
        for (int b = 0; b < C::KB; ++b) out[b] = mfma(a[b].y, own[4 * t + 1], out[b]);
#pragma unroll
        for (int b = 0; b < C::KB; ++b) out[b] = mfma(a[b].z, own[4 * t + 2], out[b]);
#pragma unroll
        for (int b = 0; b < C::KB; ++b) out[b] = mfma(a[b].w, own[4 * t + 3], out[b]);
    }
}

// acc[d][r] += sum over the tile's rows of tile[row][16 d + 4 (lane / 16) + r] * w[row][own row lane % 16]
template <int HDP>
__device__ __forceinline__ void column_product(const float *tile, const v4f (&w)[Tiling<HDP>::KB], int jq, int g,
                                               v4f (&acc)[Tiling<HDP>::DB]) {
    using C = Tiling<HDP>;
#pragma unroll
    for (int b = 0; b < C::KB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float *row = tile + (16 * b + 4 * g + r) * C::STRIDE + jq;
#pragma unroll
            for (int d = 0; d < C::DB; ++d) acc[d] = mfma(row[16 * d], w[b][r], acc[d]);
        }
}

// Workgroup i runs on XCD i % 8; the tiles of one (sequence, head) stay on one
// XCD, which then holds its rows in its L2, and the tile with the most work
// comes first.
__device__ __forceinline__ bool place(const AttnShape &s, bool last_first, int &pair, int &tile) {
    const int xcd = int(blockIdx.x) % 8, j = int(blockIdx.x) / 8;
    pair = xcd + 8 * (j / s.tiles);
    tile = last_first ? s.tiles - 1 - j % s.tiles : j % s.tiles;
    return pair < s.pairs;
}

// lse[row * H + h] = log2 of the sum of 2^(score log2 e): base 2, as the
// backward below reads it.
template <int HDP>
__global__ void __launch_bounds__(64 * kWaves)
matrix_forward_kernel(AttnShape s, const float *__restrict__ q, const float *__restrict__ k,
                      const float *__restrict__ v, float *__restrict__ y, float *__restrict__ z,
                      float *__restrict__ lse) {
    using C = Tiling<HDP>;
    __shared__ __align__(16) float Ks[C::T * C::STRIDE], Vs[C::T * C::STRIDE];
    int pair, tile;
    if (!place(s, true, pair, tile)) return;
    const int h = pair % s.H, lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
    const int jq = lane & 15, g = lane >> 4;
    const size_t first = size_t(pair / s.H) * s.sequence, base = first * s.W + h * s.hd;
    const int mine = tile * kOwn + wave * 16, qi = mine + jq;  // the wave's first query, the lane's
    float qop[C::KS];
    own_rows<HDP>(q + base, qi, s, g, s.scale_log2, qop);
    v4f acc[C::DB];
#pragma unroll
    for (int d = 0; d < C::DB; ++d) acc[d] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f;
    const int ntile = (min(tile * kOwn + kOwn, s.sequence) - 1) / C::T + 1;
    Piece<HDP> pk, pv;
    pk.load(k + base, 0, s);
    pv.load(v + base, 0, s);
    for (int t = 0; t < ntile; ++t) {
        const int t0 = t * C::T;
        __syncthreads();  // the previous tile's readers are done
        pk.store(Ks);
        pv.store(Vs);
        __syncthreads();
        if (t + 1 < ntile) {
            pk.load(k + base, t0 + C::T, s);
            pv.load(v + base, t0 + C::T, s);
        }
        if (t0 > mine + 15) continue;  // the wave's queries all precede the tile
        v4f sc[C::KB];
#pragma unroll
        for (int b = 0; b < C::KB; ++b) sc[b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        row_product<HDP>(Ks, qop, jq, g, sc);
        const bool diag = t0 + C::T - 1 > mine;
        float mx = -INFINITY;
#pragma unroll
        for (int b = 0; b < C::KB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (diag && t0 + 16 * b + 4 * g + r > qi) sc[b][r] = -INFINITY;
                mx = fmaxf(mx, sc[b][r]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float mn = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f(m - mn);
        float sum = 0.0f;
#pragma unroll
        for (int b = 0; b < C::KB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sc[b][r] = __builtin_amdgcn_exp2f(sc[b][r] - mn);
                sum += sc[b][r];
            }
        l = l * alpha + sum;
        m = mn;
#pragma unroll
        for (int d = 0; d < C::DB; ++d) acc[d] *= alpha;
        // A later row's value that is not finite must not reach this query
        // through its zero probability: such a tile (only one past the wave's
        // first query can hold it) is added key by key with a select.
        bool plain = true;
        if (diag) {
            float worst = 0.0f;
#pragma unroll
            for (int u = 0; u < C::T * HDP / 256; ++u) {
                const int i = 64 * u + lane;
                const float4 t4 =
                    *reinterpret_cast<const float4 *>(Vs + i / (HDP / 4) * C::STRIDE + i % (HDP / 4) * 4);
                worst = fmaf(0.0f, t4.x, fmaf(0.0f, t4.y, fmaf(0.0f, t4.z, fmaf(0.0f, t4.w, worst))));
            }
            plain = __all(worst == 0.0f);
        }
        if (plain) {
            column_product<HDP>(Vs, sc, jq, g, acc);
        } else {
#pragma unroll
            for (int b = 0; b < C::KB; ++b)
                for (int key = 0; key < 16; ++key) {
                    const float p0 = __shfl(sc[b][0], key / 4 * 16 + jq, 64), p1 = __shfl(sc[b][1], key / 4 * 16 + jq, 64);
                    const float p2 = __shfl(sc[b][2], key / 4 * 16 + jq, 64), p3 = __shfl(sc[b][3], key / 4 * 16 + jq, 64);
                    const float p = (key & 2) ? ((key & 1) ? p3 : p2) : ((key & 1) ? p1 : p0);
                    if (t0 + 16 * b + key > qi) continue;
#pragma unroll
                    for (int d = 0; d < C::DB; ++d)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            acc[d][r] = fmaf(p, Vs[(16 * b + key) * C::STRIDE + 16 * d + 4 * g + r], acc[d][r]);
                }
        }
    }
    l = across_groups(l);
    const float inv = 1.0f / l;
    const bool live = qi < s.sequence;
    const size_t row = base + size_t(live ? qi : 0) * s.W;
    float4 yv[C::DB], vv[C::DB];
    float dot = 0.0f, vsq = 0.0f;
#pragma unroll
    for (int d = 0; d < C::DB; ++d) {
        yv[d] = make_float4(acc[d][0] * inv, acc[d][1] * inv, acc[d][2] * inv, acc[d][3] * inv);
        if (live) store4(y + row, 16 * d + 4 * g, s.hd, yv[d]);
        vv[d] = row4(v + row, 16 * d + 4 * g, s.hd);
        dot += yv[d].x * vv[d].x + yv[d].y * vv[d].y + yv[d].z * vv[d].z + yv[d].w * vv[d].w;
        vsq += vv[d].x * vv[d].x + vv[d].y * vv[d].y + vv[d].z * vv[d].z + vv[d].w * vv[d].w;
    }
    // z = y - (y . u) u, u = v / max(|v|, 1e-12)
    const float iv = rsqrtf(fmaxf(across_groups(vsq), kXsaFloor));
    const float c = s.xsa ? across_groups(dot) * iv * iv : 0.0f;
    if (!live) return;
#pragma unroll
    for (int d = 0; d < C::DB; ++d) {
        float4 o = yv[d];
        if (s.xsa) {
            o.x -= c * vv[d].x;
            o.y -= c * vv[d].y;
            o.z -= c * vv[d].z;
            o.w -= c * vv[d].w;
        }
        store4(z + row, 16 * d + 4 * g, s.hd, o);
    }
    if (g == 0) lse[(first + qi) * s.H + h] = m + log2f(l);
}

// From dy = d loss / d y, D = dy . y per row and the forward's lse:
//   blockIdx.y = 0: dq_i = scale sum_j P_ij (dy_i . v_j - D_i) k_j
//   blockIdx.y = 1: dk_j = scale sum_i P_ij (dy_i . v_j - D_i) q_i,  dv_j += sum_i P_ij dy_i
// (the same fixed order of sums in every run).  A masked pair has weight 0 and the
// products still read its rows.  The forward keeps a later row that is not finite
// from the losses of earlier ones; here it needs no such care: with or without a
// target, the final norm's backward of that row multiplies by values that are not
// finite, and every weight's gradient adds all rows.
template <int HDP>
__global__ void __launch_bounds__(64 * kWaves)
matrix_backward_kernel(AttnShape s, const float *__restrict__ q, const float *__restrict__ k,
                       const float *__restrict__ v, const float *__restrict__ lse, const float *__restrict__ dy,
                       const float *__restrict__ dsum, float *__restrict__ dq, float *__restrict__ dk, float *dv) {
    using C = Tiling<HDP>;
    __shared__ __align__(16) float Xs[C::T * C::STRIDE], Ys[C::T * C::STRIDE], Ls[C::T], Ds[C::T];
    const bool keys = blockIdx.y == 1;
    int pair, tile;
    if (!place(s, !keys, pair, tile)) return;
    const int h = pair % s.H, lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
    const int jq = lane & 15, g = lane >> 4;
    const size_t first = size_t(pair / s.H) * s.sequence, base = first * s.W + h * s.hd;
    const int mine = tile * kOwn + wave * 16, own = mine + jq;
    const bool live = own < s.sequence;
    // Own rows a (scaled) and b, tile rows X and Y: q and dy against k and v.
    float a[C::KS], b[C::KS];
    own_rows<HDP>((keys ? k : q) + base, own, s, g, s.scale_log2, a);
    own_rows<HDP>((keys ? v : dy) + base, own, s, g, 1.0f, b);
    const float *X = (keys ? q : k) + base, *Y = (keys ? dy : v) + base;
    const size_t at = (first + (live ? own : 0)) * s.H + h;
    const float L = keys ? 0.0f : lse[at], D = keys ? 0.0f : dsum[at];
    v4f ax[C::DB], ay[C::DB];
#pragma unroll
    for (int d = 0; d < C::DB; ++d) ax[d] = ay[d] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const int end = (min(tile * kOwn + kOwn, s.sequence) - 1) / C::T + 1;
    const int from = keys ? tile * kOwn / C::T : 0, to = keys ? (s.sequence - 1) / C::T + 1 : end;
    Piece<HDP> px, py;
    float pl = 0.0f, pd = 0.0f;
    auto load = [&](int t0) {
        px.load(X, t0, s);
        py.load(Y, t0, s);
        if (keys && int(threadIdx.x) < C::T) {
            // A row past the sequence gets probability 0.
            const int i = t0 + int(threadIdx.x);
            pl = i < s.sequence ? lse[(first + i) * s.H + h] : INFINITY;
            pd = i < s.sequence ? dsum[(first + i) * s.H + h] : 0.0f;
        }
    };
    load(from * C::T);
    for (int t = from; t < to; ++t) {
        const int t0 = t * C::T;
        __syncthreads();  // the previous tile's readers are done
        px.store(Xs);
        py.store(Ys);
        if (keys && int(threadIdx.x) < C::T) {
            Ls[threadIdx.x] = pl;
            Ds[threadIdx.x] = pd;
        }
        __syncthreads();
        if (t + 1 < to) load(t0 + C::T);
        // Nothing to add where every query of the pair precedes every key.
        if (keys ? t0 + C::T - 1 < mine : t0 > mine + 15) continue;
        v4f p[C::KB], ds[C::KB];
#pragma unroll
        for (int i = 0; i < C::KB; ++i) p[i] = ds[i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        row_product<HDP>(Xs, a, jq, g, p);
        row_product<HDP>(Ys, b, jq, g, ds);
        const bool diag = keys ? t0 < mine + 15 : t0 + C::T - 1 > mine;
#pragma unroll
        for (int i = 0; i < C::KB; ++i) {
            float4 lr = make_float4(L, L, L, L), dr = make_float4(D, D, D, D);
            if (keys) {
                lr = *reinterpret_cast<const float4 *>(Ls + 16 * i + 4 * g);
                dr = *reinterpret_cast<const float4 *>(Ds + 16 * i + 4 * g);
            }
            const float ll[4] = {lr.x, lr.y, lr.z, lr.w}, dd[4] = {dr.x, dr.y, dr.z, dr.w};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int other = t0 + 16 * i + 4 * g + r;
                const bool masked = diag && (keys ? other < own : other > own);
                const float e = masked ? 0.0f : __builtin_amdgcn_exp2f(p[i][r] - ll[r]);
                ds[i][r] = masked ? 0.0f : e * (ds[i][r] - dd[r]);
                p[i][r] = e;
            }
        }
        column_product<HDP>(Xs, ds, jq, g, ax);
        if (keys) column_product<HDP>(Ys, p, jq, g, ay);
    }
    if (!live) return;
    const size_t row = base + size_t(own) * s.W;
#pragma unroll
    for (int d = 0; d < C::DB; ++d) {
        const int dim = 16 * d + 4 * g;
        store4((keys ? dk : dq) + row, dim, s.hd,
               make_float4(ax[d][0] * s.scale, ax[d][1] * s.scale, ax[d][2] * s.scale, ax[d][3] * s.scale));
        if (keys) {
            const float4 o = row4(dv + row, dim, s.hd);
            store4(dv + row, dim, s.hd,
                   make_float4(o.x + ay[d][0], o.y + ay[d][1], o.z + ay[d][2], o.w + ay[d][3]));
        }
    }
}

AttnShape attn_shape(int rows, int sequence, int W, int H, bool xsa) {
    const double scale = 1.0 / std::sqrt(double(W / H));
    return {sequence, W, H, W / H, (sequence + kOwn - 1) / kOwn, rows / sequence * H, int(xsa), float(scale),
            float(1.4426950408889634 * scale)};
}

unsigned attn_grid(const AttnShape &s) { return 8u * unsigned((s.pairs + 7) / 8) * unsigned(s.tiles); }

template <class F>
void by_padded_head(int hd, F &&f) {
    if (hd <= 16)
        f(std::integral_constant<int, 16>{});
    else if (hd <= 32)
        f(std::integral_constant<int, 32>{});
    else if (hd <= 64)
        f(std::integral_constant<int, 64>{});
    else
        f(std::integral_constant<int, 128>{});
}

}  // namespace

void matrix_attention_forward(const float *q, const float *k, const float *v, float *y, float *z, float *lse, int rows,
                              int sequence, int W, int H, bool xsa, hipStream_t stream) {
    const AttnShape s = attn_shape(rows, sequence, W, H, xsa);
    by_padded_head(s.hd, [&](auto hd) {
        hipLaunchKernelGGL(matrix_forward_kernel<decltype(hd)::value>, dim3(attn_grid(s)), dim3(64 * kWaves), 0,
                           stream, s, q, k, v, y, z, lse);
    });
}

void matrix_attention_backward(const float *q, const float *k, const float *v, const float *lse, const float *dy,
                               const float *dsum, float *dq, float *dk, float *dv, int rows, int sequence, int W,
                               int H, hipStream_t stream) {
    const AttnShape s = attn_shape(rows, sequence, W, H, false);
    by_padded_head(s.hd, [&](auto hd) {
        hipLaunchKernelGGL(matrix_backward_kernel<decltype(hd)::value>, dim3(attn_grid(s), 2), dim3(64 * kWaves), 0,
                           stream, s, q, k, v, lse, dy, dsum, dq, dk, dv);
    });
}

}  // namespace meshgpt::kern::train
