// Prefill blocks over many rows: the post-attention half of block l-1
// (reference.rs:194-216: XSA when the attention kernel left it, projection
// mesh and residual, RMSNorm, FFN mesh and residual) fused with the
// pre-attention half of block l (reference.rs:164-193: RMSNorm, Q/K/V meshes,
// QK-Norm, RoPE, K/V cache append), for a tile of R rows per workgroup.
//
// A mesh layer (reference.rs:422-453) is a two-term update of every channel
// from itself and one partner channel, so a tile is kept as R rows x W
// channels where each thread owns CPT channels of RG rows in registers, and
// only the partner values travel: each layer writes the thread's values to
// LDS, one barrier, and reads the partner channel's rows back.  LDS holds the
// tile channel-major (the R rows of a channel contiguous, in 16-byte chunks
// rotated by channel so that neighbouring lanes' 16-byte accesses fall in
// different banks), double-buffered so one barrier per layer suffices.  Each
// thread loads one [self, partner] weight pair per owned channel per layer,
// used for all of its rows.  Row reductions (RMSNorm) go through a small LDS
// scratch; head reductions (QK-Norm, XSA) and the RoPE pair exchange stay
// inside a wave (a head is hd <= 64 consecutive channels = consecutive lanes).
//
// What bounds it is instruction issue: five VALU instructions a value and layer
// (product, multiply-add, exponential, multiply-add, maximum; values are carried
// times log2(e), or it is six) and an LDS write and read of the value, behind a
// barrier each layer that only other workgroups' waves on the SIMD can fill.
// Widths 512 and 1024 keep to 128 registers for four waves a SIMD; 128 and 256,
// with 16 rows a thread, would spill and keep three.  A prefill of 256 x 128 rows
// (W1024, 12 blocks, 13 launches of this kernel, 527 us each before and 446 now): 8.84 ms,
// 7.94 with the scaled values alone, 7.68 with four waves as well.  Values above
// 2.36e38 are infinite in these units, so models whose weights could reach them
// (Shape::wide) run in their own: 7.8 ms, 456 us a launch.
// Not kept: strides of 256 and 512 from the thread's own registers (7.73 ms), weights
// loaded two layers ahead (7.74).
#include <hip/hip_runtime.h>

#include "dpp.hpp"
#include "kernels.hpp"

namespace meshgpt::kern {
namespace {

constexpr float kEps = 1e-5f;  // src/gpt/mod.rs:38
// (f64(1e-12f))^2 rounded to f32: the XSA norm floor of reference.rs:591.
constexpr float kXsaNormFloor = float(double(1e-12f) * double(1e-12f));

constexpr float kLog2e = 1.4426950408889634f, kLn2 = 0.6931471805599453f;

// What a value is multiplied by on its way into the meshes and out of them:
// SCALED ones are carried times log2(e), which the ELU's exponential would
// otherwise multiply in (Shape::wide: their own units).
template <bool SCALED>
struct Units {
    static constexpr float in = SCALED ? kLog2e : 1.0f, out = SCALED ? kLn2 : 1.0f;
};

// The ELU in these units, of t = z or z log2(e): max(z, clamp(exp(z), 0, 1) - 1)
// with the NaN-propagating maximum, which keeps a NaN NaN (kernels.hip's elu).
template <bool SCALED>
__device__ __forceinline__ float elu_units(float t) {
    const float e = __builtin_amdgcn_fmed3f(__builtin_amdgcn_exp2f(SCALED ? t : t * kLog2e), 0.0f, 1.0f);
    return __builtin_elementwise_maximum(t, SCALED ? __builtin_fmaf(e, kLog2e, -kLog2e) : e - 1.0f);
}

template <int W>
struct RowsCfg {
    static constexpr int THREADS = 256;
    static constexpr int T = W < 256 ? W : 256;   // threads per row group (one per channel slot)
    static constexpr int G = THREADS / T;         // row groups
    static constexpr int CPT = W / T;             // channels per thread: slot + T*k
    static constexpr int R = 4096 / W;            // rows per workgroup
    static constexpr int RG = R / G;              // rows per thread
    static constexpr int NCH = R / 4;             // 16-byte chunks of a channel
    static constexpr int ROT = R >= 64 ? 1 : 64 / R;  // channels per chunk rotation step
    static constexpr int TILE = W * R;            // floats of one LDS buffer
    static constexpr int WAVES = CPT > 1 ? 4 : 3;  // of a SIMD
    static constexpr int WAVES_G = T / 64 > 0 ? T / 64 : 1;  // waves per row group
    static_assert(RG % 4 == 0 && W % 64 == 0, "tile geometry");
};

// LDS offset of the 16-byte chunk holding rows [4 ch, 4 ch + 4) of channel c.
template <int W>
__device__ __forceinline__ int chunk_at(int c, int ch) {
    using C = RowsCfg<W>;
    return c * C::R + 4 * ((ch + c / C::ROT) & (C::NCH - 1));
}

template <int W, bool SCALED>
struct Tile {
    using C = RowsCfg<W>;
    static constexpr int CPT = C::CPT, RG = C::RG;
    float *lds;   // 2 * TILE floats
    float *red;   // row-reduction scratch: [4 waves][RG]
    int parity;
    int slot, rg, lane, wave;  // channel slot, row group
    __device__ int chan(int k) const { return slot + C::T * k; }
    __device__ int row(int i) const { return rg * RG + i; }

    __device__ void put(const float (&v)[CPT][RG]) {
        float *B = lds + parity * C::TILE;
#pragma unroll
        for (int k = 0; k < CPT; ++k)
#pragma unroll
            for (int j = 0; j < RG / 4; ++j)
                *reinterpret_cast<float4 *>(B + chunk_at<W>(chan(k), rg * (RG / 4) + j)) =
                    make_float4(v[k][4 * j], v[k][4 * j + 1], v[k][4 * j + 2], v[k][4 * j + 3]);
    }
    // The values of channel (own channel + st) mod W from the buffer last put.
    __device__ void partner(int st, float (&p)[CPT][RG]) const {
        const float *B = lds + parity * C::TILE;
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
            const int c = (chan(k) + st) & (W - 1);
#pragma unroll
            for (int j = 0; j < RG / 4; ++j) {
                const float4 t = *reinterpret_cast<const float4 *>(B + chunk_at<W>(c, rg * (RG / 4) + j));
                p[k][4 * j] = t.x;
                p[k][4 * j + 1] = t.y;
                p[k][4 * j + 2] = t.z;
                p[k][4 * j + 3] = t.w;
            }
        }
    }
    __device__ void flip() { parity ^= 1; }

    // One layer on v in place: v[c] w0 + p[c] w1, and the ELU unless LAST.
    template <bool LAST>
    __device__ __forceinline__ void update(float (&v)[CPT][RG], const float (&p)[CPT][RG], const float2 (&w)[CPT]) {
#pragma unroll
        for (int k = 0; k < CPT; ++k)
#pragma unroll
            for (int i = 0; i < RG; ++i) {
                const float t = v[k][i] * w[k].x + p[k][i] * w[k].y;
                v[k][i] = LAST ? t : elu_units<SCALED>(t);
            }
    }
    template <bool LAST>
    __device__ __forceinline__ void layer(float (&v)[CPT][RG], const float2 (&w)[CPT], int st) {
        float p[CPT][RG];
        put(v);
        __syncthreads();
        partner(st, p);
        update<LAST>(v, p, w);
        flip();
    }

    // A mesh stack on v in place: layer l maps v[c] to v[c] w0 + v[c + st] w1
    // with ELU on every layer but the last (reference.rs:422-453).
    // Butterfly strides double from 1 and wrap at W (W is a power of two).
    // Values are in the meshes' units.
    __device__ void mesh(float (&v)[CPT][RG], const float2 *__restrict__ w, int depth, const Shape &s) {
        float2 wc[CPT];
#pragma unroll
        for (int k = 0; k < CPT; ++k) wc[k] = w[chan(k)];
        int st = 1;
        for (int l = 0; l + 1 < depth; ++l) {
            float2 wn[CPT];
#pragma unroll
            for (int k = 0; k < CPT; ++k) wn[k] = w[size_t(l + 1) * W + chan(k)];
            layer<false>(v, wc, st);
#pragma unroll
            for (int k = 0; k < CPT; ++k) wc[k] = wn[k];
            st = s.butterfly ? (2 * st == W ? 1 : 2 * st) : 1;
        }
        layer<true>(v, wc, st);
    }

    // inv[i] = 1 / sqrt(mean over the row's W channels of v^2 + eps) for the
    // thread's rows (reference.rs:392-409 with one segment).
    __device__ void row_inv_rms(const float (&v)[CPT][RG], float (&inv)[RG]) {
        float part[RG];
#pragma unroll
        for (int i = 0; i < RG; ++i) {
            float a = 0.0f;
#pragma unroll
            for (int k = 0; k < CPT; ++k) a = fmaf(v[k][i], v[k][i], a);
            part[i] = a;
        }
#pragma unroll
        for (int i = 0; i < RG; ++i) part[i] = wave_sum(part[i]);
        __syncthreads();  // the scratch's previous readers are done
        if (lane == 0) {
#pragma unroll
            for (int i = 0; i < RG; ++i) red[wave * RG + i] = part[i];
        }
        __syncthreads();
        const int w0 = rg * C::WAVES_G;
#pragma unroll
        for (int i = 0; i < RG; ++i) {
            float a = 0.0f;
            for (int q = 0; q < C::WAVES_G; ++q) a += red[(w0 + q) * RG + i];
            inv[i] = rsqrtf(a * (1.0f / float(W)) + kEps);
        }
    }
};

// Sum over the hd lanes of a head (hd a power of two <= 64, heads aligned to
// hd lanes): DPP moves when the head width HD is a compile-time 32 or 64.
template <int HD>
__device__ __forceinline__ float head_sum(float v, int hd) {
    if constexpr (HD > 0) return group_sum<HD>(v);
    for (int m = hd >> 1; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}

// HD: the head width when it is 32 or 64 (DPP head sums), else 0.  Rows are
// whole prefill sequences (Rows.len is null: a row's position is its index
// within its sequence).
template <int W, int HD, bool SCALED>
__global__ void __launch_bounds__(256, RowsCfg<W>::WAVES) rows_block_kernel(BlockArgs a) {
    using C = RowsCfg<W>;
    using U = Units<SCALED>;
    constexpr int CPT = C::CPT, RG = C::RG;
    __shared__ __align__(16) float lds[2 * C::TILE];
    __shared__ float red[4 * RG];
    const Shape &s = a.s;
    Tile<W, SCALED> t;
    t.lds = lds;
    t.red = red;
    t.parity = 0;
    t.slot = int(threadIdx.x) % C::T;
    t.rg = int(threadIdx.x) / C::T;
    t.lane = int(threadIdx.x) & 63;
    t.wave = int(threadIdx.x) >> 6;
    const bool post = a.wproj != nullptr, pre = a.wq != nullptr;
    const int r0 = int(blockIdx.x) * C::R;

    // Rows of this thread: rbase + i; rows past the batch repeat its last row
    // and write nothing.  Only the sequences are kept; the row indices and
    // positions are formed where they are used.
    const int rbase = r0 + t.rg * RG, rps = a.ro.rows_per_seq;
    auto rowof = [&](int i) { return min(rbase + i, a.ro.rows - 1); };
    auto live = [&](int i) { return rbase + i < a.ro.rows; };
    int seq[RG];
#pragma unroll
    for (int i = 0; i < RG; ++i) seq[i] = rowof(i) / rps;
    auto grow = [&](int i) { return size_t(rowof(i)); };
    auto posof = [&](int i) { return rowof(i) - seq[i] * rps; };

    float x[CPT][RG];
    if (a.embed) {
#pragma unroll
        for (int i = 0; i < RG; ++i) {
            const uint32_t tok = a.ro.tokens[size_t(seq[i]) * a.ro.tok_stride + a.ro.tok_offset + posof(i)];
#pragma unroll
            for (int k = 0; k < CPT; ++k) x[k][i] = a.E[size_t(tok) * W + t.chan(k)];
        }
    } else {
#pragma unroll
        for (int i = 0; i < RG; ++i)
#pragma unroll
            for (int k = 0; k < CPT; ++k) x[k][i] = a.x[grow(i) * W + t.chan(k)];
    }

    if (post) {
        float y[CPT][RG];
#pragma unroll
        for (int i = 0; i < RG; ++i)
#pragma unroll
            for (int k = 0; k < CPT; ++k) y[k][i] = a.ybuf[grow(i) * W + t.chan(k)];
        if (a.xsa_post) {
            // XSA (reference.rs:577-603): z = y - (y.u)u, u = v / max(|v|, eps).
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                const int c = t.chan(k), h = c / s.hd, d = c - h * s.hd;
#pragma unroll
                for (int i = 0; i < RG; ++i) {
                    const float v =
                        a.kv_post.v[(size_t(seq[i] * s.H + h) * a.kv_post.cap + posof(i)) * s.hdp + d];
                    const float vv = head_sum<HD>(v * v, s.hd), yv = head_sum<HD>(y[k][i] * v, s.hd);
                    const float iv = rsqrtf(fmaxf(vv, kXsaNormFloor));
                    y[k][i] = y[k][i] - (yv * iv) * (v * iv);
                }
            }
        }
        if constexpr (SCALED) {
#pragma unroll
            for (int k = 0; k < CPT; ++k)
#pragma unroll
                for (int i = 0; i < RG; ++i) y[k][i] *= U::in;
        }
        t.mesh(y, reinterpret_cast<const float2 *>(a.wproj), s.A, s);
#pragma unroll
        for (int k = 0; k < CPT; ++k)
#pragma unroll
            for (int i = 0; i < RG; ++i) x[k][i] = __builtin_fmaf(y[k][i], U::out, x[k][i]);
        float inv[RG];
        t.row_inv_rms(x, inv);
        float n[CPT][RG];
#pragma unroll
        for (int k = 0; k < CPT; ++k)
#pragma unroll
            for (int i = 0; i < RG; ++i) n[k][i] = x[k][i] * (inv[i] * U::in);
        t.mesh(n, reinterpret_cast<const float2 *>(a.wffn), s.F, s);
#pragma unroll
        for (int k = 0; k < CPT; ++k)
#pragma unroll
            for (int i = 0; i < RG; ++i) x[k][i] = __builtin_fmaf(n[k][i], U::out, x[k][i]);
    }
    if (post || a.embed) {
#pragma unroll
        for (int i = 0; i < RG; ++i)
            if (live(i)) {
#pragma unroll
                for (int k = 0; k < CPT; ++k) a.x[grow(i) * W + t.chan(k)] = x[k][i];
            }
    }
    if (!a.xn && !pre) return;

    // The next RMSNorm: the final one for the head, or the block's pre-norm,
    // whose rows enter the meshes in their units.
    float n[CPT][RG];
    {
        float inv[RG];
        t.row_inv_rms(x, inv);
        if (a.xn) {
#pragma unroll
            for (int i = 0; i < RG; ++i)
                if (live(i)) {
#pragma unroll
                    for (int k = 0; k < CPT; ++k) a.xn[grow(i) * W + t.chan(k)] = x[k][i] * inv[i];
                }
        }
        if (!pre) return;
#pragma unroll
        for (int k = 0; k < CPT; ++k)
#pragma unroll
            for (int i = 0; i < RG; ++i) n[k][i] = x[k][i] * (inv[i] * U::in);
    }

    // Q, K and V meshes, one after another, each from the normalised rows.
    const bool no_q = a.q_last && (r0 + C::R) / rps == r0 / rps && r0 + C::R < a.ro.rows;  // no sequence ends here
    for (int m = no_q ? 1 : 0; m < 3; ++m) {
        const float *wm = m == 0 ? a.wq : (m == 1 ? a.wk : a.wv);
        float v[CPT][RG];
#pragma unroll
        for (int k = 0; k < CPT; ++k)
#pragma unroll
            for (int i = 0; i < RG; ++i) v[k][i] = n[k][i];
        t.mesh(v, reinterpret_cast<const float2 *>(wm), s.A, s);
        // Addresses and RoPE factors are formed here for each mesh: hoisted out of
        // the loop they would hold up to 60 registers through every layer.  (With
        // 16 rows a thread, widths 128 and 256, forming them spills.)
        int here = 0;
        if constexpr (CPT > 1) asm volatile("" : "+v"(here));
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
            const int c = t.chan(k) + here, h = c / s.hd, d = c - h * s.hd;
            if (m < 2) {
                // QK-Norm per head, then RoPE at the row's position, each when
                // its switch is on (reference.rs:174-193); the pair partner
                // d ^ half is the lane half a head away.
#pragma unroll
                for (int i = 0; i < RG; ++i) {
                    float q = v[k][i];
                    q *= s.qk_norm ? rsqrtf(head_sum<HD>(q * q, s.hd) * (1.0f / float(s.hd)) + kEps * U::in * U::in)
                                   : U::out;
                    if (s.rope) {
                        const float p = __shfl_xor(q, s.half, 64);
                        const float2 cs = a.rope[size_t(posof(i)) * s.half + (d < s.half ? d : d - s.half)];
                        q = q * cs.x + (d < s.half ? -p : p) * cs.y;
                    }
                    v[k][i] = q;
                }
            } else {
#pragma unroll
                for (int i = 0; i < RG; ++i) v[k][i] *= U::out;
            }
#pragma unroll
            for (int i = 0; i < RG; ++i) {
                if (!live(i)) continue;
                if (m == 0) {
                    a.q[grow(i) * W + c] = v[k][i];
                } else {
                    float *dst = m == 1 ? a.kv_pre.k : a.kv_pre.v;
                    dst[(size_t(seq[i] * s.H + h) * a.kv_pre.cap + posof(i)) * s.hdp + d] = v[k][i];
                }
            }
        }
    }
}

// The last rows of `nseq` sequences of n rows, for attention over whole
// sequences and blocks over single rows: q and x gathered, len filled with n.
__global__ void __launch_bounds__(256)
last_rows_kernel(const float *__restrict__ q, const float *__restrict__ x, int n, int W, float *__restrict__ q_out,
                 float *__restrict__ x_out, int *__restrict__ len) {
    const size_t from = (size_t(blockIdx.x) * n + n - 1) * W, to = size_t(blockIdx.x) * W;
    for (int c = 4 * int(threadIdx.x); c < W; c += 1024) {
        *reinterpret_cast<float4 *>(q_out + to + c) = *reinterpret_cast<const float4 *>(q + from + c);
        *reinterpret_cast<float4 *>(x_out + to + c) = *reinterpret_cast<const float4 *>(x + from + c);
    }
    if (threadIdx.x == 0) len[blockIdx.x] = n;
}

// The split states (acc[hdp], m, l; log2 domain) of one (sequence, head) per
// wave merged into its attention row, then XSA against the value row at n - 1
// (reference.rs:577-603).
__global__ void __launch_bounds__(256)
last_merge_kernel(Shape s, const float *__restrict__ part, int nsplit, KvView kv, int n, int pairs, int xsa,
                  float *__restrict__ y) {
    const int pair = (int(blockIdx.x) * 256 + int(threadIdx.x)) >> 6, lane = int(threadIdx.x) & 63;
    if (pair >= pairs) return;
    const float *p = part + size_t(pair) * nsplit * (s.hdp + 2);
    float top = -INFINITY;
    for (int i = 0; i < nsplit; ++i) top = fmaxf(top, p[size_t(i) * (s.hdp + 2) + s.hdp]);
    float sum = 0.0f, acc = 0.0f;
    for (int i = 0; i < nsplit; ++i) {
        const float *state = p + size_t(i) * (s.hdp + 2);
        const float scale = __builtin_amdgcn_exp2f(state[s.hdp] - top);
        sum = fmaf(state[s.hdp + 1], scale, sum);
        if (lane < s.hd) acc = fmaf(state[lane], scale, acc);
    }
    acc /= sum;
    const float v = lane < s.hd ? kv.v[(size_t(pair) * kv.cap + n - 1) * s.hdp + lane] : 0.0f;
    const float vv = wave_sum(v * v), yv = wave_sum(acc * v), iv = rsqrtf(fmaxf(vv, kXsaNormFloor));
    if (lane < s.hd) y[size_t(pair) * s.hd + lane] = xsa ? acc - (yv * iv) * (v * iv) : acc;
}

}  // namespace

bool rows_block_supported(const Shape &s) {
    return (s.W == 128 || s.W == 256 || s.W == 512 || s.W == 1024) && s.hdshift >= 1 && s.hd <= 64 &&
           64 % s.hd == 0;
}

template <int W, bool SCALED>
void launch_rows_block(const BlockArgs &a, hipStream_t stream) {
    const dim3 grid((a.ro.rows + RowsCfg<W>::R - 1) / RowsCfg<W>::R);
    if (a.s.hd == 32)
        hipLaunchKernelGGL((rows_block_kernel<W, 32, SCALED>), grid, dim3(256), 0, stream, a);
    else if (a.s.hd == 64)
        hipLaunchKernelGGL((rows_block_kernel<W, 64, SCALED>), grid, dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL((rows_block_kernel<W, 0, SCALED>), grid, dim3(256), 0, stream, a);
}

template <bool SCALED>
void rows_block_units(const BlockArgs &a, hipStream_t stream) {
    switch (a.s.W) {
    case 128: launch_rows_block<128, SCALED>(a, stream); break;
    case 256: launch_rows_block<256, SCALED>(a, stream); break;
    case 512: launch_rows_block<512, SCALED>(a, stream); break;
    default: launch_rows_block<1024, SCALED>(a, stream); break;
    }
}

void rows_block(const BlockArgs &a, hipStream_t stream) {
    a.s.wide ? rows_block_units<false>(a, stream) : rows_block_units<true>(a, stream);
}

void last_rows(const float *q, const float *x, int nseq, int n, int W, float *q_out, float *x_out, int *len,
               hipStream_t stream) {
    hipLaunchKernelGGL(last_rows_kernel, dim3(nseq), dim3(256), 0, stream, q, x, n, W, q_out, x_out, len);
}

void last_merge(const Shape &s, const float *part, int nsplit, KvView kv, int nseq, int n, int xsa, float *y,
                hipStream_t stream) {
    const int pairs = nseq * s.H;
    hipLaunchKernelGGL(last_merge_kernel, dim3((pairs + 3) / 4), dim3(256), 0, stream, s, part, nsplit, kv, n, pairs,
                       xsa, y);
}

}  // namespace meshgpt::kern
