// Training's row-local operators between two attentions in one launch each way,
// for widths up to 128 and stacks of few layers.
//
// What bounds a training step of a small model is its launches (a kernel of a
// captured step takes some 4.5 us however little it does, and there were 35) and
// each one's wait for its operands.  Between two attentions every operator works
// on single rows, so one wave takes a row through all of them, in registers, with
// every operand asked for before the first product:
//   forward   projection mesh, residual, RMSNorm, FFN mesh, residual (block b),
//             RMSNorm, Q, K and V meshes, QK-Norm, RoPE (block b + 1);
//   backward  QK-Norm and RoPE, Q, K and V meshes, RMSNorm (block b + 1), FFN
//             mesh, RMSNorm, projection mesh (block b).
// The first and last launches of a pass do what there is of this, the token
// gather or the final norm beside it.  Each operator is the arithmetic of its own
// kernel in train.hip on the same operands in the same order, and every stored
// activation and partial sum is the one that kernel stores, so the results are
// the same bits.  The backward keeps the sums of five stacks' weight gradients
// in registers, which limits its depths (kChainSums).
//
// One AdamW update, separate launches against these: 256 rows of width 32 (the
// demo corpus, attention by waves) 212 us and 198, 2048 rows of width 128 (512
// equations) 284 and 251.  A middle launch takes 10 us forward and 19 us backward
// at width 32, 19 and 31 at width 128.  Without the loads at the front (each
// stack's behind the one before) the updates took 219 and 275.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mesh_wave.hpp"

namespace meshgpt::kern::train {
namespace {

// Registers for weight-gradient sums: two a layer and channel of a lane.
constexpr int kChainSums = 96;

// Loads above stay above: a chain's operands are all on their way before its
// first product, so that it waits for memory once and not once a stack.
__device__ __forceinline__ void loads_first() { asm volatile("" ::: "memory"); }

// A stack's weights of this lane's channels.
template <int CPL, int D>
struct StackWeights {
    float2 wt[D][CPL];
    __device__ __forceinline__ void load(const Mesh &m, const float *__restrict__ w, int lane) {
#pragma unroll
        for (int l = 0; l < D; ++l)
#pragma unroll
            for (int j = 0; j < CPL; ++j)
                wt[l][j] = l < m.depth && lane + 64 * j < m.W
                               ? reinterpret_cast<const float2 *>(w + size_t(l) * 2 * m.W)[lane + 64 * j]
                               : make_float2(0.0f, 0.0f);
    }
    // The wave's row through the stack: every layer's output stored (and the
    // last left in x).
    __device__ __forceinline__ void forward(float (&x)[CPL], const Mesh &m, float *__restrict__ stack, int r, int rows,
                                            int lane) const {
        const int W = m.W;
#pragma unroll
        for (int l = 0; l < D; ++l) {
            if (l >= m.depth) continue;
            float p[CPL];
            channel_shift(x, stride_of(m, l), W, lane, p);
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int c = lane + 64 * j;
                float z = x[j] * wt[l][j].x + p[j] * wt[l][j].y;
                if (elu_layer(m, l)) z = elu(z);
                x[j] = z;
                if (c < W) stack[(size_t(l) * rows + r) * W + c] = z;
            }
        }
    }
};

template <int CPL>
__device__ __forceinline__ void row_load(const float *__restrict__ from, int r, int W, int lane, float (&x)[CPL]) {
#pragma unroll
    for (int j = 0; j < CPL; ++j) x[j] = lane + 64 * j < W ? from[size_t(r) * W + lane + 64 * j] : 0.0f;
}

template <int CPL>
__device__ __forceinline__ void row_store(float *__restrict__ to, int r, int W, int lane, const float (&x)[CPL]) {
#pragma unroll
    for (int j = 0; j < CPL; ++j)
        if (lane + 64 * j < W) to[size_t(r) * W + lane + 64 * j] = x[j];
}

// n = RMSNorm(x), stored with its factor (rmsnorm_forward_kernel).
template <int CPL>
__device__ __forceinline__ void row_norm(const float (&x)[CPL], float (&n)[CPL], float *__restrict__ to,
                                         float *__restrict__ inv, int r, int W, int lane) {
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < CPL; ++j) acc = fmaf(x[j], x[j], acc);
    const float iv = rsqrtf(wave_sum(acc) * (1.0f / float(W)) + kRmsEps);
#pragma unroll
    for (int j = 0; j < CPL; ++j) n[j] = x[j] * iv;
    row_store(to, r, W, lane, n);
    if (lane == 0) inv[r] = iv;
}

// The sum over each head of hd lanes (a power of two up to 64).
__device__ __forceinline__ float head_sum(float v, int hd) {
    for (int off = hd / 2; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// The same with the neighbouring lanes first, as qk_backward_kernel adds.
__device__ __forceinline__ float head_sum_up(float v, int hd) {
    switch (hd) {
        case 2: return group_sum<2>(v);
        case 4: return group_sum<4>(v);
        case 8: return group_sum<8>(v);
        case 16: return group_sum<16>(v);
        case 32: return group_sum<32>(v);
        default: return group_sum<64>(v);
    }
}

template <int CPL, int DA, int DF>
__global__ void __launch_bounds__(kThreads, 2) forward_chain_kernel(ForwardChain a) {
    const int lane = threadIdx.x & 63, W = a.ma.W, r = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
    if (r >= a.rows) return;
    StackWeights<CPL, DA> wp, wq[3];
    StackWeights<CPL, DF> wf;
    float x[CPL], t[CPL];
    if (a.E) {
        row_load(a.E, int(a.tokens[r]), W, lane, x);
    } else {
        row_load(a.z, r, W, lane, t);
        row_load(a.x_in, r, W, lane, x);
        wp.load(a.ma, a.wproj, lane);
        wf.load(a.mf, a.wffn, lane);
    }
    if (a.wqkv[0]) {
#pragma unroll
        for (int y = 0; y < 3; ++y) wq[y].load(a.ma, a.wqkv[y], lane);
    }
    loads_first();
    if (!a.E) {
        // xm = x_b + proj(z), x_{b+1} = xm + ffn(RMSNorm(xm))
        wp.forward(t, a.ma, a.ps, r, a.rows, lane);
#pragma unroll
        for (int j = 0; j < CPL; ++j) x[j] = x[j] + t[j];
        row_store(a.xm, r, W, lane, x);
        row_norm(x, t, a.n2, a.inv2, r, W, lane);
        wf.forward(t, a.mf, a.fs, r, a.rows, lane);
#pragma unroll
        for (int j = 0; j < CPL; ++j) x[j] = x[j] + t[j];
    }
    row_store(a.x_out, r, W, lane, x);
    float n[CPL];
    row_norm(x, n, a.n, a.inv, r, W, lane);
    if (!a.wqkv[0]) return;
    const int hd = W / a.qk.H, half = hd / 2;
#pragma unroll
    for (int y = 0; y < 3; ++y) {
#pragma unroll
        for (int j = 0; j < CPL; ++j) t[j] = n[j];
        wq[y].forward(t, a.ma, a.qkv[y], r, a.rows, lane);
        if (y == 2) break;
        if (a.qk.norm) {
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int c = lane + 64 * j;
                const float iv = rsqrtf(head_sum(t[j] * t[j], hd) * (1.0f / float(hd)) + kRmsEps);
                t[j] *= iv;
                if (c < W && c % hd == 0) a.qk.inv[y][size_t(r) * a.qk.H + c / hd] = iv;
            }
        }
        if (a.qk.rotate) {
            const float2 *row = a.qk.table + size_t(r % a.qk.sequence) * half;
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const float o = __shfl_xor(t[j], half, 64);
                const int d = (lane + 64 * j) % hd;
                const float2 cs = row[d < half ? d : d - half];
                t[j] = d < half ? t[j] * cs.x - o * cs.y : t[j] * cs.x + o * cs.y;
            }
        }
        row_store(a.qk.out[y], r, W, lane, t);
    }
}

// One row's layer inputs of a stack; layer l's output is layer l + 1's input.
template <int CPL, int D>
struct StackInputs {
    float xin[D][CPL];
    __device__ __forceinline__ void load(const Mesh &m, const float *__restrict__ in, const float *__restrict__ stack,
                                         int r, int rows, int lane) {
#pragma unroll
        for (int l = 0; l < D; ++l)
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int c = lane + 64 * j;
                const float *x = l == 0 ? in + size_t(r) * m.W : stack + (size_t(l - 1) * rows + r) * m.W;
                xin[l][j] = l < m.depth && c < m.W ? x[c] : 0.0f;
            }
    }
};

// A stack's weight-gradient sums over the wave's rows (mesh_backward_wave).
template <int CPL, int D>
struct StackSums {
    float gs[D][CPL], gp[D][CPL];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int l = 0; l < D; ++l)
#pragma unroll
            for (int j = 0; j < CPL; ++j) gs[l][j] = gp[l][j] = 0.0f;
    }
    // g = d loss / d (the stack's output) of the wave's row becomes
    // d loss / d (its input).
    __device__ __forceinline__ void row(float (&g)[CPL], const Mesh &m, const StackInputs<CPL, D> &s,
                                        const StackWeights<CPL, D> &w, int lane) {
        const int W = m.W;
#pragma unroll
        for (int l = D - 1; l >= 0; --l) {
            if (l >= m.depth) continue;
            const int st = stride_of(m, l);
            float xp[CPL], dz[CPL], t[CPL], back[CPL];
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int c = lane + 64 * j;
                // ELU'(z) from its output a, which the next layer read.
                const float act = l + 1 < D && elu_layer(m, l) ? s.xin[(l + 1) % D][j] : 0.0f;
                const float d = act < 0.0f ? g[j] * (act + 1.0f) : g[j];
                dz[j] = c < W ? d : 0.0f;
                t[j] = dz[j] * w.wt[l][j].y;
            }
            channel_shift(s.xin[l], st, W, lane, xp);
            channel_shift(t, W - st, W, lane, back);
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int c = lane + 64 * j;
                gs[l][j] = fmaf(dz[j], s.xin[l][j], gs[l][j]);
                gp[l][j] = fmaf(dz[j], xp[j], gp[l][j]);
                g[j] = c < W ? dz[j] * w.wt[l][j].x + back[j] : 0.0f;
            }
        }
    }
    // The workgroup's waves' sums, added in wave order, into its partial.
    __device__ __forceinline__ void flush(float *sums, float *__restrict__ partials, const Mesh &m, int lane, int wv) {
        const int W = m.W, n = m.depth * W * 2;
        __syncthreads();  // the previous stack's sums have been read
#pragma unroll
        for (int l = 0; l < D; ++l) {
            if (l >= m.depth) continue;
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int c = lane + 64 * j;
                if (c >= W) continue;
                float *o = sums + ((size_t(wv) * m.depth + l) * W + c) * 2;
                o[0] = gs[l][j];
                o[1] = gp[l][j];
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += kThreads) {
            float acc = 0.0f;
            for (int k = 0; k < kThreads / 64; ++k) acc += sums[size_t(k) * n + i];
            partials[size_t(blockIdx.x) * n + i] = acc;
        }
    }
};

// The gradient g of a RMSNorm's output through it: inv g - x inv^3 (g . x) / W.
template <int CPL>
__device__ __forceinline__ void norm_backward(const float (&g)[CPL], const float (&x)[CPL], float iv, int W,
                                              float (&d)[CPL]) {
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < CPL; ++j) acc = fmaf(g[j], x[j], acc);
    const float k = wave_sum(acc) * iv * iv * iv * (1.0f / float(W));
#pragma unroll
    for (int j = 0; j < CPL; ++j) d[j] = iv * g[j] - x[j] * k;
}

template <int CPL, int DA, int DF>
__global__ void __launch_bounds__(kThreads, 1) backward_chain_kernel(BackwardChain a) {
    extern __shared__ float sums[];  // (kThreads / 64) x depth x W x 2
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, W = a.ma.W, rows = a.rows;
    const int wave = blockIdx.x * (kThreads / 64) + wv, waves = gridDim.x * (kThreads / 64);
    const bool below = a.wqkv[0] != nullptr, post = a.wffn != nullptr;
    StackSums<CPL, DA> sq[3], sp;
    StackSums<CPL, DF> sf;
    StackWeights<CPL, DA> wq[3], wp;
    StackWeights<CPL, DF> wf;
#pragma unroll
    for (int y = 0; y < 3; ++y) {
        sq[y].clear();
        if (below) wq[y].load(a.ma, a.wqkv[y], lane);
    }
    sp.clear();
    sf.clear();
    if (post) {
        wf.load(a.mf, a.wffn, lane);
        wp.load(a.ma, a.wproj, lane);
    }
    const int hd = W / a.H, half = hd / 2;
    for (int r = wave; r < rows; r += waves) {
        // Every operand of the row.
        StackInputs<CPL, DA> iq[3], ip;
        StackInputs<CPL, DF> jf;
        float dx[CPL], top[CPL], gq[3][CPL], pre[2][CPL], iv[2][CPL], xb[CPL], xm[CPL], inv_last = 0.0f, inv1 = 0.0f,
            inv2 = 0.0f;
        float2 turn[CPL];
        if (a.dn) {
            row_load(a.dn, r, W, lane, dx);
            row_load(a.x_last, r, W, lane, top);
            inv_last = a.inv_last[r];
        } else {
            row_load(a.dx, r, W, lane, dx);
        }
        if (below) {
#pragma unroll
            for (int y = 0; y < 3; ++y) {
                row_load(a.dqkv[y], r, W, lane, gq[y]);
                iq[y].load(a.ma, a.n1, a.qkv[y], r, rows, lane);
                if (y == 2) break;
                row_load(a.qkv[y] + size_t(a.ma.depth - 1) * rows * W, r, W, lane, pre[y]);
#pragma unroll
                for (int j = 0; j < CPL; ++j) {
                    const int c = lane + 64 * j;
                    iv[y][j] = a.norm && c < W ? a.qk_inv[y][size_t(r) * a.H + c / hd] : 0.0f;
                }
            }
            row_load(a.x_below, r, W, lane, xb);
            inv1 = a.inv1[r];
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int e = (lane + 64 * j) % hd;
                turn[j] = a.rotate ? a.table[size_t(r % a.sequence) * half + (e < half ? e : e - half)]
                                   : make_float2(1.0f, 0.0f);
            }
        }
        if (post) {
            jf.load(a.mf, a.n2, a.fs, r, rows, lane);
            row_load(a.xm, r, W, lane, xm);
            inv2 = a.inv2[r];
            ip.load(a.ma, a.z, a.ps, r, rows, lane);
        }
        loads_first();
        float d[CPL];
        if (a.dn) {
            // The final norm's backward begins the residual's gradient.
            norm_backward(dx, top, inv_last, W, d);
#pragma unroll
            for (int j = 0; j < CPL; ++j) dx[j] = d[j];
        }
        if (below) {
            float sum[CPL];
#pragma unroll
            for (int y = 0; y < 3; ++y) {
                float(&g)[CPL] = gq[y];
                if (y < 2 && a.rotate) {
#pragma unroll
                    for (int j = 0; j < CPL; ++j) {
                        const float o = __shfl_xor(g[j], half, 64);
                        const int e = (lane + 64 * j) % hd;
                        g[j] = e < half ? g[j] * turn[j].x + o * turn[j].y : g[j] * turn[j].x - o * turn[j].y;
                    }
                }
                if (y < 2 && a.norm) {
#pragma unroll
                    for (int j = 0; j < CPL; ++j) {
                        const float f = iv[y % 2][j], x = pre[y % 2][j];
                        const float k = head_sum_up(fmaf(g[j], x, 0.0f), hd) * f * f * f * (1.0f / float(hd));
                        g[j] = f * g[j] - x * k;
                    }
                }
                sq[y].row(g, a.ma, iq[y], wq[y], lane);
#pragma unroll
                for (int j = 0; j < CPL; ++j) sum[j] = y == 0 ? g[j] : sum[j] + g[j];
            }
            norm_backward(sum, xb, inv1, W, d);
#pragma unroll
            for (int j = 0; j < CPL; ++j) dx[j] = dx[j] + d[j];
        }
        if (post) {
            float g[CPL];
#pragma unroll
            for (int j = 0; j < CPL; ++j) g[j] = dx[j];
            sf.row(g, a.mf, jf, wf, lane);
            norm_backward(g, xm, inv2, W, d);
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                dx[j] = dx[j] + d[j];
                g[j] = dx[j];
            }
            sp.row(g, a.ma, ip, wp, lane);
            row_store(a.dt, r, W, lane, g);
        }
        row_store(a.dx, r, W, lane, dx);
    }
    if (below) {
#pragma unroll
        for (int y = 0; y < 3; ++y) sq[y].flush(sums, a.part_qkv[y], a.ma, lane, wv);
    }
    if (post) {
        sf.flush(sums, a.part_ffn, a.mf, lane, wv);
        sp.flush(sums, a.part_proj, a.ma, lane, wv);
    }
}

template <class F>
bool by_chain_shape(const Mesh &ma, const Mesh &mf, F &&f) {
    using std::integral_constant;
    const int cpl = mesh_wave_cpl(ma.W);
    if (cpl == 1 && ma.depth <= 4 && mf.depth <= 8)
        f(integral_constant<int, 1>{}, integral_constant<int, 4>{}, integral_constant<int, 8>{});
    else if (cpl == 1 && ma.depth <= 8 && mf.depth <= 8)
        f(integral_constant<int, 1>{}, integral_constant<int, 8>{}, integral_constant<int, 8>{});
    else if (cpl == 2 && ma.depth <= 4 && mf.depth <= 8)
        f(integral_constant<int, 2>{}, integral_constant<int, 4>{}, integral_constant<int, 8>{});
    else
        return false;
    return true;
}

}  // namespace

bool chain_fits(const Mesh &ma, const Mesh &mf, int H) {
    const int hd = ma.W / H;
    return hd >= 2 && hd <= 64 && (hd & (hd - 1)) == 0 && by_chain_shape(ma, mf, [](auto, auto, auto) {});
}

// The backward keeps the sums of five stacks in registers.
bool backward_chain_fits(const Mesh &ma, const Mesh &mf, int H) { return ma.depth <= 4 && chain_fits(ma, mf, H); }

// An AdamW update (a captured step) or, without a backward, cross_entropy against
// the separate launches: the chain stores what they store and reads what one of
// them reads, so it is ahead at most sizes (1024 to 131072 rows 0.91 to 0.99 of an
// update and 0.79 to 0.96 of a cross_entropy).  Behind it is by the shuffles of
// butterfly strides where few rows wait for them: W64, seven layers, 256 rows 1.03
// of an update; W128, four, 1.01 to 1.04.
bool forward_chain_pays(const Mesh &ma, int rows, bool backward) {
    return !backward || !ma.butterfly || rows >= 1024 || (ma.depth <= 4 && ma.W <= 64);
}

// A wave takes its rows one after another and one workgroup's registers fill a
// SIMD, so the launches saved are lost again where every SIMD has several rows.
// An update with the forward chain, with this one as well (of the separate
// launches' time): W32 256 rows 0.975 and 0.982, 2048 0.968 and 0.928, 4096 0.937 and
// 0.952; W128 256 rows 0.996 and 1.033 (six blocks 0.978 and 0.941), 1024 0.973 and 0.947, 4096 0.950 and 0.939,
// 8192 0.947 and 0.991.  Stacks of up to eight layers had a form too and gained
// nothing at any size.
bool backward_chain_pays(const Mesh &ma, int layers, int rows) {
    return ma.W > 64 ? (rows >= 512 || layers >= 4) && rows <= 4096 : rows <= 3072;
}

void forward_chain(const ForwardChain &a, hipStream_t stream) {
    by_chain_shape(a.ma, a.mf, [&](auto C, auto A, auto F) {
        hipLaunchKernelGGL((forward_chain_kernel<decltype(C)::value, decltype(A)::value, decltype(F)::value>),
                           dim3(unsigned((a.rows + kThreads / 64 - 1) / (kThreads / 64))), dim3(kThreads), 0, stream, a);
    });
}

void backward_chain(const BackwardChain &a, std::vector<GradReduce> *reductions, float *const *grad,
                    hipStream_t stream) {
    const int groups = mesh_wave_groups(a.rows);
    by_chain_shape(a.ma, a.mf, [&](auto C, auto A, auto F) {
        constexpr int CC = decltype(C)::value, AA = std::min(decltype(A)::value, 4), FF = decltype(F)::value;
        static_assert(2 * CC * (4 * AA + FF) <= kChainSums, "weight-gradient sums stay in registers");
        const size_t lds = size_t(kThreads / 64) * std::max(a.ma.depth, a.mf.depth) * a.ma.W * 2 * sizeof(float);
        hipLaunchKernelGGL((backward_chain_kernel<CC, AA, FF>), dim3(unsigned(groups)), dim3(kThreads), lds, stream, a);
    });
    auto add = [&](const float *part, float *out, const Mesh &m) {
        reductions->push_back(GradReduce{part, out, groups, m.depth * m.W * 2});
    };
    if (a.wqkv[0])
        for (int y = 0; y < 3; ++y) add(a.part_qkv[y], grad[y], a.ma);
    if (a.wffn) {
        add(a.part_ffn, grad[3], a.mf);
        add(a.part_proj, grad[4], a.ma);
    }
}

}  // namespace meshgpt::kern::train
