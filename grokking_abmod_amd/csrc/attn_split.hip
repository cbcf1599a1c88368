// Causal flash attention for long prefills on the FP16 matrix cores of gfx950
// at FP32 accuracy (reference.rs:510-554, XSA 577-603).
//
// What bounds the FP32 matrix-core kernel (attn_mfma.hip) is its instruction
// rate: v_mfma_f32_16x16x4f32 does a sixteenth of the work per cycle of
// v_mfma_f32_32x32x16_f16.  So every f32 operand x is split into two halves,
// h = f16(x) and m = f16(x - h) (both rounded to nearest): h + m is x to within
// 2^-24 of it, f32's own rounding, as long as no half is so small that f16's
// fixed spacing below 2^-14 shows.  A product x y is h h' + h m' + m h'; what is
// left out, m m', is below 2^-24 of it.  Three FP16 products in FP32
// accumulators take 3/16 of the FP32 instructions' time.
//
// Scales keep the halves in range, and all are powers of two:
//  - q (times log2(e)/sqrt(hd)) by 2^14 and k by 2^12: QK-Norm bounds each of
//    a row's entries by sqrt(hd) <= 8, so nothing reaches 65504 and entries
//    2^-13 times a typical one still keep 24 bits;
//  - v by 2^(14 - e), e the exponent of its key tile's largest |v|, and the
//    probability by 2^(14 + e - E), E the largest e of the (sequence, head),
//    so that every tile adds in the same units;
//  - v's second half by 2^11 more, and the probability's first half by 2^-11
//    where it meets it: one scale serves all of a tile's channels, and so an
//    entry keeps 24 bits down to 2^-26 of the tile's largest and not to 2^-15.
// A (sequence, head) runs in the FP32 kernel instead where that is not enough:
//  - its smallest row's largest entry lies more than 2^kSplitSpread below the
//    largest of all (the probabilities' scale then takes their low bits);
//  - a tile holds more than kSplitTiny entries below 2^(e - 26), as a channel
//    that is small in every row does.  (Normally distributed values have such
//    an entry once in some 2500 tiles, by chance, and it is off by less than
//    2^-50 of the tile's largest);
//  - an entry is not finite.
//
// attn_split_prepare_kernel writes k and v of a key tile once as f16 planes in
// the order the products read them: k as [key][dim], v as [dim][key].  Each
// plane's rows are cut into 16-byte slots that are rotated by row so that the
// 16 rows a 16-byte LDS read covers lie in distinct banks.  v's keys are
// ordered within each 16 so that the probabilities a lane holds after the
// first product (keys 8 a + 4 (lane / 32) + b of query lane % 32) are, in
// order, the operand of the second.  The planes are as large as k and v.
//
// Measured on 64 pairs of 8192 rows of 64 dims (0.55 TFLOP a launch): 1.66 ms,
// 0.99 PFLOP/s of FP16 products, where a large bf16 matrix product of a library
// reaches 1.21 on the same card; the FP32 kernel takes 5.25 ms.  (v's second
// half without its own scale: 1.65 ms.)  More waves on a SIMD (128 registers,
// four waves) are slower (9.99 against 9.07 ms a prefill).  Forming the next
// tile's scores beside this one's softmax in each wave gains nothing (7.6-7.9 ms
// a prefill against 7.5): two waves a SIMD already overlap the two.
//
// The error against 64 bits is the FP32 kernel's with seeded and with normally
// distributed weights (8 x 8192 rows, three draws: 1.8e-7 and 1.8e-7, 2.1e-7 and
// 2.1e-7, 1.9e-7 and 2.0e-7; 320 rows with every third value channel 2^-12 of the
// others' size and grown back behind the attention: 9.2e-8 both).  Where XSA
// takes away all but rounding, the operands' own rounding shows: up to 1.7 times
// the FP32 kernel's error with sixteen token vectors that differ in signs only.
// The probability's scale multiplies the exponential's result: added to its
// argument it cost no instruction, but arguments near 14 round to 2^-21 and put
// a tenth on the logits' error.
#include <hip/hip_runtime.h>

#include <cmath>

#include "attn_range.hpp"
#include "kernels.hpp"
#include "lds_dma.hpp"

namespace meshgpt::kern {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));

// (f64(1e-12f))^2 rounded to f32: the XSA norm floor of reference.rs:591.
constexpr float kXsaNormFloor = float(double(1e-12f) * double(1e-12f));

constexpr int kBK = kSplitKeys;
constexpr float kLowScale = 2048.0f;  // of v's second half
constexpr float kQScale = 16384.0f, kKScale = 4096.0f, kScoreUnit = 1.0f / (16384.0f * 4096.0f);

template <int HD>
struct Split {
    static constexpr int KPLANE = kBK * HD;          // halves of one plane (k or v, h or m)
    static constexpr int TILE = 4 * KPLANE;          // halves of a tile: k h, k m, v h, v m
    static constexpr int KSTEPS = HD / 16, DB = HD / 32, VSTEPS = kBK / 16;
};

// Halves from a plane row's start to 16-byte slot c of `row`, rows of 8 * SLOTS
// halves: 16 consecutive rows at one c cover every 16-byte bank group once.
template <int SLOTS>
__device__ __forceinline__ int slot_at(int row, int c) {
    constexpr int PER = 16 / SLOTS;  // rows that share a 256-byte span
    return row * 8 * SLOTS + 8 * (c ^ ((row / PER) & (SLOTS - 1)));
}

__device__ __forceinline__ v16f mfma(h8 a, h8 b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// x as h + m / low.
__device__ __forceinline__ void split(const float (&x)[8], h8 &h, h8 &m, float low = 1.0f) {
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const f2 v = {x[i], x[i + 1]};
        const h2 a = __builtin_convertvector(v, h2);
        const f2 r = {(x[i] - float(a[0])) * low, (x[i + 1] - float(a[1])) * low};
        const h2 b = __builtin_convertvector(r, h2);
        h[i] = a[0];
        h[i + 1] = a[1];
        m[i] = b[0];
        m[i + 1] = b[1];
    }
}

__device__ __forceinline__ int exponent_of(float x) {
    int e = 0;
    (void)frexpf(x, &e);
    return e;
}

// The planes of one tile, and its range (pair_splits): the exponent of its
// largest |v| and of its smallest row's, kBadRange when an entry is not finite,
// all are below 2^-100 or more than kSplitTiny are too small beside the largest.
// Zeros have no size: they count for none of these.
template <int HD>
__global__ void __launch_bounds__(256)
attn_split_prepare_kernel(KvView kv, int n, int tiles, _Float16 *__restrict__ planes, int2 *__restrict__ range) {
    using C = Split<HD>;
    __shared__ float big[4], small[4];
    __shared__ int tiny[4];
    const int tile = int(blockIdx.x) % tiles, pair = int(blockIdx.x) / tiles, t0 = tile * kBK;
    const int lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
    const size_t slab = size_t(pair) * kv.cap * HD;
    _Float16 *out = planes + size_t(blockIdx.x) * C::TILE;
    // k: 8 dims of a key a piece.
    constexpr int KP = kBK * HD / 8 / 256;
#pragma unroll
    for (int u = 0; u < KP; ++u) {
        const int at = u * 256 + int(threadIdx.x), key = at / (HD / 8), c = at % (HD / 8);
        float x[8] = {};
        if (t0 + key < n) {
            const float4 *src = reinterpret_cast<const float4 *>(kv.k + slab + size_t(t0 + key) * HD + 8 * c);
            const float4 a = src[0], b = src[1];
            x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w, x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] *= kKScale;
        h8 h, m;
        split(x, h, m);
        *reinterpret_cast<h8 *>(out + slot_at<HD / 8>(key, c)) = h;
        *reinterpret_cast<h8 *>(out + C::KPLANE + slot_at<HD / 8>(key, c)) = m;
    }
    // v: one dim of 8 keys a piece; slot c of a dim's row holds keys
    // 16 (c / 2) + 8 (i / 4) + 4 (c % 2) + i % 4.  A wave's lanes cover 64 / HD
    // slots of all HD dims.
    constexpr int PER = 64 / HD, VP = 8 / (4 * PER);
    float x[VP][8], top = 0.0f, low = INFINITY;
    bool finite = true;
#pragma unroll
    for (int u = 0; u < VP; ++u) {
        const int d = lane % HD, c = (u * 4 + wave) * PER + lane / HD;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int key = 16 * (c / 2) + 8 * (i / 4) + 4 * (c % 2) + i % 4;
            x[u][i] = t0 + key < n ? kv.v[slab + size_t(t0 + key) * HD + d] : 0.0f;
            finite = finite && isfinite(x[u][i]);
            float row = fabsf(x[u][i]);
#pragma unroll
            for (int k = 1; k < HD; k <<= 1) row = fmaxf(row, __shfl_xor(row, k, 64));
            top = fmaxf(top, row);
            low = fminf(low, row > 0.0f ? row : INFINITY);
        }
    }
    if (HD < 64) {
        top = fmaxf(top, __shfl_xor(top, 32, 64));
        low = fminf(low, __shfl_xor(low, 32, 64));
    }
    finite = __all(finite);
    if (lane == 0) {
        big[wave] = finite ? top : INFINITY;
        small[wave] = low;
    }
    __syncthreads();
    top = fmaxf(fmaxf(big[0], big[1]), fmaxf(big[2], big[3]));
    low = fminf(fminf(small[0], small[1]), fminf(small[2], small[3]));
    const int e = isfinite(top) && top > 0.0f ? exponent_of(top) : 0;
    const bool good = isfinite(top) && e >= -100;
    const float scale = good ? ldexpf(1.0f, 14 - e) : 0.0f;
    int few = 0;
#pragma unroll
    for (int u = 0; u < VP; ++u) {
        const int d = lane % HD, c = (u * 4 + wave) * PER + lane / HD;
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            y[i] = x[u][i] * scale;
            few += int(__popcll(__ballot(fabsf(y[i]) < 0x1p-12f && x[u][i] != 0.0f)));
        }
        h8 h, m;
        split(y, h, m, kLowScale);
        *reinterpret_cast<h8 *>(out + 2 * C::KPLANE + slot_at<8>(d, c)) = h;
        *reinterpret_cast<h8 *>(out + 3 * C::KPLANE + slot_at<8>(d, c)) = m;
    }
    if (lane == 0) tiny[wave] = few;
    __syncthreads();
    const bool even = tiny[0] + tiny[1] + tiny[2] + tiny[3] <= kSplitTiny;
    if (threadIdx.x == 0)
        range[blockIdx.x] = !good || !even       ? make_int2(kBadRange, 0)
                            : isfinite(low)      ? make_int2(e, exponent_of(low))
                                                 : make_int2(-kNoRow, kNoRow);
}

// A workgroup of WAVES waves takes 32 WAVES queries of one (sequence, head),
// 32 a wave (query lane % 32), and streams its key tiles through LDS, double
// buffered.  Per tile a wave forms the transposed scores S^T = K Q^T (two
// 32-key blocks) and O^T += V^T P^T (HD / 32 blocks of 32 dims), so that each
// lane keeps one query's scores, probabilities and outputs.
// Workgroup i runs on XCD i % 8: the query tiles of a (sequence, head) are
// consecutive on one XCD, longest first, so that they share its L2.
template <int HD, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, 2)
attn_split_kernel(Shape s, const float *__restrict__ q, KvView kv, const _Float16 *__restrict__ planes,
                  const int2 *__restrict__ range, int nseq, int n, float *__restrict__ y, float scale_log2, int xsa) {
    using C = Split<HD>;
    __shared__ __align__(16) _Float16 lds[2 * C::TILE];
    constexpr int QT = 32 * WAVES, DMA = C::TILE / 512 / WAVES;
    const int qtiles = (n + QT - 1) / QT, ktiles = (n + kBK - 1) / kBK;
    const int xcd = int(blockIdx.x) % 8, j8 = int(blockIdx.x) / 8;
    const int pair = xcd + 8 * (j8 / qtiles), qt = qtiles - 1 - j8 % qtiles;
    if (pair >= nseq * s.H) return;
    const int seq = pair / s.H, h = pair - seq * s.H;
    const int lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6, jq = lane & 31, hf = lane >> 5;
    const int qwave = qt * QT + wave * 32, qi = qwave + jq, qlast = min(qt * QT + QT, n) - 1;
    const int2 *tile_range = range + size_t(pair) * ktiles;
    int E;
    if (!pair_splits(tile_range, ktiles, lane, E)) return;

    h8 qh[C::KSTEPS], qm[C::KSTEPS];
#pragma unroll
    for (int k = 0; k < C::KSTEPS; ++k) {
        const float4 *src =
            reinterpret_cast<const float4 *>(q + (size_t(seq) * n + min(qi, n - 1)) * s.W + h * HD + 16 * k + 8 * hf);
        const float4 a = src[0], b = src[1];
        const float sc = scale_log2 * kQScale;
        const float x[8] = {a.x * sc, a.y * sc, a.z * sc, a.w * sc, b.x * sc, b.y * sc, b.z * sc, b.w * sc};
        split(x, qh[k], qm[k]);
    }
    v16f acc[C::DB];
#pragma unroll
    for (int d = 0; d < C::DB; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] = 0.0f;
    float m = -INFINITY, l = 0.0f;

    const int ntile = qlast / kBK + 1;
    const char *src = reinterpret_cast<const char *>(planes + size_t(pair) * ktiles * C::TILE) + 16 * lane;
    auto issue = [&](int t) {
        char *to = reinterpret_cast<char *>(lds + (t & 1) * C::TILE);
#pragma unroll
        for (int u = 0; u < DMA; ++u) {
            const int piece = wave * DMA + u;
            dma16(src + size_t(t) * (2 * C::TILE) + 1024 * piece, to + 1024 * piece);
        }
    };
    issue(0);
    for (int t = 0; t < ntile; ++t) {
        // Probabilities of this tile are in units of 2^-unit; a tile of zeros
        // adds to their sum only.
        const int top = tile_range[t].x, unit = top == -kNoRow ? 14 : 14 + top - E;
        wait_vm<0>();
        barrier_lds();  // tile t has landed, and every wave is done with tile t - 1
        if (t + 1 < ntile) issue(t + 1);
        const int t0 = t * kBK;
        if (t0 <= qwave + 31) {
            const _Float16 *kp = lds + (t & 1) * C::TILE, *vp = kp + 2 * C::KPLANE;
            v16f sc[2];
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[b][i] = 0.0f;
#pragma unroll
            for (int k = 0; k < C::KSTEPS; ++k) {
                h8 kh[2], km[2];
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    kh[b] = *reinterpret_cast<const h8 *>(kp + slot_at<HD / 8>(32 * b + jq, 2 * k + hf));
                    km[b] = *reinterpret_cast<const h8 *>(kp + C::KPLANE + slot_at<HD / 8>(32 * b + jq, 2 * k + hf));
                }
#pragma unroll
                for (int b = 0; b < 2; ++b) sc[b] = mfma(km[b], qh[k], sc[b]);
#pragma unroll
                for (int b = 0; b < 2; ++b) sc[b] = mfma(kh[b], qm[k], sc[b]);
#pragma unroll
                for (int b = 0; b < 2; ++b) sc[b] = mfma(kh[b], qh[k], sc[b]);
            }
            if (t0 + kBK - 1 > qwave) {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (t0 + 32 * b + 8 * (i / 4) + 4 * hf + i % 4 > qi) sc[b][i] = -INFINITY;
            }
            float mx = sc[0][0];
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sc[b][i]);
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * kScoreUnit;
            const float mn = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f(m - mn);
            const float up = ldexpf(1.0f, unit);
            m = mn;
            float sum = 0.0f;
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    sc[b][i] = __builtin_amdgcn_exp2f(fmaf(sc[b][i], kScoreUnit, -mn));
                    sum += sc[b][i];
                }
            l = fmaf(l, alpha, sum);
            if (!__all(alpha == 1.0f)) {
#pragma unroll
                for (int d = 0; d < C::DB; ++d)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[d][i] *= alpha;
            }
#pragma unroll
            for (int k = 0; k < C::VSTEPS; ++k) {
                float p[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) p[i] = sc[k / 2][8 * (k % 2) + i] * up;
                h8 ph, pm;
                split(p, ph, pm);
                const h8 pl = ph * _Float16(1.0f / kLowScale);
                h8 vh[C::DB], vm[C::DB];
#pragma unroll
                for (int d = 0; d < C::DB; ++d) {
                    vh[d] = *reinterpret_cast<const h8 *>(vp + slot_at<8>(32 * d + jq, 2 * k + hf));
                    vm[d] = *reinterpret_cast<const h8 *>(vp + C::KPLANE + slot_at<8>(32 * d + jq, 2 * k + hf));
                }
#pragma unroll
                for (int d = 0; d < C::DB; ++d) acc[d] = mfma(vm[d], pl, acc[d]);
#pragma unroll
                for (int d = 0; d < C::DB; ++d) acc[d] = mfma(vh[d], pm, acc[d]);
#pragma unroll
                for (int d = 0; d < C::DB; ++d) acc[d] = mfma(vh[d], ph, acc[d]);
            }
        }
    }

    // y = O / l, then XSA against the query's own value row.  acc is in units
    // of 2^(28 - E).
    l += __shfl_xor(l, 32, 64);
    const float inv = ldexpf(1.0f / l, E - 28);
    const float *own = kv.v + size_t(pair) * kv.cap * HD + size_t(min(qi, n - 1)) * HD;
    float dot = 0.0f, vsq = 0.0f;
#pragma unroll
    for (int d = 0; d < C::DB; ++d)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const float4 v = *reinterpret_cast<const float4 *>(own + 32 * d + 8 * a + 4 * hf);
            const float vr[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc[d][4 * a + r] *= inv;
                dot = fmaf(acc[d][4 * a + r], vr[r], dot);
                vsq = fmaf(vr[r], vr[r], vsq);
            }
        }
    dot += __shfl_xor(dot, 32, 64);
    vsq += __shfl_xor(vsq, 32, 64);
    const float iv = rsqrtf(fmaxf(vsq, kXsaNormFloor));
    const float c = xsa ? dot * iv : 0.0f;
    if (qi >= n) return;
    float *to = y + (size_t(seq) * n + qi) * s.W + h * HD;
#pragma unroll
    for (int d = 0; d < C::DB; ++d)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const float4 v = *reinterpret_cast<const float4 *>(own + 32 * d + 8 * a + 4 * hf);
            *reinterpret_cast<float4 *>(to + 32 * d + 8 * a + 4 * hf) =
                make_float4(acc[d][4 * a] - c * (v.x * iv), acc[d][4 * a + 1] - c * (v.y * iv),
                            acc[d][4 * a + 2] - c * (v.z * iv), acc[d][4 * a + 3] - c * (v.w * iv));
        }
}

}  // namespace

bool attn_split_supported(const Shape &s) {
    return s.hd == s.hdp && (s.hd == 32 || s.hd == 64) && s.W % 4 == 0 && s.qk_norm;
}

// Writing the planes and the launch that looks for pairs left to FP32 cost some
// 5 us a block, which the faster products gain back where there are enough of
// them.  A forward against the FP32 kernel alone (us, W512, 6 blocks, head width
// 64): 288 rows and 8 pairs 383 and 356, 96 498 and 471, 128 569 and 579; 350 rows
// and 64 pairs 483 and 489, 96 574 and 619; 449 rows and 32 pairs 460 and 446, 64
// 510 and 586; 576 rows and 8 pairs 453 and 464, 32 505 and 542.  Head width 32:
// 384 rows and 64 pairs 388 and 375, 128 451 and 476; 449 rows and 16 pairs 364 and
// 381.  8 x 256 rows 0.51 and 0.47 ms.
bool attn_split_pays(const Shape &s, int nseq, int rows_per_seq) {
    const int pairs = nseq * s.H;
    if (rows_per_seq >= 576) return true;
    if (rows_per_seq >= 448) return s.hd == 32 || pairs >= 64;
    return pairs >= 128 ? rows_per_seq >= 288 : pairs >= 80 && rows_per_seq > 320;
}

size_t attn_split_bytes(const Shape &s, int nseq, int rows_per_seq) {
    const size_t tiles = size_t(nseq) * s.H * ((rows_per_seq + kBK - 1) / kBK);
    return tiles * (4 * kBK * s.hd * sizeof(_Float16) + sizeof(int2));
}

const int2 *attn_split(const Shape &s, const float *q, KvView kv, int nseq, int rows_per_seq, float *y, int xsa,
                       void *scratch, hipStream_t stream) {
    const float scale_log2 = float(1.4426950408889634 / std::sqrt(double(s.hd)));
    const int n = rows_per_seq, ktiles = (n + kBK - 1) / kBK, pairs = nseq * s.H;
    const size_t halves = size_t(4) * kBK * s.hd;
    _Float16 *planes = static_cast<_Float16 *>(scratch);
    int2 *range = reinterpret_cast<int2 *>(planes + size_t(pairs) * ktiles * halves);
    auto launch = [&](auto prepare, auto attend, int waves) {
        hipLaunchKernelGGL(prepare, dim3(unsigned(pairs) * ktiles), dim3(256), 0, stream, kv, n, ktiles, planes, range);
        const int qtiles = (n + 32 * waves - 1) / (32 * waves);
        hipLaunchKernelGGL(attend, dim3(8 * ((pairs + 7) / 8) * qtiles), dim3(64 * waves), 0, stream, s, q, kv, planes,
                           range, nseq, n, y, scale_log2, xsa);
    };
    // 256 queries a workgroup share each tile's loads (8 x 8192 rows: 9.07 ms a
    // prefill against 9.42 with 128); below 2048 rows 128 balance the diagonal
    // better (9 x 1001 rows, W512, 6 blocks: 1.31 ms against 1.48).
    const bool longer = n >= 2048;
    if (s.hd == 32)
        longer ? launch(attn_split_prepare_kernel<32>, attn_split_kernel<32, 8>, 8)
               : launch(attn_split_prepare_kernel<32>, attn_split_kernel<32, 4>, 4);
    else
        longer ? launch(attn_split_prepare_kernel<64>, attn_split_kernel<64, 8>, 8)
               : launch(attn_split_prepare_kernel<64>, attn_split_kernel<64, 4>, 4);
    return range;
}

}  // namespace meshgpt::kern
