// Split products: the projections of several tokens (tla_matmul_batch,
// tla_prefill_forward, a layer over several sequences) as bf16 matrix-core products that
// keep fp32 accuracy: the batched form of the matmuls forward() makes per
// token (src/forward.cpp:180-228, matmul() src/ops.cpp:959-983; weight
// blocks src/gguf.h:56-135).
//
//   out[t][row] (+)= sum_k W[row][k] x[t][k]
//
// Exact splitting.  Every fp32 x is the sum of three bf16 numbers, x = x0 +
// x1 + x2 (x0 = x rounded to bf16, x1 = the remainder rounded, x2 the exact
// rest: 8 + 8 + 8 significant bits).  A quantised weight is d * q (Q4_0,
// Q8_0) or d * (sc * q) (Q6_K) with a small integer q that bf16 holds
// exactly (Q6_K's sc * q, up to 13 bits, as two bf16 pieces); an F16 weight
// is the sum of two bf16 pieces, an F32 weight of three.  Each product of
// two pieces is exact in the fp32 accumulator of v_mfma_f32_16x16x32_bf16,
// so for a block
//   sum_k q x = sum_k q x0 + sum_k q x1 + sum_k q x2
// is an fp32 sum of exact products, and the block scale d multiplies it in
// fp32, once per 32-column block.  Products of pieces below 2^-24 of the
// full product (F16 / Q6_K: w1 x2; F32: w1 x2, w2 x1, w2 x2) are left out.
// Results are fp32 sums of the reference's products in another order: the
// reference's accuracy, not its bits.  The matrix cores' bf16 rate is 16
// times their fp32 rate, so 3-6 bf16 products per fp32 multiply-add still
// leave the product well inside it.
//
// Layout.  x as bf16 planes, in the order the A operand reads them: for each
// tile of 16 tokens, 32-column block kb and plane, 1 KiB whose 16-byte piece
// 16 g + i holds the plane of x[16 tile + i][32 kb + 8 g .. + 7].  A wave's
// operand read is then 1 KiB contiguous, and a wave's K slice of a tile one
// run of memory.  Rows past the last token are never used: a row of A only
// reaches the same row of the result.
//
// The tokens are the A operand and the weight rows the B operand of
// v_mfma_f32_16x16x32_bf16: lane l = 16 g + j supplies token j's and row j's
// values for columns 8 g .. 8 g + 7 of the block, and holds the sums of
// tokens 4 g .. 4 g + 3 for row j -- one block scale per lane.  The weights
// are dequantised in registers.
//
// Three kernels, by the number of tokens (plan_product):
//   direct    up to 16 tokens, or few rows: K over the waves of a workgroup,
//             x split (and normalised) by the workgroup itself;
//   resident  more tokens: a workgroup keeps its rows' decoded weights in
//             registers and streams the x planes of all token tiles past them;
//   tiled     past 64 tokens, where its estimated time is less (weights of several
//             pieces, of which the registers hold few rows; several K ranges): a
//             64 kRW row x 64 token tile per workgroup, x through LDS.
// Every output is a sum in a fixed order, which the shape, the CU count and
// TLA_OPT_SPLIT_K choose: the same bits on every run and for any tiling of the rows
// and tokens.
#include <algorithm>
#include <type_traits>

#include "batch.h"
#include "bf16_split.h"
#include "row_math.h"

namespace tla {
namespace {

constexpr int kThreads = 256;          // the row kernels, range sums
constexpr int kWaves = 8;              // waves per direct / resident workgroup
constexpr int kMaxSlice = 8;           // resident: 32-column blocks per wave, at most
constexpr int kRangeBlocks = kWaves * kMaxSlice;  // and so blocks of one K range, at most
constexpr int kRing = 4;               // resident: blocks of x ahead per wave
constexpr int kMaxRows = 3;            // 16-row subtiles per workgroup, at most

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __attribute__((address_space(1))) void* global_ptr;

// the tiled product
constexpr int kTileThreads = 256;
constexpr int kTileWaves = kTileThreads / 64;
constexpr int kTW = 4;                 // token tiles per workgroup
constexpr int kStages = 3;             // LDS stages, x register stages and weight register stages
constexpr int kStageBytes = 3 * kTW * 1024;
constexpr int kChunksPerWave = kStageBytes / 1024 / kTileWaves;  // 1 KiB copies per wave and stage

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));  // 16 raw bytes

__device__ __forceinline__ floatx4 mfma(bf16x8 a, bf16x8 b, floatx4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float half_to_float(unsigned h)
{
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<unsigned short>(h)));
}

// silu(v) * u, with the reference's operation order (src/ops.cpp:1107-1148).
__device__ __forceinline__ float gated(float v, float u)
{
    const float sigmoid = 1.0f / (1.0f + expf(-v));
    return (v * sigmoid) * u;
}

// Byte offset of plane p of block kb, token tile s, in the split x.
__device__ __forceinline__ long long plane_chunk(int s, int kb, int p, int n_blk)
{
    return (static_cast<long long>(s * n_blk + kb) * 3 + p) * 1024;
}

// The three planes of eight values.  An infinity keeps its products: (inf, 0,
// 0), not (inf, NaN, NaN); a finite value that rounds to a bf16 infinity is
// truncated instead (its rest still fits the other two pieces).
__device__ __forceinline__ void split_any(const float (&v)[8], bf16x8 (&x)[3])
{
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        __bf16 a, b, c;
        split3(v[e], a, b, c);
        if (__builtin_isinf(static_cast<float>(a))) {
            if (__builtin_isinf(v[e])) {
                b = c = static_cast<__bf16>(0.f);
            } else {
                const float t = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v[e]) & 0xFFFF0000u);
                a = static_cast<__bf16>(t);
                split2(v[e] - t, b, c);
            }
        }
        x[0][e] = a;
        x[1][e] = b;
        x[2][e] = c;
    }
}

// Eight values of token t, columns 8 c8 .. + 7, into the planes.
__device__ __forceinline__ void store_pieces(unsigned char* xs, int t, int c8, int n_blk, const float (&v)[8])
{
    bf16x8 x[3];
    split_any(v, x);
    const int slot = 16 * (c8 & 3) + (t & 15);
#pragma unroll
    for (int pl = 0; pl < 3; ++pl)
        *reinterpret_cast<bf16x8*>(xs + plane_chunk(t >> 4, c8 >> 2, pl, n_blk) + 16 * slot) = x[pl];
}

__device__ __forceinline__ void load8(const float* p, float (&v)[8])
{
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// One thread per (token tile s, block kb, lane slot 16 g + i): the three
// planes of x[16 s + i][32 kb + 8 g .. + 7].
// kGated: x rows are [gate | up] (2 cols floats) and the value is silu(gate)
// * up, with the reference's operation order (src/ops.cpp:1107-1148).
template <bool kGated>
__global__ __launch_bounds__(kThreads) void split_rows_kernel(const float* __restrict__ x, long long x_stride,
                                                              int n, int n_tiles, int n_blk,
                                                              unsigned char* __restrict__ xs)
{
    const long long id = static_cast<long long>(blockIdx.x) * kThreads + threadIdx.x;
    if (id >= static_cast<long long>(n_blk) * n_tiles * 64) return;
    const int slot = static_cast<int>(id & 63), g = slot >> 4, i = slot & 15;
    const long long rest = id >> 6;
    const int kb = static_cast<int>(rest % n_blk), t = 16 * static_cast<int>(rest / n_blk) + i;
    if (t >= n) return;
    float v[8];
    const float* const row = x + t * x_stride + 32 * kb + 8 * g;
    load8(row, v);
    if constexpr (kGated) {
        float u[8];
        load8(row + 32 * n_blk, u);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = gated(v[e], u[e]);
    }
    store_pieces(xs, t, 4 * kb + g, n_blk, v);
}

// rmsnorm of each row of x into the planes, one workgroup per row (its pieces
// are 16-byte stores into 16-token chunks; one launch of ~5 us at 64 rows in place of
// the norm's and the split's).  With
// k_splits > 0 the row first takes the K-range sums part[z][t][c] of the
// product before (in range order, as range_sum_kernel adds them), and is
// written back.
__global__ __launch_bounds__(kThreads) void norm_split_rows_kernel(float* x, const float* part, int k_splits,
                                                                   long long plane, const float* w, int cols,
                                                                   float eps, unsigned char* xs)
{
    __shared__ float s_sum[kThreads / 64];
    const int t = blockIdx.x;
    float* const row = x + static_cast<long long>(t) * cols;
    const float* const prow = part + static_cast<long long>(t) * cols;
    const auto take = [&](int c8, float (&v)[8]) __attribute__((always_inline)) {
        load8(row + 8 * c8, v);
        if (k_splits > 0) {
            float a[8];
            load8(prow + 8 * c8, a);
            for (int z = 1; z < k_splits; ++z) {
                float b[8];
                load8(prow + z * plane + 8 * c8, b);
#pragma unroll
                for (int e = 0; e < 8; ++e) a[e] += b[e];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += a[e];
        }
    };
    float first[8];
    float ss = 0.f;
    for (int c8 = threadIdx.x; c8 < cols / 8; c8 += kThreads) {
        float v[8];
        take(c8, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
        if (k_splits > 0) {
            reinterpret_cast<float4*>(row + 8 * c8)[0] = make_float4(v[0], v[1], v[2], v[3]);
            reinterpret_cast<float4*>(row + 8 * c8)[1] = make_float4(v[4], v[5], v[6], v[7]);
        }
        if (c8 == static_cast<int>(threadIdx.x))
#pragma unroll
            for (int e = 0; e < 8; ++e) first[e] = v[e];
    }
    ss = block_sum<kThreads>(ss, s_sum);
    const float rms = 1.0f / sqrtf(ss / static_cast<float>(cols) + eps);
    for (int c8 = threadIdx.x; c8 < cols / 8; c8 += kThreads) {
        float v[8], nw[8];
        load8(w + 8 * c8, nw);
        if (c8 == static_cast<int>(threadIdx.x)) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = first[e];
        } else {
            load8(row + 8 * c8, v);  // this thread's own stores, read back
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = v[e] * rms * nw[e];
        store_pieces(xs, t, c8, cols / 32, v);
    }
}

// One lane's raw weight bits for one row and block, as loaded (decoded only
// when the block's turn comes, so that the loads ahead stay in flight).
template <int kType>
struct WRaw;
template <>
struct WRaw<kF32> {
    uint4 a, b;  // the lane's 8 floats
};
template <>
struct WRaw<kF16> {
    uint4 h;  // the lane's 8 halves
};
template <>
struct WRaw<kQ8_0> {
    unsigned u[3];  // 12 bytes holding the lane's 8 bytes of qs (and the scale for g = 0)
};
template <>
struct WRaw<kQ4_0> {
    unsigned u[3];
};
template <>
struct WRaw<kQ6_K> {
    unsigned ql[2], qh[2];  // the lane's 8 bytes of ql and of qh
    unsigned sd;            // the lane's sub-block scale (bits 0..7) and d (bits 16..31)
};

// B pieces per format, and whether a block scale multiplies each block's sum.
template <int kType>
struct Fmt {
    static constexpr int kN = kType == kF32 ? 3 : (kType == kF16 || kType == kQ6_K) ? 2 : 1;
    static constexpr bool kScaled = kType == kQ4_0 || kType == kQ8_0 || kType == kQ6_K;
};

// Loads of block kb of one weight row (wrow) for lane group g.  kRowLoads:
// the memory instructions they are at least (separate addresses the
// compiler cannot merge), which the tiled kernel's wait for its LDS copies
// counts.
template <int kType>
constexpr int kRowLoads = kType == kF32 ? 2 : 1;

template <int kType>
__device__ __forceinline__ void load_w(WRaw<kType>& w, const unsigned char* wrow, int kb, int g)
{
    if constexpr (kType == kF32) {
        const uint4* q = reinterpret_cast<const uint4*>(wrow + 4LL * (32 * kb + 8 * g));
        w.a = q[0];
        w.b = q[1];
    } else if constexpr (kType == kF16) {
        w.h = *reinterpret_cast<const uint4*>(wrow + 2LL * (32 * kb + 8 * g));
    } else if constexpr (kType == kQ6_K) {
        // Q6_K super-block (ql[128] qh[64] scales[16] d; 210 bytes, 256
        // values): value r = 32 (kb % 8) + 8 g + e lies in half h = (kb % 8)
        // / 4, quarter k = kb % 4, at l = 8 g + e; its 6-bit q is a nibble of
        // ql[64 h + 32 (k % 2) + l] (low for k < 2) and bits 2k of
        // qh[32 h + l]; its scale scales[8 h + 2 k + l / 16].
        const unsigned char* sb = wrow + 210LL * (kb >> 3);
        const int h = (kb & 7) >> 2, k = kb & 3;
        __builtin_memcpy(w.ql, sb + 64 * h + 32 * (k & 1) + 8 * g, 8);
        __builtin_memcpy(w.qh, sb + 128 + 32 * h + 8 * g, 8);
        const unsigned sc = sb[192 + 8 * h + 2 * k + (g >> 1)];
        unsigned short d;
        __builtin_memcpy(&d, sb + 208, 2);
        w.sd = sc | (static_cast<unsigned>(d) << 16);
    } else {
        // One dword-aligned 12-byte load holding the lane's 8 bytes of qs: from
        // byte 0 of the block (+ 8 h) for an even block, from 2 bytes before
        // it for an odd one (rows start on dwords and hold whole pairs of
        // blocks, so the load stays inside the row).  The lanes with h = 0
        // get the block's scale with it.
        constexpr int kBlock = kType == kQ8_0 ? 34 : 18;
        const int h = kType == kQ8_0 ? g : (g & 1);  // which 8 bytes of qs
        const unsigned char* p = wrow + static_cast<long long>(kBlock) * kb + 8 * h - 2 * (kb & 1);
        const unsigned* const q = reinterpret_cast<const unsigned*>(p);
        w.u[0] = q[0];
        w.u[1] = q[1];
        w.u[2] = q[2];
    }
}

// The lane's B pieces (their sum: the lane's 8 weights of block kb, divided
// by the block scale where there is one) and the block scale.
template <int kType>
__device__ __forceinline__ void decode_w(const WRaw<kType>& w, int kb, int g, bf16x8 (&b)[Fmt<kType>::kN],
                                         unsigned& d)
{
    d = 0;
    if constexpr (kType == kF32) {
        const unsigned u[8] = {w.a.x, w.a.y, w.a.z, w.a.w, w.b.x, w.b.y, w.b.z, w.b.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            __bf16 p0, p1, p2;
            split3(__builtin_bit_cast(float, u[e]), p0, p1, p2);
            b[0][e] = p0;
            b[1][e] = p1;
            b[2][e] = p2;
        }
    } else if constexpr (kType == kF16) {
        const unsigned u[4] = {w.h.x, w.h.y, w.h.z, w.h.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            __bf16 p0, p1;
            split2(half_to_float((u[e >> 1] >> (16 * (e & 1))) & 0xFFFFu), p0, p1);
            b[0][e] = p0;
            b[1][e] = p1;
        }
    } else if constexpr (kType == kQ6_K) {
        const int k = kb & 3;
        const int sc = static_cast<signed char>(w.sd & 0xFFu);
        d = w.sd >> 16;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const unsigned lo = (w.ql[e >> 2] >> (8 * (e & 3))) & 0xFFu;
            const unsigned hi = (w.qh[e >> 2] >> (8 * (e & 3))) & 0xFFu;
            const int q = static_cast<int>(((k < 2 ? lo & 0x0Fu : lo >> 4) | (((hi >> (2 * k)) & 3u) << 4))) - 32;
            __bf16 p0, p1;
            split2(static_cast<float>(sc * q), p0, p1);
            b[0][e] = p0;
            b[1][e] = p1;
        }
    } else {
        // the scale from the row's lane of g = 0; the 8 bytes at byte 2 of the
        // load for an even block, at byte 4 for an odd one
        const bool odd = kb & 1;
        d = static_cast<unsigned>(__shfl(odd ? w.u[0] >> 16 : w.u[0], threadIdx.x & 15)) & 0xFFFFu;
        const unsigned q[2] = {odd ? w.u[1] : (w.u[0] >> 16) | (w.u[1] << 16),
                               odd ? w.u[2] : (w.u[1] >> 16) | (w.u[2] << 16)};
        // Each byte u (Q4_0: the nibble masked in place; Q8_0: the byte with
        // its sign bit flipped, q + 128) becomes the float 2^23 + u by one
        // byte permute into the mantissa of 2^23 (0x4B000000), and one
        // subtraction leaves u - 8 (Q4_0) or u - 128 = q (Q8_0): two
        // operations per weight.  Small integers: the bf16 packing is exact.
        constexpr float kBase = kType == kQ8_0 ? 8388736.f : 8388616.f;  // 2^23 + 128, 2^23 + 8
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const unsigned m = kType == kQ8_0 ? q[i] ^ 0x80808080u : (q[i] >> ((g >> 1) * 4)) & 0x0F0F0F0Fu;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // bytes: [m.byte e, 0, 0, 0x4B] (selector 0x0C reads zero)
                const unsigned f = __builtin_amdgcn_perm(0x4B000000u, m, 0x070C0C00u + e);
                b[0][4 * i + e] = static_cast<__bf16>(__builtin_bit_cast(float, f) - kBase);
            }
        }
    }
}

// Weight c of a row, as the reference dequantises it.
template <int kType>
__device__ __forceinline__ float weight_at(const unsigned char* wrow, int c)
{
    const auto half_at = [](const unsigned char* p) { return half_to_float(p[0] | (p[1] << 8)); };
    if constexpr (kType == kF32) {
        return reinterpret_cast<const float*>(wrow)[c];
    } else if constexpr (kType == kF16) {
        return half_at(wrow + 2LL * c);
    } else if constexpr (kType == kQ8_0) {
        const unsigned char* const b = wrow + 34LL * (c >> 5);
        return static_cast<float>(static_cast<signed char>(b[2 + (c & 31)])) * half_at(b);
    } else if constexpr (kType == kQ4_0) {
        const unsigned char* const b = wrow + 18LL * (c >> 5);
        const int q = b[2 + (c & 15)] >> ((c & 16) ? 4 : 0) & 15;
        return static_cast<float>(q - 8) * half_at(b);
    } else {
        const unsigned char* const b = wrow + 210LL * (c >> 8);
        const int h = c >> 7 & 1, k = c >> 5 & 3, l = c & 31;
        const int lo = b[64 * h + 32 * (k & 1) + l] >> (k < 2 ? 0 : 4) & 15, hi = b[128 + 32 * h + l] >> (2 * k) & 3;
        const float sc = static_cast<float>(static_cast<signed char>(b[192 + 8 * h + 2 * k + (l >> 4)]));
        return half_at(b + 208) * sc * static_cast<float>((lo | hi << 4) - 32);
    }
}

__device__ __forceinline__ float plane_value(const unsigned char* xs, int t, int c, int n_blk)
{
    float v = 0.f;
#pragma unroll
    for (int pl = 2; pl >= 0; --pl)
        v += static_cast<float>(*reinterpret_cast<const __bf16*>(
            xs + plane_chunk(t >> 4, c >> 5, pl, n_blk) + 16 * (16 * (c >> 3 & 3) + (t & 15)) + 2 * (c & 7)));
    return v;
}

// Pieces of an infinite operand can cancel to a NaN (inf - inf, 0 * inf), and a
// block's unscaled sum can pass the largest float, where the products
// themselves do neither: a sum that is not finite (redo) is taken again in plain
// fp32 over columns [c0, c1), multiples of 32, of weight row wrow and token t,
// x_at(t, c, scale) from its row or from the planes; bad8(c8): whether the eight
// columns 8 c8 .. of the lane's own token make every sum NaN.  All lanes of the
// wave call it, the sixteen of a group with one t: they share the search for
// NaNs, and the wave takes the other sums one after another, all lanes on each.
// (One token of 512 with a NaN / an infinity, Q4_0, 11264 x 2048, 103 us without:
// a lane per sum 1110 / 1110 us; so 109 / 341.)
template <int kType, class B, class X>
__device__ __forceinline__ float taken_again(float sum, bool redo, const unsigned char* wrow, int t, float scale,
                                             int c0, int c1, B&& bad8, X&& x_at)
{
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));  // nothing of this is computed ahead, in registers the loops need
    bool bad = false;
#pragma unroll 1
    for (int c8 = c0 / 8 + (lane & 15); c8 < c1 / 8; c8 += 16) bad |= bad8(c8);
    bad = (__ballot(bad) >> (lane & 48) & 0xFFFF) != 0;
    if (redo && bad) sum = __builtin_nanf("");
    const unsigned long long row = reinterpret_cast<unsigned long long>(wrow);
#pragma unroll 1
    for (unsigned long long left = __ballot(redo && !bad); left; left &= left - 1) {
        const int from = __builtin_ctzll(left);
        const unsigned lo = __builtin_amdgcn_readlane(static_cast<unsigned>(row), from);
        const unsigned hi = __builtin_amdgcn_readlane(static_cast<unsigned>(row >> 32), from);
        const unsigned char* const w = reinterpret_cast<const unsigned char*>(static_cast<unsigned long long>(hi) << 32 | lo);
        const int tok = __builtin_amdgcn_readlane(t, from);
        const float sc = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, scale), from));
        float s = 0.f;
#pragma unroll 1
        for (int c = c0 + lane; c < c1; c += 64) s += weight_at<kType>(w, c) * x_at(tok, c, sc);
#pragma unroll
        for (int d = 32; d; d >>= 1) s += __shfl_xor(s, d);
        sum = lane == from ? s : sum;
    }
    return sum;
}

// The same for x in the planes.
template <int kType>
__device__ __forceinline__ float taken_again(float sum, bool redo, const unsigned char* wrow, int t, int c0, int c1,
                                             const unsigned char* xs, int n_blk)
{
    return taken_again<kType>(
        sum, redo, wrow, t, 1.f, c0, c1,
        [&](int c8) {
            const bf16x8 x0 = *reinterpret_cast<const bf16x8*>(xs + plane_chunk(t >> 4, c8 >> 2, 0, n_blk) +
                                                               16 * (16 * (c8 & 3) + (t & 15)));
            bool nan = false;
#pragma unroll
            for (int e = 0; e < 8; ++e) nan |= __builtin_isnan(static_cast<float>(x0[e]));
            return nan;
        },
        [&](int tok, int c, float) { return plane_value(xs, tok, c, n_blk); });
}

// The segment holding a row: selected field by field (an index into the
// kernel-argument array would copy it to scratch memory).
struct RowSeg {
    const unsigned char* w;
    float* out;
    long long stride;
    int row;  // within the segment
};
template <class Params>
__device__ __forceinline__ RowSeg row_seg(const Params& p, int row)
{
    RowSeg r{p.seg[0].w, p.seg[0].out, p.seg[0].out_stride, row};
    int cur = 0;  // the segment r is in so far; only its successor can take the row
#pragma unroll
    for (int i = 1; i < kGemvMaxSeg; ++i) {
        const bool next = cur == i - 1 && i < p.n_seg && r.row >= p.seg[i - 1].rows;
        cur = next ? i : cur;
        r.row = next ? r.row - p.seg[i - 1].rows : r.row;
        r.w = next ? p.seg[i].w : r.w;
        r.out = next ? p.seg[i].out : r.out;
        r.stride = next ? p.seg[i].out_stride : r.stride;
    }
    return r;
}

// The lane's 8 weights of an F32 block.
template <int kType>
__device__ __forceinline__ split_f32x8 float_w(const WRaw<kType>& w)
{
    split_f32x8 v{};
    if constexpr (kType == kF32) {
        const unsigned u[8] = {w.a.x, w.a.y, w.a.z, w.a.w, w.b.x, w.b.y, w.b.z, w.b.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = __builtin_bit_cast(float, u[e]);
    }
    return v;
}

// One block's products for kR row subtiles: acc (+)= the products of pieces
// (x_p, b_i) with i + p <= 2, smallest terms first, scaled by the block scale
// (the bits of a half) where there is one.  Each block is summed from zero:
// carried through the matrix cores from block to block, F16 sums were 2.2e-7
// off fp64 at 2048 columns against 1e-7.
template <int kType, int kR>
__device__ __forceinline__ void block_products(const bf16x8 (&x)[3], const bf16x8 (&b)[kR][Fmt<kType>::kN],
                                               const unsigned (&d)[kR], floatx4 (&acc)[kR])
{
    constexpr int kN = Fmt<kType>::kN;
    floatx4 t[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) t[r] = floatx4{0.f, 0.f, 0.f, 0.f};
    if constexpr (kN >= 3) {
#pragma unroll
        for (int r = 0; r < kR; ++r) t[r] = mfma(x[0], b[r][kN - 1], t[r]);
    }
    if constexpr (kN >= 2) {
#pragma unroll
        for (int r = 0; r < kR; ++r) t[r] = mfma(x[1], b[r][1], t[r]);
#pragma unroll
        for (int r = 0; r < kR; ++r) t[r] = mfma(x[0], b[r][1], t[r]);
    }
#pragma unroll
    for (int pl = 2; pl >= 0; --pl)
#pragma unroll
        for (int r = 0; r < kR; ++r) t[r] = mfma(x[pl], b[r][0], t[r]);
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        if constexpr (Fmt<kType>::kScaled) {
            const float s = half_to_float(d[r]);
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[r][q] = fmaf(s, t[r][q], acc[r][q]);
        } else {
            acc[r] += t[r];
        }
    }
}

// Row j of row subtile `sub`: row 16 sub + j of the segments laid end to end,
// or, paired, gate row 8 sub + j (j < 8) and up row 8 sub + j - 8.  Past the
// end: the last row, not ok.
struct TileRow : RowSeg {
    bool ok;
};
__device__ __forceinline__ TileRow tile_row(const ProductParams& p, int sub, int j)
{
    TileRow r;
    if (p.pair) {
        const int row = 8 * sub + (j & 7), last = p.seg[0].rows - 1;
        const bool up = j >= 8;
        r.w = up ? p.seg[1].w : p.seg[0].w;
        r.out = up ? p.seg[1].out : p.seg[0].out;
        r.stride = up ? p.seg[1].out_stride : p.seg[0].out_stride;
        r.row = min(row, last);
        r.ok = row <= last;
    } else {
        const int row = 16 * sub + j;
        static_cast<RowSeg&>(r) = row_seg(p, min(row, p.total_rows - 1));
        r.ok = row < p.total_rows;
    }
    return r;
}

// Paired, after the raw products: lanes j < 8 hold token t's gate sums of the
// eight rows 8 sub .. + 7, lanes j + 8 their up sums: silu(gate) * up into the
// planes of the down projection's input, where those eight columns of the
// token are one 16-byte piece.  All lanes call it.
__device__ __forceinline__ void store_gated(const ProductParams& p, float sum, int t, int row, bool ok, int j)
{
    const float up = __shfl(sum, (threadIdx.x & 63) ^ 8);
    if (j >= 8 || !ok) return;
    float v[8] = {gated(sum, up), 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    bf16x8 x[3];
    split_any(v, x);
    const int slot = 16 * (row >> 3 & 3) + (t & 15), n_blk = p.seg[0].rows >> 5;
#pragma unroll
    for (int pl = 0; pl < 3; ++pl)
        *reinterpret_cast<__bf16*>(p.hs + plane_chunk(t >> 4, row >> 5, pl, n_blk) + 16 * slot + 2 * (row & 7)) =
            x[pl][0];
}

// ---- direct --------------------------------------------------------------------
// kR row subtiles x one token tile per workgroup, K over its 8 waves (wave w
// blocks w, w + 8, ...; the waves' sums meet in LDS in wave order).  Every
// load a wave makes for 2048 columns is in flight at once: the launch is one
// memory round trip and the vector work after it (splitting x, about 44 operations a
// block, and dequantising, about 30 a subtile; counters: vector units active 27-35
// % of the busy cycles, matrix cores 4-7 %, the rest waits).  With kXNormRows x is
// multiplied by the norm's weights before it is split and the sums by the
// row's 1 / rms at the end, so that no launch goes before it.  Q8_0, 12
// tokens, TinyLlama's layer (kernel trace): rmsnorm + Q/K/V 11.4 us, W_o 8.8,
// rmsnorm + gate | up + SwiGLU 15.0, W_down 12.3, where matrix-vector launches
// (weights read once per 2 to 6 vectors) took 56, 39, 78 and 142 us.  16 waves of
// 128 registers spilled; two row subtiles where one round of workgroups takes
// one cost 2-3 us more; loads behind branches made every block wait for all of
// them (2560 x 2048, Q8_0, 3 tokens, 6.9 against 6.4 us).  F32 weights from fp32 rows take the fp32 matrix cores
// instead (kFp32: lane group g the columns 8 g + e of step e, each block summed
// from zero): one token tile does not repay splitting both operands (2560 x
// 2048, 3 tokens, 9.2 us split, 8.4 so; F16 with three row subtiles 12.9
// split, 15.1 so).
//
// Up to 16 / kShare tokens leave rows of the x operand free: its row set u (of
// kShare) holds the tokens in block u of kShare consecutive ones, so that one
// load and split of x serves them all.  Block u's products go into accumulators
// of their own, of which only row set u counts; the sets meet with the waves'
// sums.  4 tokens, kShare 1 / 2 / 4: F16, 2048 x 5632 13.6 / 11.0 / 10.5 us;
// Q8_0, 2048 x 5632 12.3 / 9.7 / 8.9, 2560 x 2048 6.6 / 5.7 / 5.5.  (More blocks in
// flight instead, 12 or 16: F16, 2048 x 5632, 13.2 -> 14.4 and 16.2.)
enum XSource { kXRows, kXNormRows, kXPlanes };

template <int kType, int kR, int kSrc, int kDepth, int kShare>
__global__ __launch_bounds__(kWaves * 64) void direct_product_kernel(const ProductParams p)
{
    constexpr int kN = Fmt<kType>::kN;
    constexpr bool kNorm = kSrc == kXNormRows;
    constexpr bool kFp32 = kSrc != kXPlanes && kType == kF32;
    constexpr int kCombos = 4 * kR;
    constexpr int kTok = 16 / kShare;  // tokens per tile row set
    __shared__ float s_red[kWaves][kCombos][64];
    __shared__ float s_ss[kWaves][16];
    __shared__ __align__(16) float s_norm[kNorm ? kProductMaxNorm : 4];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int j = lane & 15, g = lane >> 4;
    const int n_blk = p.cols >> 5, tile = blockIdx.y;
    const int sub0 = blockIdx.x * kR;
    // groups of kShare blocks: wave + kWaves i, i < nb
    const int n_grp = (n_blk + kShare - 1) / kShare;
    const int nb = wave < n_grp ? (n_grp - wave + kWaves - 1) / kWaves : 0;
    const int jt = j % kTok, jb = j / kTok;  // this lane's token, and its block of a group
    const unsigned char* wrow[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const TileRow rs = tile_row(p, sub0 + r, j);
        wrow[r] = rs.w + static_cast<long long>(rs.row) * p.row_bytes;
    }
    const float* const xrow = p.x + static_cast<long long>(min(16 * tile + jt, p.n - 1)) * p.x_stride + 8 * g;

    struct Stage {
        WRaw<kType> w[kShare][kR];
        u32x4 x[kSrc == kXPlanes ? 3 : 2];  // eight floats, or their planes
    } st[kDepth];
    // (past the wave's last block that one again, never used: no load sits
    // behind a branch, where the compiler would wait for all in flight)
    const auto load = [&](Stage& t, int i) __attribute__((always_inline)) {
        const int kb = kShare * min(wave + kWaves * min(i, max(nb - 1, 0)), n_grp - 1);
        const int xb = min(kb + jb, n_blk - 1);
        const unsigned char* const src =
            kSrc == kXPlanes ? p.xs + plane_chunk(tile, xb, 0, n_blk) + 16 * (16 * g + jt)
                             : reinterpret_cast<const unsigned char*>(xrow + 32 * xb);
#pragma unroll
        for (int i2 = 0; i2 < (kSrc == kXPlanes ? 3 : 2); ++i2)
            t.x[i2] = *reinterpret_cast<const u32x4*>(src + (kSrc == kXPlanes ? 1024 : 16) * i2);
#pragma unroll
        for (int u = 0; u < kShare; ++u)
#pragma unroll
            for (int r = 0; r < kR; ++r) load_w<kType>(t.w[u][r], wrow[r], min(kb + u, n_blk - 1), g);
    };
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
        load(st[d], d);
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (kNorm) {
        for (int c = 4 * threadIdx.x; c < p.cols; c += 4 * kWaves * 64)
            *reinterpret_cast<float4*>(s_norm + c) = *reinterpret_cast<const float4*>(p.norm_w + c);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the loads above stay in flight
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }
    floatx4 acc[kShare][kR];
#pragma unroll
    for (int u = 0; u < kShare; ++u)
#pragma unroll
        for (int r = 0; r < kR; ++r) acc[u][r] = floatx4{0.f, 0.f, 0.f, 0.f};
    float ss = 0.f;
    const auto block = [&](const Stage& t, int i) __attribute__((always_inline)) {
        const int kb = kShare * (wave + kWaves * i);
        const bool in = kShare == 1 || kb + jb < n_blk;  // a block past the row adds zeros
        split_f32x8 v;
        if constexpr (kSrc != kXPlanes) {
            const float4 xa = __builtin_bit_cast(float4, t.x[0]), xb = __builtin_bit_cast(float4, t.x[1]);
            v = split_f32x8{xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
            if (kShare > 1) v = in ? v : split_f32x8{};
            if constexpr (kNorm) {
                const float4* const nw = reinterpret_cast<const float4*>(s_norm + 32 * (kShare == 1 ? kb : min(kb + jb, n_blk - 1)) + 8 * g);
                const float4 na = nw[0], nb4 = nw[1];
                ss += kShare == 1 || in ? sum_sq4(xa) + sum_sq4(xb) : 0.f;
                v *= split_f32x8{na.x, na.y, na.z, na.w, nb4.x, nb4.y, nb4.z, nb4.w};
            }
        }
        if constexpr (kFp32) {
#pragma unroll
            for (int u = 0; u < kShare; ++u) {
                floatx4 sum[kR];
                split_f32x8 w[kR];
#pragma unroll
                for (int r = 0; r < kR; ++r) {
                    sum[r] = floatx4{0.f, 0.f, 0.f, 0.f};
                    w[r] = float_w<kType>(t.w[u][r]);
                }
#pragma unroll
                for (int e = 0; e < 8; ++e)
#pragma unroll
                    for (int r = 0; r < kR; ++r)
                        sum[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], w[r][e], sum[r], 0, 0, 0);
#pragma unroll
                for (int r = 0; r < kR; ++r) acc[u][r] += sum[r];
            }
        } else {
            bf16x8 x[3];
            if constexpr (kSrc == kXPlanes) {
#pragma unroll
                for (int pl = 0; pl < 3; ++pl) x[pl] = in ? __builtin_bit_cast(bf16x8, t.x[pl]) : bf16x8{};
            } else {
                split3x8(v, x[0], x[1], x[2]);
            }
#pragma unroll
            for (int u = 0; u < kShare; ++u) {
                bf16x8 b[kR][kN];
                unsigned d[kR];
#pragma unroll
                for (int r = 0; r < kR; ++r) decode_w<kType>(t.w[u][r], min(kb + u, n_blk - 1), g, b[r], d[r]);
                block_products<kType, kR>(x, b, d, acc[u]);
            }
        }
    };
    int i0 = 0;
    for (; i0 + kDepth < nb; i0 += kDepth) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            block(st[d], i0 + d);
            __builtin_amdgcn_sched_barrier(0);
            load(st[d], i0 + d + kDepth);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < kDepth; ++d)
        if (i0 + d < nb) block(st[d], i0 + d);  // uniform
#pragma unroll
    for (int r = 0; r < kR; ++r)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            // the set of block g kShare / 4 has its tokens in this lane group's rows
            float sum = acc[0][r][q];
#pragma unroll
            for (int u = 1; u < kShare; ++u) sum = g * kShare / 4 == u ? acc[u][r][q] : sum;
            s_red[wave][4 * r + q][lane] = sum;
        }
    if constexpr (kNorm) {
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        if (g == 0) s_ss[wave][j] = ss;
    }
    __syncthreads();
    // combination c: token 4 g + c % 4 of row subtile c / 4
#pragma unroll
    for (int c0 = 0; c0 < kCombos; c0 += kWaves) {
        const int c = c0 + wave, t = 16 * tile + 4 * g + (c & 3);
        if (c >= kCombos) return;
        float sum = 0.f;
#pragma unroll
        for (int u = 0; u < kShare; ++u)
#pragma unroll
            for (int w = 0; w < kWaves; ++w) sum += s_red[w][c][(lane + 64 / kShare * u) & 63];
        const TileRow rs = tile_row(p, sub0 + (c >> 2), j);
        const bool ok = rs.ok && t < p.n;
        float rms = 1.f;
        if constexpr (kNorm) {
            float s2 = 0.f;
#pragma unroll
            for (int u = 0; u < kShare; ++u)
#pragma unroll
                for (int w = 0; w < kWaves; ++w) s2 += s_ss[w][(4 * g + (c & 3) + kTok * u) & 15];
            rms = 1.0f / sqrtf(s2 / static_cast<float>(p.cols) + p.eps);
        }
        const bool redo = ok && !(fabsf(sum) < __builtin_huge_valf());
        if (__builtin_expect(__any(redo), 0)) {
            const unsigned char* const wr = rs.w + static_cast<long long>(rs.row) * p.row_bytes;
            if constexpr (kSrc == kXPlanes) {
                sum = taken_again<kType>(sum, redo, wr, t, 0, p.cols, p.xs, n_blk);
            } else {
                // normalised value by value: 1 / rms may be zero for a finite
                // row, and makes an infinity NaN
                const int tok = min(t, p.n - 1);
                sum = taken_again<kType>(
                    sum, redo, wr, tok, rms, 0, p.cols,
                    [&](int c8) {
                        float v[8];
                        load8(p.x + tok * p.x_stride + 8 * c8, v);
                        bool bad = false;
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            bad |= kNorm ? !(fabsf(v[e]) < __builtin_huge_valf()) : __builtin_isnan(v[e]);
                        return bad;
                    },
                    [&](int of, int c, float scale) {
                        const float v = p.x[of * p.x_stride + c];
                        return kNorm ? v * scale * s_norm[c] : v;
                    });
            }
        }
        if constexpr (kNorm) sum = redo ? sum : sum * rms;
        if (ok && rs.out) {
            float* const o = rs.out + rs.row + t * rs.stride;
            *o = p.add ? *o + sum : sum;
        }
        if (p.pair) store_gated(p, sum, t, rs.row, ok, j);
    }
}

// ---- resident ------------------------------------------------------------------
// A workgroup of 8 waves holds the decoded weights of kR row subtiles x one K
// range (up to 2048 columns, one slice of kSlice blocks per wave) in registers
// and streams the x planes of its share of the token tiles past them: the
// weights are read and dequantised once per share, and nothing but the planes
// moves per tile.  Each wave keeps kRing blocks of x ahead in registers; the
// waves' sums meet in LDS.  Bound by the planes' way into the CU: a tile is 196 KB per
// workgroup, against 0.96 us of matrix work with three subtiles (measured per tile:
// 1.77 / 1.94 / 2.1 us with 1 / 2 / 3 subtiles in short launches, 46 to 39 B a clock;
// 33 over 512 tokens, where counters show the matrix cores busy 38 % and the vector
// units 41 % of the time, waves waiting for loads for the rest; L2 hits 93 %).  All
// workgroups walk their tiles in the same order, so an
// XCD's share of them meets in its L2; a flat split of (group, tile) units over
// the CUs did not (4 us a tile).  An LDS ring filled by direct loads was slower
// (1.5 us + 0.31 a subtile: written and read, x passes the LDS port twice), and
// so were loads of the weights' 8 bytes at their own 2-byte alignment (gate |
// up, 64 tokens, 49 against 22 us).  Q4_0, 11264 x 2048 with the planes'
// launch, tiled / resident: 65 tokens 37 / 22 us, 160 55 / 34, 512 94 / 80.
template <int kType, int kR, int kSlice>
__global__ __launch_bounds__(kWaves * 64) void resident_product_kernel(const ProductParams p)
{
    constexpr int kN = Fmt<kType>::kN;
    constexpr int kCombos = 4 * kR;                         // (row subtile, token of four) sums per lane
    constexpr int kOuts = (kCombos + kWaves - 1) / kWaves;  // of which each wave finishes
    __shared__ float s_red[2][kWaves][kCombos][64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int j = lane & 15, g = lane >> 4;
    const int n_blk = p.cols >> 5;
    const int tiles = p.n_tiles;
    int buf = 0;
    {
        const int share = blockIdx.x % p.shares, group = blockIdx.x / p.shares;
        const int tile0 = static_cast<int>(static_cast<long long>(tiles) * share / p.shares);
        const int here = static_cast<int>(static_cast<long long>(tiles) * (share + 1) / p.shares) - tile0;
        const int z = group / p.row_groups, sub0 = (group % p.row_groups) * kR;
        // this wave's blocks [kb0, kb0 + nb) of K range z
        const int kb_lo = z * p.blk_per_split, kb_hi = min(kb_lo + p.blk_per_split, n_blk);
        const int per_wave = (kb_hi - kb_lo + 2 * kWaves - 1) / (2 * kWaves) * 2;
        const int kb0 = kb_lo + wave * per_wave;
        const int nb = max(0, min(per_wave, kb_hi - kb0));
        // past the slice: a block of the same parity, loaded but not used
        const auto block_of = [&](int b) { return min(kb0 + b, kb_hi - 2 + (b & 1)); };
        bf16x8 ring[kRing][3];
        const auto load_x = [&](int b, int tile) __attribute__((always_inline)) {
            const unsigned char* const src = p.xs + plane_chunk(tile, block_of(b), 0, n_blk) + 16 * lane;
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) ring[b % kRing][pl] = *reinterpret_cast<const bf16x8*>(src + 1024 * pl);
        };

        // the row group's weights, all requested at once, then the first
        // tile's x; decoded into registers for every tile of the group
        bf16x8 held[kR][kSlice][kN];
        unsigned scale[kR][kSlice / 2];  // two block scales a word, as halves
        {
            WRaw<kType> raw[kR][kSlice];
#pragma unroll
            for (int r = 0; r < kR; ++r) {
                const TileRow rs = tile_row(p, sub0 + r, j);
                const unsigned char* const wrow = rs.w + static_cast<long long>(rs.row) * p.row_bytes;
#pragma unroll
                for (int b = 0; b < kSlice; ++b) load_w<kType>(raw[r][b], wrow, block_of(b), g);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < kRing; ++b) load_x(b, tile0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < kR; ++r)
#pragma unroll
                for (int b = 0; b < kSlice; ++b) {
                    unsigned d;
                    decode_w<kType>(raw[r][b], block_of(b), g, held[r][b], d);
                    scale[r][b / 2] = b % 2 ? scale[r][b / 2] | (d << 16) : d;
                }
        }

        // where this wave's finished sums go: tokens 4 g + c % 4 of row j of
        // subtile c / 4 for its combinations c
        float* out[kOuts];
        long long stride[kOuts];
        bool row_ok[kOuts];
#pragma unroll
        for (int i = 0; i < kOuts; ++i) {
            const int c = wave + kWaves * i;
            const TileRow rs = tile_row(p, sub0 + (c >> 2), j);
            row_ok[i] = c < kCombos && rs.ok;
            if (p.part) {
                out[i] = p.part + static_cast<long long>(z) * p.n * p.total_rows + 16 * (sub0 + (c >> 2)) + j;
                stride[i] = p.total_rows;
            } else {
                out[i] = rs.out ? rs.out + rs.row : nullptr;
                stride[i] = rs.stride;
            }
        }

        const auto tile_step = [&](int tile, auto next) __attribute__((always_inline)) {
            constexpr bool kNext = decltype(next)::value;
            floatx4 acc[kR];
#pragma unroll
            for (int r = 0; r < kR; ++r) acc[r] = floatx4{0.f, 0.f, 0.f, 0.f};
            const auto block_step = [&](int b) __attribute__((always_inline)) {
                if (b >= nb) return;  // uniform
                const bf16x8(&x)[3] = ring[b % kRing];
                bf16x8 w[kR][kN];
                unsigned d[kR];
#pragma unroll
                for (int r = 0; r < kR; ++r) {
                    d[r] = b % 2 ? scale[r][b / 2] >> 16 : scale[r][b / 2] & 0xFFFFu;
#pragma unroll
                    for (int i = 0; i < kN; ++i) w[r][i] = held[r][b][i];
                }
                block_products<kType, kR>(x, w, d, acc);
            };
#pragma unroll
            for (int b = 0; b < kSlice; ++b) {
                block_step(b);
                __builtin_amdgcn_sched_barrier(0);
                if (b + kRing < kSlice)
                    load_x(b + kRing, tile);
                else if constexpr (kNext)
                    load_x(b + kRing - kSlice, tile + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            // the waves' sums in wave order; two buffers, so one barrier a tile
#pragma unroll
            for (int r = 0; r < kR; ++r)
#pragma unroll
                for (int q = 0; q < 4; ++q) s_red[buf][wave][4 * r + q][lane] = acc[r][q];
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the copies ahead stay in flight
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int i = 0; i < kOuts; ++i) {
                const int c = min(wave + kWaves * i, kCombos - 1);
                float sum = s_red[buf][0][c][lane];
#pragma unroll
                for (int w = 1; w < kWaves; ++w) sum += s_red[buf][w][c][lane];
                const int t = 16 * tile + 4 * g + (c & 3);
                const bool ok = row_ok[i] && t < p.n;
                const bool redo = ok && !(fabsf(sum) < __builtin_huge_valf());
                if (__builtin_expect(__any(redo), 0)) {
                    int j_here = j;
                    asm volatile("" : "+v"(j_here));
                    const TileRow rs = tile_row(p, sub0 + (c >> 2), j_here);
                    sum = taken_again<kType>(sum, redo, rs.w + static_cast<long long>(rs.row) * p.row_bytes, t,
                                             32 * kb_lo, 32 * kb_hi, p.xs, n_blk);
                }
                if (ok && out[i]) {
                    float* const o = out[i] + t * stride[i];
                    *o = p.add && !p.part ? *o + sum : sum;
                }
                if (p.pair && wave + kWaves * i < kCombos)
                    store_gated(p, sum, t, 8 * (sub0 + (c >> 2)) + (j & 7), ok, j);
            }
            asm volatile("" ::: "memory");
            buf ^= 1;
        };
#pragma unroll 1
        for (int i = 0; i + 1 < here; ++i) tile_step(tile0 + i, std::true_type{});
        tile_step(tile0 + here - 1, std::false_type{});
    }
}

// ---- tiled ---------------------------------------------------------------------
// A workgroup of 4 waves owns 64 kRW weight rows x 64 tokens (4 token tiles);
// wave w owns rows 16 kRW w .. + 16 kRW - 1 for all 64 tokens.  The x blocks
// pass through a ring of three LDS stages (12 KiB each) filled by direct
// loads two blocks ahead; each wave loads its rows' weights three blocks
// ahead.  Bound by the barrier per block between short stretches of decoding, LDS
// reads and products: neither unit is the limit (counters, 512 tokens: Q4_0 2048 x
// 5632 matrix cores busy 35 %, vector units 55 %; F16 5632 x 2048 51 / 53 %), and
// every XCD reads all the weights.  Carrying the sums
// of types without a scale through the matrix cores was 3-6 % faster and put a
// layer of F16 over 100 sequences 3.6e-7 off fp64 against 1.4e-7.
template <int kType, int kRW>
__global__ __launch_bounds__(kTileThreads) void tiled_product_kernel(const ProductParams p)
{
    // The ring's stages as separate arrays, so that the compiler sees that a
    // stage being read is not the one a copy in flight writes.
    __shared__ __align__(16) unsigned char s_x0[kStageBytes], s_x1[kStageBytes], s_x2[kStageBytes];
    auto stage_base = [&](int u) __attribute__((always_inline)) { return u == 0 ? s_x0 : u == 1 ? s_x1 : s_x2; };
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int j = lane & 15, g = lane >> 4;
    // Tiles by linear workgroup id L, token tile fastest (y = L mod the
    // token tiles): workgroups run on XCD L mod 8, so each XCD's workgroups
    // share a few token tiles' x planes in its L2 (at 512 tokens one XCD one
    // tile, 0.8 MB) while the weights stream through.
    const unsigned L = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const unsigned ty = L % gridDim.y, rest = L / gridDim.y;
    const unsigned tx = rest % gridDim.x, tz = rest / gridDim.x;
    const int n_blk = p.cols >> 5;
    const int row0 = (tx * kTileWaves + wave) * 16 * kRW;
    const int s0 = ty * kTW;  // first token subtile
    const int live = min(kTW, (p.n + 15) / 16 - s0);  // subtiles with tokens
    // K range of this workgroup: blocks [kb_lo, kb_hi) (grid z splits K)
    const int kb_lo = tz * p.blk_per_split;
    const int kb_hi = min(kb_lo + p.blk_per_split, n_blk);

    // this lane's weight row in each row subtile (the last row for rows past
    // the end: loaded, never stored)
    const unsigned char* wrow[kRW];
#pragma unroll
    for (int r = 0; r < kRW; ++r) {
        const RowSeg rs = row_seg(p, min(row0 + 16 * r + j, p.total_rows - 1));
        wrow[r] = rs.w + static_cast<long long>(rs.row) * p.row_bytes;
    }

    // x stage of block kb: 12 chunks of 1 KiB, chunk c = plane c / 4 of
    // token subtile s0 + c % 4, copied by direct global-to-LDS loads, three
    // per wave (lane l's 16 bytes land at byte 16 l of the chunk).  Past the
    // end the last block is copied again (never read), so every iteration
    // issues the same memory operations.
    auto copy_x = [&](int kb, int stage) __attribute__((always_inline)) {
        kb = min(kb, kb_hi - 1);
#pragma unroll
        for (int i = 0; i < kChunksPerWave; ++i) {
            const int c = kChunksPerWave * wave + i;
            __builtin_amdgcn_global_load_lds(
                (global_ptr)(p.xs + plane_chunk(s0 + c % kTW, kb, c / kTW, n_blk) + 16 * lane),
                (lds_ptr)(stage_base(stage) + 1024 * c), 16, 0, 0);
        }
    };
    auto load_ws = [&](WRaw<kType> (&wr)[kRW], int kb) __attribute__((always_inline)) {
        kb = kb < kb_hi ? kb : kb_hi - 2 + (kb & 1);
#pragma unroll
        for (int r = 0; r < kRW; ++r) load_w<kType>(wr[r], wrow[r], kb, g);
    };

    floatx4 acc[kRW][kTW];
#pragma unroll
    for (int r = 0; r < kRW; ++r)
#pragma unroll
        for (int s = 0; s < kTW; ++s) acc[r][s] = floatx4{0.f, 0.f, 0.f, 0.f};

    // Block b: LDS stage b % 3 (copied two iterations before it is read),
    // weights wr<b % 3> (loaded three iterations before use).  Iteration kb:
    // wait for block kb's copy, barrier (every wave's copy has landed and
    // every wave is done with block kb - 1), copy block kb + 2 into block
    // kb - 1's stage, multiply block kb, load block kb + 3's weights.  The
    // wait counts memory operations: after block kb's copy this wave issued
    // block kb + 1's and kb + 2's weights (at least kRowLoads per row each)
    // and block kb + 1's copy (kChunksPerWave), so waiting until no more than
    // that many are outstanding means the copy has landed (they complete in
    // order; a count below the true one only waits longer).  Scheduling
    // barriers keep that order.  Separate arrays per ring
    // slot, chosen at compile time, stay in registers.
    // The prologue issues its operations in the loop's order (weights of
    // block b + 3 after the copy of block b + 2), as if iterations kb_lo - 3
    // .. kb_lo - 1 had run.
    WRaw<kType> wr0[kRW], wr1[kRW], wr2[kRW];
    load_ws(wr0, kb_lo);
    __builtin_amdgcn_sched_barrier(0);
    copy_x(kb_lo, 0);
    __builtin_amdgcn_sched_barrier(0);
    load_ws(wr1, kb_lo + 1);
    __builtin_amdgcn_sched_barrier(0);
    copy_x(kb_lo + 1, 1);
    __builtin_amdgcn_sched_barrier(0);
    load_ws(wr2, kb_lo + 2);
    __builtin_amdgcn_sched_barrier(0);

    constexpr int kAfterCopy = kChunksPerWave + 2 * kRW * kRowLoads<kType>;
    static_assert(kAfterCopy < 64, "vmcnt holds 6 bits");
    constexpr int kVmcntWait = (kAfterCopy & 15) | ((kAfterCopy >> 4) << 14) | 0xF70;  // vmcnt(kAfterCopy)
    auto iteration = [&](int kb, auto& wr_this, const int u, const int u2) __attribute__((always_inline)) {
        // A bare barrier: __syncthreads' release fence would wait for every
        // outstanding load (the copies write LDS through the vector memory
        // path), weights included.  The LDS reads of block kb - 1 were used
        // before this point, so its stage is free once every wave is here.
        __builtin_amdgcn_s_waitcnt(kVmcntWait);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        copy_x(kb + 2, u2);
        __builtin_amdgcn_sched_barrier(0);
        if (kb < kb_hi) {  // uniform
            // the row subtiles' weights first, then the token subtiles one
            // at a time (their x pieces read from LDS just before use)
            bf16x8 b[kRW][Fmt<kType>::kN];
            unsigned d[kRW];
#pragma unroll
            for (int r = 0; r < kRW; ++r) decode_w<kType>(wr_this[r], kb, g, b[r], d[r]);
            const auto token_tile = [&](int s) __attribute__((always_inline)) {
                bf16x8 a[3];
#pragma unroll
                for (int pl = 0; pl < 3; ++pl)
                    a[pl] = *reinterpret_cast<const bf16x8*>(stage_base(u) + (pl * kTW + s) * 1024 + 16 * lane);
#pragma unroll
                for (int r = 0; r < kRW; ++r) {
                    floatx4 one[1] = {acc[r][s]};
                    block_products<kType, 1>(
                        a, reinterpret_cast<const bf16x8(&)[1][Fmt<kType>::kN]>(b[r]),
                        reinterpret_cast<const unsigned(&)[1]>(d[r]), one);
                    acc[r][s] = one[0];
                }
            };
            if (live == kTW) {
#pragma unroll
                for (int s = 0; s < kTW; ++s) token_tile(s);
            } else {
#pragma unroll
                for (int s = 0; s < kTW - 1; ++s)
                    if (s < live) token_tile(s);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        load_ws(wr_this, kb + 3);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll 1
    for (int kb0 = kb_lo; kb0 < kb_hi; kb0 += kStages) {
        iteration(kb0, wr0, 0, 2);
        iteration(kb0 + 1, wr1, 1, 0);
        iteration(kb0 + 2, wr2, 2, 1);
    }
    // the copies past the end land before the workgroup's LDS is released
    __builtin_amdgcn_s_waitcnt(0);

    // lane (g, j) holds tokens 16 (s0 + s) + 4 g + q of row row0 + 16 r + j;
    // with K split, the sums go to part[z][t][row] for range_sum_kernel.  Checked:
    // sums that are not finite are left out (bit 16 r + 4 s + q of the result).
    float* const part = p.part ? p.part + static_cast<long long>(tz) * p.n * p.total_rows : nullptr;
    const auto store = [&](auto checked) __attribute__((always_inline)) {
        unsigned redo = 0;
        static_assert(kRW * kTW * 4 <= 32, "one bit per sum");
#pragma unroll
        for (int r = 0; r < kRW; ++r) {
            const int row = row0 + 16 * r + j;
            if (row >= p.total_rows) continue;
            const auto rows = [&](float* out, long long stride, bool add) __attribute__((always_inline)) {
#pragma unroll
                for (int s = 0; s < kTW; ++s)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int t = 16 * (s0 + s) + 4 * g + q;
                        if (t >= p.n) continue;
                        if (checked && !(fabsf(acc[r][s][q]) < __builtin_huge_valf())) {
                            redo |= 1u << (16 * r + 4 * s + q);
                            continue;
                        }
                        float* const o = out + static_cast<long long>(t) * stride;
                        *o = add ? *o + acc[r][s][q] : acc[r][s][q];
                    }
            };
            if (part) {
                rows(part + row, p.total_rows, false);
                continue;
            }
            const RowSeg rs = row_seg(p, row);
            rows(rs.out + rs.row, rs.stride, p.add);
        }
        return redo;
    };
    // Zero times every sum is zero unless one is not finite: one branch for the
    // wave (F16, 11264 x 2048, 100 tokens 42.9 -> 43.4 us; a branch before each
    // store was 1-4 % of most shapes).
    floatx4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < kRW; ++r)
#pragma unroll
        for (int s = 0; s < kTW; ++s)
#pragma unroll
            for (int q = 0; q < 4; ++q) zero[q] = fmaf(0.f, acc[r][s][q], zero[q]);
    if (__builtin_expect(!__any(!(zero[0] + zero[1] + zero[2] + zero[3] == 0.f)), 1)) {
        store(std::false_type{});
        return;
    }
    const unsigned redo = store(std::true_type{});
#pragma unroll 1
    for (int i = 0; i < 16 * kRW; ++i) {
        const bool mine = redo >> i & 1;
        if (!__any(mine)) continue;
        const int row = min(row0 + 16 * (i >> 4) + j, p.total_rows - 1), t = 16 * (s0 + (i >> 2 & 3)) + 4 * g + (i & 3);
        const RowSeg rs = row_seg(p, row);
        const float sum = taken_again<kType>(0.f, mine, rs.w + static_cast<long long>(rs.row) * p.row_bytes, t, 32 * kb_lo,
                                             32 * kb_hi, p.xs, n_blk);
        if (!mine) continue;
        if (part) {
            part[static_cast<long long>(t) * p.total_rows + row] = sum;
        } else {
            float* const o = rs.out + rs.row + t * rs.stride;
            *o = p.add ? *o + sum : sum;
        }
    }
}

// out[t][row] (+)= sum over the K splits z, in order, of part[z][t][row]:
// one thread per (t, row).
__global__ __launch_bounds__(kThreads) void range_sum_kernel(const ProductParams p)
{
    const long long id = static_cast<long long>(blockIdx.x) * kThreads + threadIdx.x;
    if (id >= static_cast<long long>(p.n) * p.total_rows) return;
    const int t = static_cast<int>(id / p.total_rows), row = static_cast<int>(id % p.total_rows);
    const long long plane = static_cast<long long>(p.n) * p.total_rows;
    float sum = p.part[id];
    for (int z = 1; z < p.k_splits; ++z) sum += p.part[z * plane + id];
    const RowSeg rs = row_seg(p, row);
    float* const o = rs.out + rs.row + static_cast<long long>(t) * rs.stride;
    *o = p.add ? *o + sum : sum;
}

// Row subtiles per workgroup that the registers hold: a direct workgroup's raw
// weights, a resident one's decoded weights (4 registers per block, piece and
// subtile).
constexpr int direct_rows(int type) { return type == kQ6_K ? 2 : kMaxRows; }
constexpr int resident_rows(int type) { return type == kF32 ? 1 : type == kF16 || type == kQ6_K ? 2 : kMaxRows; }

template <int kType, int kR, int kDepth, int kShare>
hipError_t launch_direct_depth(const ProductParams& p, hipStream_t s)
{
    const dim3 grid(static_cast<unsigned>(p.row_groups), static_cast<unsigned>(p.n_tiles)), block(kWaves * 64);
    if (p.planes)
        hipLaunchKernelGGL((direct_product_kernel<kType, kR, kXPlanes, kDepth, kShare>), grid, block, 0, s, p);
    else if (p.norm_w)
        hipLaunchKernelGGL((direct_product_kernel<kType, kR, kXNormRows, kDepth, kShare>), grid, block, 0, s, p);
    else
        hipLaunchKernelGGL((direct_product_kernel<kType, kR, kXRows, kDepth, kShare>), grid, block, 0, s, p);
    return hipGetLastError();
}

// Blocks in flight per wave: all of 2048 columns with one row subtile (fewer
// where the row has fewer: a load past the end is made, not used), else four,
// which is what the registers hold beside three subtiles.
template <int kType, int kR, int kShare>
hipError_t launch_direct_share(const ProductParams& p, hipStream_t s)
{
    if constexpr (kR == 1) {
        const int groups = (p.cols / 32 + kShare * kWaves - 1) / (kShare * kWaves);
        if constexpr (kShare == 4)
            return launch_direct_depth<kType, 1, 2, 4>(p, s);
        else if constexpr (kShare == 2)
            return groups <= 1   ? launch_direct_depth<kType, 1, 1, 2>(p, s)
                   : groups <= 2 ? launch_direct_depth<kType, 1, 2, 2>(p, s)
                                 : launch_direct_depth<kType, 1, 4, 2>(p, s);
        else
            return groups <= 2   ? launch_direct_depth<kType, 1, 2, 1>(p, s)
                   : groups <= 4 ? launch_direct_depth<kType, 1, 4, 1>(p, s)
                                 : launch_direct_depth<kType, 1, 8, 1>(p, s);
    } else {
        return launch_direct_depth<kType, kR, kShare == 1 ? 4 : 2, kShare>(p, s);
    }
}

template <int kType, int kR>
hipError_t launch_direct(const ProductParams& p, hipStream_t s)
{
    if constexpr (kR <= direct_rows(kType)) {
        if constexpr (kR == 1)
            if (p.x_share == 4) return launch_direct_share<kType, kR, 4>(p, s);
        return p.x_share == 2 ? launch_direct_share<kType, kR, 2>(p, s) : launch_direct_share<kType, kR, 1>(p, s);
    } else {
        return hipErrorInvalidValue;
    }
}

template <int kType, int kR>
hipError_t launch_resident(const ProductParams& p, hipStream_t s)
{
    if constexpr (kR <= resident_rows(kType)) {
        const dim3 grid(static_cast<unsigned>(p.row_groups * p.k_splits * p.shares)), block(kWaves * 64);
        if (p.blk_per_split <= 4 * kWaves)
            hipLaunchKernelGGL((resident_product_kernel<kType, kR, 4>), grid, block, 0, s, p);
        else
            hipLaunchKernelGGL((resident_product_kernel<kType, kR, kMaxSlice>), grid, block, 0, s, p);
        return hipGetLastError();
    } else {
        return hipErrorInvalidValue;
    }
}

template <int kType, int kR>
hipError_t launch_tiled(const ProductParams& p, hipStream_t s)
{
    if constexpr (kType == kQ6_K) {
        return hipErrorInvalidValue;
    } else {
        const dim3 grid(static_cast<unsigned>(p.row_groups), static_cast<unsigned>(p.n_tiles / kTW),
                        static_cast<unsigned>(p.k_splits));
        hipLaunchKernelGGL((tiled_product_kernel<kType, kR>), grid, dim3(kTileThreads), 0, s, p);
        return hipGetLastError();
    }
}

template <int kType>
hipError_t launch_typed(const ProductParams& p, hipStream_t s)
{
    const int r = p.rows_per_group;
    if (p.kind == kProductDirect)
        return r == 1   ? launch_direct<kType, 1>(p, s)
               : r == 2 ? launch_direct<kType, 2>(p, s)
                        : launch_direct<kType, 3>(p, s);
    const hipError_t err = p.kind == kProductTiled ? (r == 1 ? launch_tiled<kType, 1>(p, s) : launch_tiled<kType, 2>(p, s))
                           : r == 1                ? launch_resident<kType, 1>(p, s)
                           : r == 2                ? launch_resident<kType, 2>(p, s)
                                                   : launch_resident<kType, 3>(p, s);
    if (err != hipSuccess || !p.part || p.defer_reduce) return err;
    const long long n = static_cast<long long>(p.n) * p.total_rows;
    hipLaunchKernelGGL(range_sum_kernel, dim3(static_cast<unsigned>((n + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                       s, p);
    return hipGetLastError();
}

}  // namespace

namespace {

// K cut into `splits` ranges of an even number of blocks.
void cut_k(int splits, ProductParams* p)
{
    const int n_blk = p->cols / 32;
    p->blk_per_split = (n_blk / 2 + splits - 1) / splits * 2;
    p->k_splits = (n_blk + p->blk_per_split - 1) / p->blk_per_split;
}

void plan_resident(int type, int n_cu, int opt_rows, int opt_tiles, int opt_k, ProductParams* p)
{
    const int n_blk = p->cols / 32, sub = (p->total_rows + 15) / 16, tiles = p->n_tiles;
    const int splits = std::max((n_blk + kRangeBlocks - 1) / kRangeBlocks, std::min(opt_k, n_blk / 2));
    p->kind = kProductResident;
    // The rows per workgroup and the shares of the token tiles with the
    // least estimated time, in microseconds: per round of workgroups, the
    // weights (3 + 1.5 per row subtile) and each token tile (1.6 to load
    // its planes, 0.17 per row subtile not hidden behind that).  A round that
    // leaves CUs idle takes as long as a full one: each of its workgroups is bound
    // by its own CU's way to the planes.
    double best = 0;
    const int most = resident_rows(type);
    for (int r = 1; r <= most; ++r) {
        if (opt_rows > 0 && r != std::min(opt_rows, most)) continue;
        const long long groups = static_cast<long long>((sub + r - 1) / r) * splits;
        for (int shares = 1; shares <= (opt_tiles > 0 ? tiles : std::min(tiles, 8)); ++shares) {
            const int each = (tiles + shares - 1) / shares;
            if (opt_tiles > 0 && each > opt_tiles) continue;
            const double rounds = static_cast<double>((groups * shares + n_cu - 1) / n_cu);
            const double cost = rounds * (3.0 + 1.5 * r + each * (1.6 + 0.17 * r));
            if (best == 0 || cost < best) {
                best = cost;
                p->rows_per_group = r;
                p->row_groups = (sub + r - 1) / r;
                p->shares = shares;
            }
        }
    }
    cut_k(splits, p);
}

void plan_tiled(int n_cu, int opt_rows, int opt_k, ProductParams* p)
{
    const int n_blk = p->cols / 32;
    p->kind = kProductTiled;
    p->n_tiles = (p->n + 16 * kTW - 1) / (16 * kTW) * kTW;
    // Two row subtiles per wave where that gives half the CUs a
    // workgroup; K cut until the grid holds about 2.5 workgroups per CU,
    // ranges of at least 8 blocks.
    const auto groups = [&](int r) { return (p->total_rows + 64LL * r - 1) / (64LL * r) * (p->n_tiles / kTW); };
    int r = 2 * groups(2) >= n_cu ? 2 : 1;
    const long long target = 5LL * n_cu / 2;
    int splits = static_cast<int>(std::min<long long>((target + groups(r) - 1) / groups(r), n_blk / 8));
    if (opt_k > 0) splits = std::min(opt_k, n_blk / 2);
    if (opt_rows > 0) r = std::min(opt_rows, 2);  // (the ranges stay the shape's)
    p->rows_per_group = r;
    p->row_groups = (p->total_rows + 64 * r - 1) / (64 * r);
    cut_k(std::max(1, splits), p);
}

}  // namespace

// Fitted to both kernels' times at 992 shapes (plan_product), within 6 %.
// Resident: per round of workgroups the weights of a row subtile (2.6 at 2048
// columns) and each token tile, whose planes and products overlap in part; a wave
// loads a slice of 4 or 8 blocks of it, used or not.  Tiled: a block of a
// workgroup takes 0.23 where its CU has no other, else the CU's workgroups share
// its matrix cores, vector units and LDS.  Several ranges: the launch that adds
// their sums, a step per range, and its bytes.
double product_us(int type, int n_cu, const ProductParams& p)
{
    const double sums = p.k_splits > 1 ? 1.85 + 0.26 * p.k_splits + 1e-6 * p.n * p.total_rows * (p.k_splits + 1.0) : 0;
    const auto rounds = [&](long long groups) { return static_cast<double>((groups + n_cu - 1) / n_cu); };
    const int r = p.rows_per_group;
    if (p.kind == kProductTiled) {
        const double block = type == kF32 ? 0.372 * r : type == kF16 ? 0.257 * r : 0.05 + 0.184 * r;
        const double per_cu = rounds(static_cast<long long>(p.row_groups) * (p.n_tiles / kTW) * p.k_splits);
        return sums + 3.7 + 0.33 * per_cu + p.blk_per_split * std::max(0.23, per_cu * block);
    }
    const int each = (p.n_tiles + p.shares - 1) / p.shares;
    const double slice = p.blk_per_split <= 4 * kWaves ? 0.5 : 1.0;
    const double tile = (0.9 + (type == kF32 ? 1.18 : type == kF16 || type == kQ6_K ? 0.54 : 0.4) * r) * slice;
    return sums + rounds(static_cast<long long>(p.row_groups) * p.k_splits * p.shares) *
                      (1.7 + 2.6 * r * p.blk_per_split / kRangeBlocks + each * tile);
}

void plan_product(int type, int n_cu, int opt_rows, int opt_tiles, int opt_k, ProductParams* p)
{
    const int n_blk = p->cols / 32, sub = (p->total_rows + 15) / 16, tiles = (p->n + 15) / 16;
    p->n_tiles = tiles;
    p->k_splits = 1;
    p->blk_per_split = n_blk;
    p->x_share = 1;
    p->shares = 1;
    // Up to 16 tokens, or where the row subtiles and token tiles fit the CUs
    // in one round: no launch for the planes.  As many rows per workgroup as
    // bring the grid into one round (11264 x 2048, 3 tokens, 1 / 2 / 3
    // subtiles: Q4_0 17.9 / 17.6 / 12.2 us); past that two, whose registers let
    // a CU hold two workgroups (32000 rows 28.2 / 23.2 / 29.5).
    if (tiles == 1 || static_cast<long long>(sub) * tiles <= n_cu) {
        p->kind = kProductDirect;
        int r = 1;
        while (r < direct_rows(type) && static_cast<long long>((sub + r - 1) / r) * tiles > n_cu) ++r;
        if (static_cast<long long>((sub + r - 1) / r) * tiles > n_cu) r = 2;
        // Up to 8 tokens two blocks share an x operand, up to 4 tokens four:
        // with one row subtile (the accumulators of four for three subtiles
        // leave no registers for loads: F32, 11264 x 2048, 3 tokens 28 against
        // 18 us; Q4_0, 32000 rows, 26 against 22) and more than one group of
        // them per wave (900 x 1024, F16 4.5 against 4.3 us).  The choice is the
        // shape's: it sets the order of the sums, so the row option, which
        // does not, leaves four blocks their one subtile.
        p->x_share = p->n <= 4 && r == 1 && n_blk > 4 * kWaves ? 4 : p->n <= 8 ? 2 : 1;
        if (opt_rows > 0 && p->x_share < 4) r = std::min(opt_rows, direct_rows(type));
        p->rows_per_group = r;
        p->row_groups = (sub + r - 1) / r;
        return;
    }
    // Resident or tiled by the shape's estimates (the options change no kind).
    // Of 992 shapes measured in both kernels (F16, F32, Q4_0, Q8_0; 512 to 32000
    // rows, 256 to 8192 columns, 65 to 1000 tokens) this takes the slower one by
    // more than 5 % in 20 (lines of rows and tokens fitted to 2048 columns: 178),
    // 0.3 % on average (2.5 %).  Us, resident / tiled: F16 8192 x 2048, 81 tokens
    // 25.4 / 34.9, 11264 x 2048, 128 tokens 53.1 / 45.8, 8192 x 1024, 128 18.7 /
    // 26.4; F32 4096 x 2048, 160 31.6 / 35.8, 2048 x 5632, 65 38.3 / 33.9; Q8_0
    // 4096 x 5632, 128 46.1 / 40.6, 2048 x 4096, 256 34.3 / 35.1; F32 3000 x 256, 512
    // tokens 34.8 / 17.2.
    // Up to one column of 64 tokens the resident product stays, for its shorter
    // chains of sums (F16 11264 x 2048, 56 tokens: 1.00e-7 off fp64 in 33.1 us,
    // tiled 1.07e-7 in 28.9).
    // Neither a pair's epilogue nor Q6_K's decoding is in the tiled kernel.
    ProductParams tiled = *p;
    plan_resident(type, n_cu, 0, 0, 0, p);
    if (!p->pair && type != kQ6_K && p->n > 16 * kTW) {
        plan_tiled(n_cu, 0, 0, &tiled);
        if (product_us(type, n_cu, tiled) < product_us(type, n_cu, *p)) {
            *p = tiled;
            if (opt_rows > 0 || opt_k > 0) plan_tiled(n_cu, opt_rows, opt_k, p);
            return;
        }
    }
    if (opt_rows > 0 || opt_tiles > 0 || opt_k > 0) plan_resident(type, n_cu, opt_rows, opt_tiles, opt_k, p);
}

size_t product_planes_bytes(int n, int cols)
{
    return static_cast<size_t>((n + 16 * kTW - 1) / (16 * kTW) * (16 * kTW)) * static_cast<size_t>(cols) * 6;
}

size_t product_part_bytes(int n, int total_rows, int k_splits)
{
    return static_cast<size_t>(n) * static_cast<size_t>(total_rows) * static_cast<size_t>(k_splits) * sizeof(float);
}

namespace {
bool a16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }
}  // namespace

hipError_t load_product_code()
{
    hipFuncAttributes a;
    return hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&norm_split_rows_kernel));
}

hipError_t launch_split_rows(const float* x, long long x_stride, int n, int cols, bool gated, unsigned char* xs,
                             hipStream_t s)
{
    if (n < 1 || cols < 32 || cols % 32 != 0 || x_stride % 4 != 0 || !a16(x) || !a16(xs)) return hipErrorInvalidValue;
    const int n_tiles = (n + 15) / 16, n_blk = cols / 32;
    const long long threads = static_cast<long long>(n_blk) * n_tiles * 64;
    const dim3 grid(static_cast<unsigned>((threads + kThreads - 1) / kThreads));
    if (gated)
        hipLaunchKernelGGL((split_rows_kernel<true>), grid, dim3(kThreads), 0, s, x, x_stride, n, n_tiles, n_blk, xs);
    else
        hipLaunchKernelGGL((split_rows_kernel<false>), grid, dim3(kThreads), 0, s, x, x_stride, n, n_tiles, n_blk, xs);
    return hipGetLastError();
}

hipError_t launch_norm_split_rows(float* x, const float* part, int k_splits, int n, int cols, const float* w, float eps,
                                  unsigned char* xs, hipStream_t s)
{
    if (n < 1 || cols < 32 || cols % 32 != 0 || k_splits < 0 || !a16(x) || !a16(w) || !a16(xs) ||
        (k_splits > 0 && (!part || !a16(part))))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(norm_split_rows_kernel, dim3(n), dim3(kThreads), 0, s, x, part, k_splits,
                       static_cast<long long>(n) * cols, w, cols, eps, xs);
    return hipGetLastError();
}

hipError_t launch_product(int type, const ProductParams& p, hipStream_t s)
{
    const int n_blk = p.cols / 32, sub = (p.total_rows + 15) / 16, tiles = (p.n + 15) / 16, r = p.rows_per_group;
    if (p.n < 1 || p.total_rows < 1 || p.cols < 64 || p.cols % 64 != 0 || (type == kQ6_K && p.cols % 256 != 0) ||
        p.n_seg < 1 || p.n_seg > kGemvMaxSeg || p.row_bytes != static_cast<long long>(weight_row_bytes(type, p.cols)) ||
        r < 1 || p.k_splits < 1 || p.blk_per_split < 2 || p.blk_per_split % 2 != 0 ||
        static_cast<long long>(p.k_splits - 1) * p.blk_per_split >= n_blk ||
        static_cast<long long>(p.k_splits) * p.blk_per_split < n_blk || (p.k_splits > 1) != (p.part != nullptr) ||
        p.shares < 1)
        return hipErrorInvalidValue;
    if (p.pair && (p.n_seg != 2 || p.seg[0].rows != p.seg[1].rows || p.seg[0].rows % 32 != 0 || !p.hs ||
                   p.kind == kProductTiled || p.k_splits > 1 || p.add))
        return hipErrorInvalidValue;
    const bool planes = p.planes || p.kind != kProductDirect;
    if (planes ? !p.xs || !a16(p.xs) || p.norm_w : !p.x || !a16(p.x) || p.x_stride % 4 != 0) return hipErrorInvalidValue;
    if (p.norm_w && (!a16(p.norm_w) || p.cols > kProductMaxNorm)) return hipErrorInvalidValue;
    bool fits = false;
    switch (p.kind) {
    case kProductDirect:
        fits = (p.x_share == 1 || (p.x_share == 2 && p.n <= 8) || (p.x_share == 4 && p.n <= 4 && r == 1)) &&
               r <= direct_rows(type) && p.row_groups == (sub + r - 1) / r && p.n_tiles == tiles && p.k_splits == 1;
        break;
    case kProductResident:
        fits = r <= resident_rows(type) && p.row_groups == (sub + r - 1) / r && p.n_tiles == tiles &&
               p.shares <= tiles && p.blk_per_split <= kRangeBlocks;
        break;
    case kProductTiled:
        fits = r <= 2 && p.row_groups == (p.total_rows + 64 * r - 1) / (64 * r) &&
               p.n_tiles == (p.n + 16 * kTW - 1) / (16 * kTW) * kTW;
        break;
    }
    if (!fits) return hipErrorInvalidValue;
    int rows = 0;
    for (int i = 0; i < p.n_seg; ++i) {
        const uintptr_t align = type == kF32 || type == kF16 ? 16 : type == kQ6_K ? 2 : 4;
        if (p.seg[i].rows < 1 || reinterpret_cast<uintptr_t>(p.seg[i].w) % align != 0 || (!p.seg[i].out && !p.pair))
            return hipErrorInvalidValue;
        rows += p.seg[i].rows;
    }
    if (rows != p.total_rows) return hipErrorInvalidValue;
    switch (type) {
    case kF32: return launch_typed<kF32>(p, s);
    case kF16: return launch_typed<kF16>(p, s);
    case kQ8_0: return launch_typed<kQ8_0>(p, s);
    case kQ4_0: return launch_typed<kQ4_0>(p, s);
    case kQ6_K: return launch_typed<kQ6_K>(p, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace tla
