// Causal prefill attention for gfx950: products on the bf16 matrix cores
// with fp32 accuracy, fp32 accumulation.
//
// Reference semantics: the prompt is fed token by token (src/generate.cpp:
// 56-59); for the attention block that is, for t = 0..n_tok-1 at position
// P = pos0 + t: rope(q_t, k_t, P) (src/ops.cpp:1223-1281), append k_t,v_t at
// P (src/ops.cpp:1370-1371), then attention of q_t over cache positions
// 0..P (src/ops.cpp:1377-1511).  Because token t only ever sees keys
// 0..P, the whole prompt is one causal (lower-triangular) attention over
// the cache after all appends -- which is what these kernels compute.
//
// Exact splitting.  Every fp32 operand (q, k, v and the probabilities P) is
// the sum of three bf16 pieces, x = x0 + x1 + x2 (bf16_split.h); a product
// of two pieces is exact in fp32, so a . b is computed as the six piece
// products down to 2^-16 of a b (a0b0, a0b1, a1b0, a0b2, a1b1, a2b0) on
// v_mfma_f32_32x32x16_bf16, whose rate is 16 times that of fp32 MFMA.  The
// three left out are below 2^-24 of a b: the reference's accuracy, not its
// bits.
//
// prefill_append_kernel: one workgroup per (layer, kv head, 32-key tile):
//   rotates the prompt's k rows (when asked) and writes k and v rows to the
//   cache, bit-exact with the reference's append, and writes every key of
//   the tile (earlier ones read back from the cache) as K and V planes in
//   the layout the attention kernel's MFMA operands are read in.
//
// prefill_attention_kernel: one workgroup = 4 waves = 4 q heads of one kv
//   head, over one tile of 32 query tokens.  Each wave:
//     S^T[32 keys][32 queries] = K[32][64] . Q^T[64][32]   24 MFMAs
//     causal mask, online softmax per query row (the running max moves
//       only when it grows by more than 2^8, so most tiles skip rescaling O)
//     O^T[64 d][32 queries]   += V^T[64][32] . P^T[32][32] 24 MFMAs
//   The S accumulator layout is the B operand of the P.V product as is (K
//   rows are stored permuted, kperm), so P never leaves registers.  Q
//   (rotated in registers with the host-built table) is split once.  Tiles
//   come from the planes into LDS with direct global-to-LDS loads.
//
// prefill_short_kernel: both in one launch, for launches of about one
//   workgroup per CU (short prompts, and few tokens after a long context).
//
// Scheduling: key/value tiles of one (layer, kv head) are read by all its
//   query tiles and q heads, so those workgroups are placed on one XCD
//   (workgroup i runs on XCD i % 8) to share that XCD's L2, and each XCD
//   starts the query tiles with the most key tiles first, across all of its
//   (layer, kv head) pairs, so the last workgroups to start are short ones.
#include <algorithm>

#include "prefill.h"
#include "bf16_split.h"
#include "lane_math.h"
#include "rope_math.h"
#include "tla_internal.h"

namespace tla {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
typedef float floatx8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kQTile = 32;
constexpr int kKTile = 32;
constexpr int kWavesP = 4;
constexpr int kXcds = 8;

// Planes of one 32-key tile, K then V, three bf16 planes each, each plane
// in the order the attention kernel's waves read it as an MFMA operand
// (1 KiB per read, lane l at byte 16 l):
//   K plane: byte 512 c + 16 i = dims 8c .. 8c+7 of key kperm(i);
//   V plane: byte 2048 dt + 1024 s + 512 h + 16 i = keys 16s + 8h .. +7
//            of dim 2i + dt.
constexpr int kPlane = kKTile * kHeadDim * 2;  // bytes of one bf16 plane of a tile
constexpr int kHalfTile = 3 * kPlane;          // K (or V) of a tile: 12 KiB
constexpr int kTileBytes = 2 * kHalfTile;

// Row i of a K tile holds key kperm(i) of the tile (bits 2 and 3 of the
// index swapped; its own inverse).  Score register r of lane 32 h + j then
// holds key 16 (r / 8) + 8 h + r % 8 for query j, which is what lane 32 h +
// j supplies as the B operand (P^T) of the P.V product at k step r / 8,
// element r % 8.
__device__ __forceinline__ int kperm(int i)
{
    return (i & ~12) | ((i & 4) << 1) | ((i & 8) >> 1);
}

// The three planes of eight fp32 values.
__device__ __forceinline__ void split8(floatx8 v, bf16x8 (&o)[3])
{
    split3x8(v, o[0], o[1], o[2]);
}

// One workgroup per (layer, kv head, 32-key tile) of positions 0 ..
// pos0+n_tok-1, tile fastest.  Keys from pos0 on are the prompt's; earlier
// keys are read from the cache; keys past the last position are zeros.
//   K: thread t holds dims 8c .. 8c+7 of key kk (c = t / 32, kk = t % 32);
//   V: thread t holds dim d of keys 8kg .. 8kg+7 (kg = t / 64, d = 2 (t % 32)
//      + (t / 32) % 2), so each of its plane pieces is one 16-byte store and
//      each wave's cache store instruction one 256-byte key row.
__global__ __launch_bounds__(256) void prefill_append_kernel(const PrefillParams p)
{
    const int tile = (int)(blockIdx.x % (unsigned)p.n_ptiles);
    const int pair = (int)(blockIdx.x / (unsigned)p.n_ptiles);  // lb * n_head_kv + kvh
    const int kvh = pair % p.n_head_kv, lb = pair / p.n_head_kv;
    const int n_pos = p.pos0 + p.n_tok;
    const int kv_dim = p.n_head_kv * kHeadDim;
    const long long layer_off = (long long)(p.layer0 + lb) * p.layer_stride + (long long)kvh * kHeadDim;
    float* const kc = p.kc + layer_off;
    float* const vc = p.vc + layer_off;
    unsigned char* const planes = p.kvp + ((long long)pair * p.n_ptiles + tile) * kTileBytes;

    // Every load is issued before the first store (one memory round trip).
    const int kk = threadIdx.x & 31, c = threadIdx.x >> 5;
    const int kkey = tile * kKTile + kk;
    const bool k_new = kkey >= p.pos0 && kkey < n_pos;
    float* const kdst = kc + (long long)kkey * kv_dim + 8 * c;
    float4 ka = make_float4(0.f, 0.f, 0.f, 0.f), kb = ka, ca = ka, cb = ka;
    if (k_new) {
        const float* src = p.k + (((long long)lb * p.n_tok + (kkey - p.pos0)) * p.n_head_kv + kvh) * kHeadDim + 8 * c;
        const float* tab = reinterpret_cast<const float*>(p.rope + (long long)kkey * kPairs) + 8 * c;
        ka = ldg4(src);
        kb = ldg4(src + 4);
        ca = ldg4(tab);
        cb = ldg4(tab + 4);
    } else if (kkey < n_pos) {
        ka = ldg4(kdst);
        kb = ldg4(kdst + 4);
    }
    const int kg = threadIdx.x >> 6, d = 2 * (threadIdx.x & 31) + ((threadIdx.x >> 5) & 1);
    floatx8 vx;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int key = tile * kKTile + 8 * kg + e;
        float val = 0.f;
        if (key >= p.pos0 && key < n_pos)
            val = p.v[(((long long)lb * p.n_tok + (key - p.pos0)) * p.n_head_kv + kvh) * kHeadDim + d];
        else if (key < n_pos)
            val = vc[(long long)key * kv_dim + d];
        vx[e] = val;
    }

    if (k_new) {
        if (p.rotate) {
            ka = rotate4(ka, ca);
            kb = rotate4(kb, cb);
        }
        stg4(kdst, ka);
        stg4(kdst + 4, kb);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int key = tile * kKTile + 8 * kg + e;
        if (key >= p.pos0 && key < n_pos) vc[(long long)key * kv_dim + d] = vx[e];
    }
    bf16x8 pc[3];
    split8(floatx8{ka.x, ka.y, ka.z, ka.w, kb.x, kb.y, kb.z, kb.w}, pc);
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8*>(planes + q * kPlane + 512 * c + 16 * kperm(kk)) = pc[q];
    split8(vx, pc);
#pragma unroll
    for (int q = 0; q < 3; ++q)
        *reinterpret_cast<bf16x8*>(planes + kHalfTile + q * kPlane + 2048 * (d & 1) + 1024 * (kg >> 1) +
                                   512 * (kg & 1) + 16 * (d >> 1)) = pc[q];
}

struct PrefillGrid {
    int n_qt;     // query tiles
    int n_hg;     // head groups of 4 waves per kv head
    int n_pairs;  // n_lb * n_head_kv
    // Pair groups: 8 (pair i on XCD i % 8) for at least 8 pairs, else 1 (all
    // query tiles over the whole GPU: one layer has 4 pairs).
    int n_grp, grp_shift;  // n_grp = 1 << grp_shift
    int per_grp;           // workgroup slots per group: ceil(n_pairs / n_grp) * n_hg * n_qt
    // Quotients by the launch's divisors as multiply-highs: q = mulhi(n, m)
    // with m = ceil(2^32 / d), exact for n * d < 2^32 (checked at launch); a
    // divisor of 1 has m = 0 and takes q = n.  The groups below
    // n_pairs % n_grp (all when it is 0) hold ceil(n_pairs / n_grp) pairs,
    // the others one fewer.
    unsigned m_rank_big, m_rank_small;  // pairs per group x n_hg
    unsigned m_hg;                      // n_hg
    unsigned m_kv;                      // n_head_kv
    unsigned m_ch;                      // n_ch
    int n_ch;       // most workgroups that share a query tile
    float* part;    // their states
    int* counters;  // their arrivals, zero between launches
};

// The rotation of rotate4 with fused multiply-adds: 8 operations per float4
// instead of 12, each output within an ulp or so of the separately rounded
// form.  For operands that are not stored (q).
__device__ __forceinline__ float4 rotate4_fma(float4 x, float4 cs)
{
    return make_float4(__builtin_fmaf(x.x, cs.x, -(x.y * cs.y)), __builtin_fmaf(x.x, cs.y, x.y * cs.x),
                       __builtin_fmaf(x.z, cs.z, -(x.w * cs.w)), __builtin_fmaf(x.z, cs.w, x.w * cs.z));
}

__device__ __forceinline__ unsigned div_magic(unsigned n, unsigned m)
{
    return m ? __umulhi(n, m) : n;
}

constexpr float kRescaleSlack = 8.f;  // log2 units

// Products of two split operands on v_mfma_f32_32x32x16_bf16: a . b for
// a = a0 + a1 + a2 and b = b0 + b1 + b2, the six piece products down to
// 2^-16 of a b, smallest first.
__device__ __forceinline__ floatx16 split_products(const bf16x8 (&a)[3], const bf16x8 (&b)[3], floatx16 c)
{
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], c, 0, 0, 0);
    return c;
}

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __attribute__((address_space(1))) void* global_ptr;

// Copies half a tile (12 KiB, K or V) from the planes into LDS: 12 chunks
// of 1 KiB over kWaves waves, each one direct global-to-LDS load of 16
// bytes per lane (lane l's bytes land at byte 16 l of the chunk).
template <int kWaves>
__device__ __forceinline__ void copy_half(const unsigned char* src, unsigned char* dst, int wave, int lane)
{
    constexpr int kPer = 12 / kWaves;
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
        const int chunk = kPer * wave + c;
        __builtin_amdgcn_global_load_lds((global_ptr)(src + 1024 * chunk + 16 * lane), (lds_ptr)(dst + 1024 * chunk),
                                         16, 0, 0);
    }
}

typedef float4 QueryRow[kHeadDim / 4];
constexpr int kRowBytes = sizeof(QueryRow);

constexpr int kXchFloats = 34 * 64;  // a wave's softmax state: max, sum, O
constexpr int kXchBytes = 4 * kXchFloats;
static_assert(kXchBytes == kPrefillStateBytes, "the engine sizes the workspace");
constexpr int kDeviceScope = 16;             // cache-policy bit SC1: device scope
constexpr int kRawBufferWord3 = 0x00020000;  // untyped 32-bit buffer (gfx9 family)

// One wave's share of the work: a q head over 32 query tokens, its Q operand
// and running softmax state.
struct WaveState {
    bf16x8 qp[4][3];
    floatx16 o0 = {}, o1 = {};
    float m_run = -INFINITY;
    float l_run = 0.f;

    // Q^T operand: lane 32 h + j holds, for k step s, dims 16s + 8h .. +7 of
    // query j, times scale * log2(e), as three bf16 planes.  q4(c), tab4(c):
    // float4 c of the query's row and of its (cos, sin) row.
    template <class Q, class T>
    __device__ __forceinline__ void load_q(Q&& q4, T&& tab4, int half, float scale_log2, int rotate)
    {
        // All sixteen loads are issued before any is used.
        float4 qv[8], cs[8];
#pragma unroll
        for (int f = 0; f < 8; ++f) {
            qv[f] = q4(4 * (f >> 1) + 2 * half + (f & 1));
            cs[f] = tab4(4 * (f >> 1) + 2 * half + (f & 1));  // (cos, sin) pairs of those dims
        }
        // Scaled first, then rotated with fused multiply-adds: q only enters
        // the scores, so it needs the reference's accuracy, not its bits (the
        // cache rows, which must match bit for bit, are rotated by the append
        // kernel).
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            floatx8 v;
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
                const float4 x0 = qv[2 * s + h2];
                const float4 x = make_float4(x0.x * scale_log2, x0.y * scale_log2, x0.z * scale_log2,
                                             x0.w * scale_log2);
                const float4 r = rotate ? rotate4_fma(x, cs[2 * s + h2]) : x;
                v[4 * h2 + 0] = r.x;
                v[4 * h2 + 1] = r.y;
                v[4 * h2 + 2] = r.z;
                v[4 * h2 + 3] = r.w;
            }
            split8(v, qp[s]);
        }
    }

    // S^T = K.Q^T for the tile in K buffer kb: s[r] = S[query col][key
    // 16 (r / 8) + 8 half + r % 8 of the tile].
    __device__ __forceinline__ floatx16 scores(const unsigned char* kb, int lane) const
    {
        floatx16 s = {};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            bf16x8 a[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) a[q] = *reinterpret_cast<const bf16x8*>(kb + q * kPlane + 1024 * ks + 16 * lane);
            s = split_products(a, qp[ks], s);
        }
        return s;
    }
    // Online softmax of one tile's scores (log2 units) into P, in place.
    __device__ __forceinline__ void softmax(floatx16& s, int j0, bool masked, int half, int qpos, int last_key)
    {
        if (masked) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = j0 + 16 * (r >> 3) + 8 * half + (r & 7);
                s[r] = (key <= qpos && key <= last_key) ? s[r] : -INFINITY;
            }
        }
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
        mx = max_xor32(mx);  // the other half of the keys
        // The running max only moves when some row's tile max exceeds it by
        // more than 2^8: probabilities then stay <= 256 and the sums in fp32
        // range, and most tiles skip the rescale of O.  The result is the
        // same softmax: O and l share whatever max they were scaled by.
        // A row whose keys have all been masked so far keeps m_run = -inf
        // (a workgroup's first tile can lie past some rows' positions): its
        // probabilities are 0, and nothing is rescaled.
        if (__any(mx > m_run + kRescaleSlack)) {
            const float m_new = fmaxf(m_run, mx);
            const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);  // 0 on the first tile
            m_run = m_new;
            l_run *= alpha;
            o0 *= alpha;
            o1 *= alpha;
        }
        const float m_use = m_run == -INFINITY ? 0.f : m_run;
        float lsum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = __builtin_amdgcn_exp2f(s[r] - m_use);
            lsum += s[r];
        }
        l_run += lsum;
    }
    // O^T += V^T.P^T for the tile in V buffer vb: o_dt[r] accumulates dim
    // 2 (8 (r / 4) + 4 half + r % 4) + dt of query col.  P^T at k step ks is
    // s[8 ks .. 8 ks + 7], split into planes just before its products.
    __device__ __forceinline__ void accumulate(const floatx16& s, const unsigned char* vb, int lane)
    {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            floatx8 pv;
#pragma unroll
            for (int e = 0; e < 8; ++e) pv[e] = s[8 * ks + e];
            bf16x8 pp[3];
            split8(pv, pp);
            bf16x8 a0[3], a1[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                a0[q] = *reinterpret_cast<const bf16x8*>(vb + q * kPlane + 1024 * ks + 16 * lane);
                a1[q] = *reinterpret_cast<const bf16x8*>(vb + q * kPlane + 2048 + 1024 * ks + 16 * lane);
            }
            o0 = split_products(a0, pp, o0);
            o1 = split_products(a1, pp, o1);
        }
    }

    // The output row of the lane's query (orow: 8 h floats into it).
    __device__ __forceinline__ void store(float* orow, bool ok)
    {
        l_run = sum_xor32(l_run);
        if (!ok) return;
        const float inv = 1.0f / l_run;
        // o_dt[4a+b] = O[row][16a + 8*half + 2b + dt]
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            stg4(orow + 16 * a, make_float4(o0[4 * a + 0] * inv, o1[4 * a + 0] * inv,
                                            o0[4 * a + 1] * inv, o1[4 * a + 1] * inv));
            stg4(orow + 16 * a + 4, make_float4(o0[4 * a + 2] * inv, o1[4 * a + 2] * inv,
                                                o0[4 * a + 3] * inv, o1[4 * a + 3] * inv));
        }
    }

    // The state as kXchFloats floats, lane fastest (xch: already at the lane).
    __device__ __forceinline__ void put(float* xch) const
    {
        xch[0] = m_run;
        xch[64] = l_run;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            xch[64 * (2 + i)] = o0[i];
            xch[64 * (18 + i)] = o1[i];
        }
    }
    // Both scaled to the larger max.  A side with no unmasked key (max -inf)
    // adds nothing.
    __device__ __forceinline__ void merge(const float* xch)
    {
        merge(xch[0], xch[64], [&](int i) { return xch[64 * (2 + i)]; });
    }
    template <class F>
    __device__ __forceinline__ void merge(float m_b, float l_b, F&& o_b)
    {
        const float m_new = fmaxf(m_run, m_b);
        const float fa = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new);
        const float fb = m_b == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_b - m_new);
        m_run = m_new;
        l_run = l_run * fa + l_b * fb;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            o0[i] = o0[i] * fa + o_b(i) * fb;
            o1[i] = o1[i] * fa + o_b(16 + i) * fb;
        }
    }
    // Hand-over between workgroups: device-scope accesses (they bypass what an
    // XCD's L2 may hold), as in decode.hip; eight float4 rows of O, then (max,
    // sum).  One 16-byte access of a wave covers 1 KiB.
    __device__ __forceinline__ void put_device(float* part, int lane) const
    {
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(part, 0, kXchBytes, kRawBufferWord3);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            floatx4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = i < 4 ? o0[4 * (i & 3) + e] : o1[4 * (i & 3) + e];
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uintx4, x), rs, 1024 * i + 16 * lane, 0,
                                                   kDeviceScope);
        }
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uintx2, floatx2{m_run, l_run}), rs,
                                              8192 + 8 * lane, 0, kDeviceScope);
    }
    // This wave's state = the n states at part, part + stride, ..
    __device__ __forceinline__ void merge_device(float* part, int stride, int n, int lane)
    {
        constexpr int kBatch = 3;  // states whose loads are in flight together
        m_run = -INFINITY;
        l_run = 0.f;
        o0 = floatx16{};
        o1 = floatx16{};
#pragma unroll 1
        for (int b0 = 0; b0 < n; b0 += kBatch) {
            floatx4 x[kBatch][8];
            floatx2 ml[kBatch];
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {  // a state past the last is not merged
                const auto rs = __builtin_amdgcn_make_buffer_rsrc(
                    part + (long long)min(b0 + b, n - 1) * stride, 0, kXchBytes, kRawBufferWord3);
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    x[b][i] = __builtin_bit_cast(
                        floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, 1024 * i + 16 * lane, 0, kDeviceScope));
                ml[b] = __builtin_bit_cast(
                    floatx2, __builtin_amdgcn_raw_buffer_load_b64(rs, 8192 + 8 * lane, 0, kDeviceScope));
            }
#pragma unroll
            for (int b = 0; b < kBatch; ++b)
                if (b0 + b < n) merge(ml[b][0], ml[b][1], [&](int i) { return x[b][i >> 2][i & 3]; });
        }
    }
};

// Counts this workgroup in after its device-scope stores are acknowledged;
// true for the last of n, which also returns the counter to zero.  All
// threads of the workgroup call it.
__device__ __forceinline__ bool last_to_arrive(int* counter, int n, int& s_last)
{
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0)
        s_last = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
    __syncthreads();
    const bool last = s_last;
    if (last && threadIdx.x == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return last;
}

// Where the query tiles of a launch do not fill the GPU, each tile's walk over
// the keys is shared by up to g.n_ch workgroups (at least two tiles each):
// workgroup c of n takes key tiles c, c + n, .. .  They leave their softmax
// states in the workspace and the last to arrive merges them, in order
// (device-scope stores and an arrival counter, as in decode.hip).
__global__ __launch_bounds__(64 * kWavesP) __attribute__((amdgpu_waves_per_eu(3, 3))) void
prefill_attention_kernel(const PrefillParams p, const PrefillGrid g)
{
    // K and V tiles (three bf16 planes each, the planes' layout), shared by the
    // waves, double-buffered.
    constexpr int kNB = 2;
    // The first K tile has a place of its own: the other three buffers hold the
    // query rows and their (cos, sin) (40 KiB) while it arrives.  52 KiB: three
    // workgroups per CU.
    constexpr int kFirst = (kWavesP + 1) * kQTile * kRowBytes;
    static_assert(kFirst >= 3 * kHalfTile && kNB == 2, "the other buffers");
    __shared__ __align__(16) unsigned char s_buf[kFirst + kHalfTile];
    __shared__ int s_last;

    // ---- XCD-aware, heavy-first mapping of workgroups to tiles ----
    // Workgroup b runs on XCD b % 8 and XCDs start their workgroups in order
    // of b / 8.  With 8 groups, (layer, kv head) pair i belongs to XCD i % 8,
    // so all query tiles of a pair share one L2; within an XCD, query tiles
    // are handed out longest first (most key tiles) across all its pairs.
    // With one group (fewer than 8 pairs: their tiles fit every L2) the same
    // order runs over the whole GPU.
    // The quotients are multiply-highs on scalar registers: a workgroup that
    // starts beside MFMA-bound waves gets few vector issue slots, and the
    // compiler's divisions go through the vector unit.
    const int grp = blockIdx.x & (g.n_grp - 1);
    const int slot = blockIdx.x >> g.grp_shift;
    const int grp_pairs = (g.n_pairs - grp + g.n_grp - 1) >> g.grp_shift;
    const bool big = (grp_pairs << g.grp_shift) >= g.n_pairs;  // this group holds ceil(n_pairs / n_grp) pairs
    const int per_rank = grp_pairs * g.n_hg;
    if (slot >= per_rank * g.n_qt * g.n_ch) return;  // whole workgroup
    const int rank = (int)div_magic((unsigned)slot, big ? g.m_rank_big : g.m_rank_small);
    const int tile_rank = (int)div_magic((unsigned)rank, g.m_ch);
    const int qt = g.n_qt - 1 - tile_rank;
    const int chunk = rank - tile_rank * g.n_ch;
    const int rem = slot - rank * per_rank;
    const int pg = (int)div_magic((unsigned)rem, g.m_hg);
    const int pair = grp + (pg << g.grp_shift);  // (lb, kvh)
    const int hg = rem - pg * g.n_hg;
    const int lb = (int)div_magic((unsigned)pair, g.m_kv);
    const int kvh = pair - lb * p.n_head_kv;

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // scalar
    const int lane = threadIdx.x & 63;
    const int hq = hg * kWavesP + wave;
    const bool computes = hq < p.gqa;  // uniform per wave; others only copy tiles
    const int qh = kvh * p.gqa + (computes ? hq : 0);

    const int col = lane & 31;  // query row within the tile
    const int half = lane >> 5; // which 8 of each 16 dims (Q, K) / keys (P, V)
    const int i0 = qt * kQTile;
    const int qpos = p.pos0 + i0 + col;           // this row's position
    const int last_key = p.pos0 + min(i0 + kQTile - 1, p.n_tok - 1);
    const int n_kt = last_key / kKTile + 1;  // key tiles covering 0..last_key
    const int n_ch = min(g.n_ch, (n_kt + 1) / 2);
    if (chunk >= n_ch) return;  // whole workgroup
    // Tiles below (pos0 + i0 + 1) / 32 end at or before the tile's first query
    // position: no key in them is masked for any row.
    const int n_plain = min((p.pos0 + i0 + 1) / kKTile, n_kt - 1);

    const auto sk = [&](int b) { return s_buf + (b ? 0 : kFirst); };
    const auto sv = [&](int b) { return s_buf + (1 + b) * kHalfTile; };

    // The pair's tiles in the planes (tile j's K at tiles + j kTileBytes, its
    // V kHalfTile further).
    const unsigned char* const tiles = p.kvp + ((long long)lb * p.n_head_kv + kvh) * p.n_ptiles * kTileBytes;
    // Past the last tile the last one is copied again (never read).
    auto copy_k = [&](int j, int b) {
        copy_half<kWavesP>(tiles + (long long)min(j, n_kt - 1) * kTileBytes, sk(b), wave, lane);
    };
    auto copy_v = [&](int j, int b) {
        copy_half<kWavesP>(tiles + (long long)min(j, n_kt - 1) * kTileBytes + kHalfTile, sv(b), wave, lane);
    };

    // Software pipeline over the key tiles j_m = chunk + m n_ch: step m
    // computes the scores of tile j_{m+1} (MFMA) while the softmax of tile
    // j_m (VALU) runs, then P.V of tile j_m.  Tile j_m's K and V sit in
    // buffer m % kNB.  Step m copies K[j_{m+2}] and V[j_{m+1}] into the buffers
    // of K[j_m] and V[j_{m-1}] (both read in step m - 1), and waits for them
    // before the barrier that ends it.
    constexpr int kWaitCopies = 0xF70;  // vmcnt(0)
    const int n_steps = (n_kt - chunk + n_ch - 1) / n_ch;
    auto tile_of = [&](int m) { return chunk + m * n_ch; };
    copy_k(tile_of(0), 0);
    // The heads' query rows and the rows' (cos, sin), staged through LDS as in
    // prefill_short_kernel (a lane per row touches 32 lines an access).
    constexpr int kQLoads = (8 * kWavesP + 8) / kWavesP;
    float4 qx[kQLoads];
#pragma unroll
    for (int u = 0; u < kQLoads; ++u) {
        const int r4 = wave + u * kWavesP;
        const int r = min(i0 + 4 * (r4 & 7) + (lane >> 4), p.n_tok - 1);
        const int head = kvh * p.gqa + min(hg * kWavesP + (r4 >> 3), p.gqa - 1);
        const float* const src = r4 < 8 * kWavesP
                                     ? p.q + (((long long)lb * p.n_tok + r) * p.n_head + head) * kHeadDim
                                     : reinterpret_cast<const float*>(p.rope + (long long)(p.pos0 + r) * kPairs);
        qx[u] = ldg4(src + 4 * (lane & 15));
    }
    QueryRow* const s_q = reinterpret_cast<QueryRow*>(s_buf);
#pragma unroll
    for (int u = 0; u < kQLoads; ++u) {
        const int r4 = wave + u * kWavesP, r = 4 * (r4 & 7) + (lane >> 4);
        s_q[(r4 >> 3) * kQTile + r][(lane & 15) ^ (r & 15)] = qx[u];
    }
    __builtin_amdgcn_s_waitcnt(0);  // and the first K tile
    __syncthreads();
    WaveState w;
    w.load_q([&](int c) { return s_q[wave * kQTile + col][c ^ (col & 15)]; },
             [&](int c) { return s_q[kWavesP * kQTile + col][c ^ (col & 15)]; }, half, p.scale_log2, p.rotate);
    __syncthreads();  // the rows' place is free
#pragma unroll
    for (int b = 1; b < kNB; ++b) copy_k(tile_of(b), b);
#pragma unroll
    for (int b = 0; b + 1 < kNB; ++b) copy_v(tile_of(b), b);
    floatx16 s_cur = {};
    if (computes) s_cur = w.scores(sk(0), lane);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // K[j_0]'s buffer is refilled in step 0

    // The scores of tile j_m in s_this, tile j_{m+1}'s into s_next.  Two
    // steps per loop trip, the two accumulators trading roles, so that no
    // copy of the scores is needed between steps.  Only the last one or two
    // tiles reach the diagonal (masked).
    auto step = [&](int m, floatx16& s_this, floatx16& s_next) {
        const int j = tile_of(m), jn = tile_of(m + 1);
        const bool last = m + 1 == n_steps;  // uniform
        copy_k(tile_of(m + kNB), m % kNB);
        copy_v(tile_of(m + kNB - 1), (m + kNB - 1) % kNB);
        if (computes && j < n_kt) {
            if (jn < n_kt) s_next = w.scores(sk((m + 1) % kNB), lane);
            w.softmax(s_this, j * kKTile, j >= n_plain, half, qpos, last_key);
            w.accumulate(s_this, sv(m % kNB), lane);
        }
        if (!last) {
            // A bare barrier: __syncthreads' release fence would wait for
            // every copy in flight (they write LDS through the vector memory
            // path).  This step's LDS reads were used before this point.
            __builtin_amdgcn_s_waitcnt(kWaitCopies);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
    };
    floatx16 s_alt = {};
    int m = 0;
    for (; m + 1 < n_steps; m += 2) {
        step(m, s_cur, s_alt);
        step(m + 1, s_alt, s_cur);
    }
    if (m < n_steps) step(m, s_cur, s_alt);
    __builtin_amdgcn_s_waitcnt(0);  // the copies past the end land before the LDS is reused or released

    float* const orow = p.out + (((long long)lb * p.n_tok + i0 + col) * p.n_head + qh) * kHeadDim + 8 * half;
    const bool ok = i0 + col < p.n_tok;
    if (n_ch == 1) {
        if (computes) w.store(orow, ok);
        return;
    }
    // The chunks of a query tile: the last to arrive merges them, in order.
    const long long unit = ((long long)pair * g.n_hg + hg) * g.n_qt + qt;
    float* const part = g.part + (unit * g.n_ch * kWavesP + wave) * kXchFloats;  // chunk 0's
    if (computes) w.put_device(part + chunk * kWavesP * kXchFloats, lane);
    if (!last_to_arrive(g.counters + unit, n_ch, s_last)) return;
    if (computes) w.merge_device(part, kWavesP * kXchFloats, n_ch, lane);
    if (computes) w.store(orow, ok);
}

// Append and attention in one launch.  Workgroup = (32 query tokens, kStage
// key tiles of a kv head, up to four of its q heads): every thread loads its
// pieces of the tiles' K and V (the prompt's from the inputs, k rotated;
// earlier positions' from the cache), splits them and writes the planes into
// LDS (the tiles' layout above); then wave w takes q head w % heads and the
// tiles t = w / heads, w / heads + splits, .. of the stage, and the splits
// merge in LDS.  A query tile with more than kStage key tiles is shared by
// several workgroups, which leave their states in the workspace; the last to
// arrive merges them in order (the stores and the counter as in decode.hip:
// device scope, acknowledged before the arrival).
//
// Bound by latency: the launch, one round of loads, 48 MFMAs and a softmax a
// tile, a merge.  What costs beside it is the CU's address unit, which takes a
// cache line an access and cycle: query rows read a lane per row straight into
// the MFMA layout (32 lines an access, sixteen accesses a wave) made 64 tokens
// of one layer 11.9 us, staged through LDS (eight lines an access) 9.1 us.
//
// No workgroup reads a cache row that another writes: the prompt's rows are
// written, bit-exact, by the workgroups of head group 0 over the query tile
// that holds them.
struct ShortGrid {
    int n_hg;        // head groups per kv head
    int heads;       // q heads per group: 1, 2 or 4
    float* part;     // states of workgroups that share a query tile
    int* counters;   // their arrivals, zero between launches
};

template <int kStage>
constexpr int kShortWaves = kStage == 1 ? 4 : 8;

template <int kStage>
__global__ __launch_bounds__(64 * kShortWaves<kStage>) void prefill_short_kernel(const PrefillParams p,
                                                                                 const ShortGrid g)
{
    constexpr int kWaves = kShortWaves<kStage>;
    constexpr int kGroups = kWaves / 4;                  // 256 threads stage one tile
    constexpr int kPer = (kStage + kGroups - 1) / kGroups;  // tiles per thread
    __shared__ __align__(16) unsigned char s_tile[kStage][kTileBytes];
    static_assert(kStage == 1 || 4 * kXchBytes <= sizeof s_tile, "at most four waves hand a state over");
    __shared__ QueryRow s_q[5][kQTile];  // the heads' query rows, then (cos, sin)
    __shared__ int s_last;

    const int qt = blockIdx.x, chunk = blockIdx.y;
    const int i0 = qt * kQTile;
    const int last_key = p.pos0 + min(i0 + kQTile - 1, p.n_tok - 1);
    const int n_kt = last_key / kKTile + 1;
    const int t0 = chunk * kStage;
    if (t0 >= n_kt) return;  // whole workgroup
    const int n_ch = (n_kt + kStage - 1) / kStage;
    const int n_t = min(kStage, n_kt - t0);
    const int pair = (int)(blockIdx.z / (unsigned)g.n_hg), hg = (int)blockIdx.z - pair * g.n_hg;
    const int lb = (int)((unsigned)pair / (unsigned)p.n_head_kv), kvh = pair - lb * p.n_head_kv;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int split = wave / g.heads, hw = wave - split * g.heads;
    const int n_split = min(kWaves / g.heads, kStage);
    const int hq = hg * g.heads + hw;
    const bool computes = hq < p.gqa && split < n_split;  // uniform per wave; others only stage
    const int qh = kvh * p.gqa + min(hq, p.gqa - 1);
    const int col = lane & 31, half = lane >> 5;
    const int qpos = p.pos0 + i0 + col;
    const int n_plain = min((p.pos0 + i0 + 1) / kKTile, n_kt - 1);

    const int kv_dim = p.n_head_kv * kHeadDim;
    const long long layer_off = (long long)(p.layer0 + lb) * p.layer_stride + (long long)kvh * kHeadDim;
    float* const kc = p.kc + layer_off;
    float* const vc = p.vc + layer_off;
    const long long in_off = ((long long)lb * p.n_tok * p.n_head_kv + kvh) * kHeadDim;
    // Row of position `key` (clamped to the last one needed).
    const auto row = [&](const float* in, const float* cache, int key) {
        key = min(key, last_key);
        return key >= p.pos0 ? in + in_off + (long long)(key - p.pos0) * kv_dim : cache + (long long)key * kv_dim;
    };
    // The pieces a thread stages, as in prefill_append_kernel.
    const int group = threadIdx.x >> 8, piece = threadIdx.x & 255;
    const int kk = piece & 31, c = piece >> 5;
    const int kg = piece >> 6, d = 2 * (piece & 31) + ((piece >> 5) & 1);
    const auto appends = [&](int key) { return hg == 0 && key >= p.pos0 + i0 && key <= last_key; };

    // Every load before its first use.
    float4 ka[kPer], kb[kPer], ca[kPer], cb[kPer];
    floatx8 vx[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int first = (t0 + group + u * kGroups) * kKTile;
        const float* const src = row(p.k, kc, first + kk) + 8 * c;
        const float* const tab =
            reinterpret_cast<const float*>(p.rope + (long long)min(first + kk, last_key) * kPairs) + 8 * c;
        ka[u] = ldg4(src);
        kb[u] = ldg4(src + 4);
        ca[u] = ldg4(tab);
        cb[u] = ldg4(tab + 4);
#pragma unroll
        for (int e = 0; e < 8; ++e) vx[u][e] = row(p.v, vc, first + 8 * kg + e)[d];
    }
    // The heads' query rows and the rows' (cos, sin), 8 KiB each: an access of
    // a wave covers four whole rows (16 lanes each; a lane per row touches 32
    // lines an access).  Row r's float4 c is stored at c ^ (r & 15), so that
    // the reads below, a lane per row, spread over the banks.
    constexpr int kQLoads = (8 * 4 + 8) / kWaves;
    const int n_rows4 = 8 * g.heads + 8;  // groups of four rows: the heads', then (cos, sin)
    float4 qx[kQLoads];
#pragma unroll
    for (int u = 0; u < kQLoads; ++u) {
        const int r4 = min(wave + u * kWaves, n_rows4 - 1);
        const int r = min(i0 + 4 * (r4 & 7) + (lane >> 4), p.n_tok - 1);
        const int head = kvh * p.gqa + min(hg * g.heads + (r4 >> 3), p.gqa - 1);
        const float* const src = r4 < 8 * g.heads
                                     ? p.q + (((long long)lb * p.n_tok + r) * p.n_head + head) * kHeadDim
                                     : reinterpret_cast<const float*>(p.rope + (long long)(p.pos0 + r) * kPairs);
        qx[u] = ldg4(src + 4 * (lane & 15));
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int t = group + u * kGroups;
        if (t >= n_t) break;  // uniform per wave
        unsigned char* const tile = s_tile[t];
        const int key = (t0 + t) * kKTile + kk;
        if (p.rotate && key >= p.pos0) {
            ka[u] = rotate4(ka[u], ca[u]);
            kb[u] = rotate4(kb[u], cb[u]);
        }
        if (appends(key)) {
            float* const dst = kc + (long long)key * kv_dim + 8 * c;
            stg4(dst, ka[u]);
            stg4(dst + 4, kb[u]);
        }
        // keys past the last one are zeros
        const floatx8 kx = {ka[u].x, ka[u].y, ka[u].z, ka[u].w, kb[u].x, kb[u].y, kb[u].z, kb[u].w};
        bf16x8 pc[3];
        split8(key <= last_key ? kx : floatx8{}, pc);
#pragma unroll
        for (int q = 0; q < 3; ++q)
            *reinterpret_cast<bf16x8*>(tile + q * kPlane + 512 * c + 16 * kperm(kk)) = pc[q];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int vkey = (t0 + t) * kKTile + 8 * kg + e;
            if (appends(vkey)) vc[(long long)vkey * kv_dim + d] = vx[u][e];
            vx[u][e] = vkey <= last_key ? vx[u][e] : 0.f;
        }
        split8(vx[u], pc);
#pragma unroll
        for (int q = 0; q < 3; ++q)
            *reinterpret_cast<bf16x8*>(tile + kHalfTile + q * kPlane + 2048 * (d & 1) + 1024 * (kg >> 1) +
                                       512 * (kg & 1) + 16 * (d >> 1)) = pc[q];
    }
#pragma unroll
    for (int u = 0; u < kQLoads; ++u) {
        const int r4 = wave + u * kWaves, r = 4 * (r4 & 7) + (lane >> 4);
        if (r4 < n_rows4) s_q[r4 >> 3][r][(lane & 15) ^ (r & 15)] = qx[u];
    }
    __syncthreads();
    WaveState w;
    if (computes) {
        w.load_q([&](int c) { return s_q[hw][col][c ^ (col & 15)]; },
                 [&](int c) { return s_q[g.heads][col][c ^ (col & 15)]; }, half, p.scale_log2, p.rotate);
#pragma unroll 1
        for (int t = split; t < n_t; t += n_split) {
            floatx16 sc = w.scores(s_tile[t], lane);
            w.softmax(sc, (t0 + t) * kKTile, t0 + t >= n_plain, half, qpos, last_key);
            w.accumulate(sc, s_tile[t] + kHalfTile, lane);
        }
    }

    // The splits' states meet in LDS, halving: at most 4 waves hand over at a time.
    if constexpr (kStage > 1) {
        float* const xch = reinterpret_cast<float*>(s_tile) + lane;
        for (int n = n_split; n > 1; n >>= 1) {  // n_split: 2 or 4
            const int h = n >> 1;
            __syncthreads();
            if (computes && split >= h && split < n) w.put(xch + ((split - h) * g.heads + hw) * kXchFloats);
            __syncthreads();
            if (computes && split < h) w.merge(xch + (split * g.heads + hw) * kXchFloats);
        }
    }
    const bool owner = computes && split == 0;
    float* const orow = p.out + (((long long)lb * p.n_tok + i0 + col) * p.n_head + qh) * kHeadDim + 8 * half;
    const bool ok = i0 + col < p.n_tok;
    if (n_ch == 1) {
        if (owner) w.store(orow, ok);
        return;
    }
    const long long unit = (long long)blockIdx.z * gridDim.x + qt;
    float* const part = g.part + ((unit * gridDim.y) * g.heads + hw) * kXchFloats;  // chunk 0's
    const int chunk_floats = g.heads * kXchFloats;
    if (owner) w.put_device(part + (long long)chunk * chunk_floats, lane);
    if (!last_to_arrive(g.counters + unit, n_ch, s_last)) return;
    if (owner) w.merge_device(part, chunk_floats, n_ch, lane);
    if (owner) w.store(orow, ok);
}

}  // namespace

size_t prefill_planes_bytes(int n_lb, int n_head_kv, int pos0, int n_tok)
{
    const long long tiles = ((long long)pos0 + n_tok + kKTile - 1) / kKTile;
    return (size_t)n_lb * n_head_kv * tiles * kTileBytes;
}

hipError_t load_prefill_code()
{
    hipFuncAttributes a;
    return hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&prefill_append_kernel));
}

hipError_t launch_prefill_append(const PrefillParams& p, hipStream_t s)
{
    if (!p.kvp || p.n_ptiles != (p.pos0 + p.n_tok + kKTile - 1) / kKTile) return hipErrorInvalidValue;
    const long long blocks = (long long)p.n_lb * p.n_head_kv * p.n_ptiles;
    if (blocks >= (1LL << 31)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(prefill_append_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p);
    return hipGetLastError();
}

namespace {

// Compute units of the current device (cached per device).
int device_cus()
{
    static int cus[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cus[dev]) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
        cus[dev] = n;
    }
    return cus[dev];
}

hipError_t launch_attention(const PrefillParams& p, int n_ch, float* part, int* counters, hipStream_t s)
{
    PrefillGrid g;
    g.n_qt = (p.n_tok + kQTile - 1) / kQTile;
    g.n_hg = (p.gqa + kWavesP - 1) / kWavesP;
    g.n_pairs = p.n_lb * p.n_head_kv;
    g.n_grp = g.n_pairs >= kXcds ? kXcds : 1;
    g.grp_shift = g.n_grp == kXcds ? 3 : 0;
    static_assert(kXcds == 8, "grp_shift");
    g.n_ch = n_ch;
    g.part = part;
    g.counters = counters;
    g.per_grp = (g.n_pairs + g.n_grp - 1) / g.n_grp * g.n_hg * g.n_qt * g.n_ch;
    // m = ceil(2^32 / d) (0 for d <= 1); mulhi(n, m) = n / d whenever n * d < 2^32.
    auto magic = [](long long d) -> unsigned {
        return d <= 1 ? 0u : (unsigned)(((1ULL << 32) + (unsigned long long)d - 1) / (unsigned long long)d);
    };
    const long long rank_big = (long long)((g.n_pairs + g.n_grp - 1) / g.n_grp) * g.n_hg;
    const long long rank_small = (long long)(g.n_pairs / g.n_grp) * g.n_hg;
    if ((long long)g.per_grp * rank_big >= (1LL << 32) || (long long)g.n_qt * g.n_ch * g.n_ch >= (1LL << 32) ||
        (long long)rank_big * g.n_hg >= (1LL << 32) ||
        (long long)g.n_pairs * p.n_head_kv >= (1LL << 32))
        return hipErrorInvalidValue;  // quotients by multiply-high would not be exact
    g.m_rank_big = magic(rank_big);
    g.m_rank_small = magic(rank_small);
    g.m_hg = magic(g.n_hg);
    g.m_kv = magic(p.n_head_kv);
    g.m_ch = magic(g.n_ch);
    hipLaunchKernelGGL(prefill_attention_kernel, dim3(g.per_grp * g.n_grp), dim3(64 * kWavesP), 0, s, p, g);
    return hipGetLastError();
}

}  // namespace

namespace {

struct ShortShape {
    int stage;   // key tiles per workgroup
    int heads, n_hg;
    int n_qt, n_ch;
    long long z;  // (layer, kv head, head group)
};

ShortShape short_shape(int n_lb, int n_head_kv, int gqa, int pos0, int n_tok)
{
    const int n_kt = (pos0 + n_tok + kKTile - 1) / kKTile;
    ShortShape s;
    s.stage = n_kt <= 1 ? 1 : n_kt == 2 ? 2 : 4;
    s.heads = gqa >= 3 ? 4 : gqa;
    s.n_hg = (gqa + s.heads - 1) / s.heads;
    s.n_qt = (n_tok + kQTile - 1) / kQTile;
    s.n_ch = (n_kt + s.stage - 1) / s.stage;
    s.z = (long long)n_lb * n_head_kv * s.n_hg;
    return s;
}

}  // namespace

// One launch pays while its workgroups run at once, about one per CU (LDS;
// two with one key tile): every workgroup that reads a key tile splits it
// again, and with a second round the planes' two launches are as fast.
// Measured, us per call, this / the two launches: one layer of 32/4 heads,
// 32 tokens 7.6 / 12.1, 128 tokens 12.4 / 13.7, 384 tokens (192 workgroups
// with keys) 16.4 / 19.0, 448 (256) 24.1 / 21.0, 11 tokens after 1400 20.0 /
// 23.4; 22 layers, 32 tokens 8.6 / 14.4, 64 tokens (352) 19.8 / 19.1, 3 tokens
// after 477 (704) 46.8 / 36.4.
bool prefill_is_short(int n_lb, int n_head_kv, int gqa, int pos0, int n_tok)
{
    const ShortShape s = short_shape(n_lb, n_head_kv, gqa, pos0, n_tok);
    if (s.z > 65535 || s.n_ch > 65535) return false;  // grid limits
    if (s.z * s.n_qt > kPrefillCounters || s.z * s.n_qt * s.n_ch * s.heads > kPrefillStates) return false;
    const long long cus = device_cus();
    if (s.z * s.n_qt * s.n_ch <= cus) return true;
    long long n = 0;  // workgroups with keys
    for (int qt = 0; qt < s.n_qt; ++qt) {
        const int last_key = pos0 + std::min((qt + 1) * kQTile, n_tok) - 1;
        n += s.z * ((last_key / kKTile + s.stage) / s.stage);
    }
    return s.stage == 1 ? n <= 2 * cus : 4 * n <= 3 * cus;
}

hipError_t launch_prefill_short(const PrefillParams& p, float* part, int* counters, hipStream_t s)
{
    if (!prefill_is_short(p.n_lb, p.n_head_kv, p.gqa, p.pos0, p.n_tok)) return hipErrorInvalidValue;
    const ShortShape h = short_shape(p.n_lb, p.n_head_kv, p.gqa, p.pos0, p.n_tok);
    if (h.n_ch > 1 && (!part || !counters)) return hipErrorInvalidValue;
    const ShortGrid g{h.n_hg, h.heads, part, counters};
    const dim3 grid(h.n_qt, h.n_ch, (unsigned)h.z);
    if (h.stage == 1)
        hipLaunchKernelGGL((prefill_short_kernel<1>), grid, dim3(64 * kShortWaves<1>), 0, s, p, g);
    else if (h.stage == 2)
        hipLaunchKernelGGL((prefill_short_kernel<2>), grid, dim3(64 * kShortWaves<2>), 0, s, p, g);
    else
        hipLaunchKernelGGL((prefill_short_kernel<4>), grid, dim3(64 * kShortWaves<4>), 0, s, p, g);
    return hipGetLastError();
}

// Workgroups per query tile of the planes' kernel, by the launch's query tiles
// (units: of a kv head's group of four q heads) per CU: a launch that leaves
// CUs idle, or has one or two workgroups on each, takes the longest walk's
// time.  Few units: as many workgroups as the CUs take one each, or two each
// where one would leave every walk a third of the keys or more; a workgroup more than
// that and some CUs hold one too many.  Measured, us per call by workgroups per
// query tile:
//   32 units (one layer of 32/4 heads, 128 tokens after 1900), 4 .. 10: 39.6 /
//     35.9 / 33.5 / 33.0 / 31.8 (256 workgroups) / 36.3 / 35.8;
//   64 (256 tokens after 1000), 3 .. 9: 35.4 / 31.0 (256) / 33.5 / 32.2 / 33.2 /
//     33.6 (512) / 37.6;
//   88 (333 tokens after 1500), 1 .. 6: 97.7 / 59.7 / 53.0 / 48.0 / 44.2 (440) /
//     48.9; 96 (384 after 900), 4 .. 6: 38.7 / 36.8 (480) / 39.9;
//   160 (640 tokens), 1 .. 4: 40.5 / 30.0 / 27.4 / 30.0; 256 (1024 tokens), 1 .. 5
//     61.1 / 42.7 / 41.3 / 44.5 / 45.3;
//   352 (two layers, 700 tokens), 1 .. 3: 47.9 / 39.9 / 41.9; 352 of few key
//     tiles (22 layers, 40 tokens after 140) 30.6 / 29.8 / 35.1;
//   616 (22 layers of 16/2 heads, 429 tokens), 1 / 2: 71.4 / 78.2.
// Two key splits in each workgroup, merged in LDS (one workgroup per CU), took
// 62.0, 28.1 and 46.3 us for 88, 160 and 256 units; two layers of 288 to 300 tokens
// (144 to 160 units of few key tiles), 20.5 and 21.5 us so, take 21.3 and 22.3.
namespace {

int attention_chunks(long long units, int n_kt)
{
    const long long cus = device_cus();
    long long n = 4 * units <= cus       ? cus / units
                  : 5 * units <= 2 * cus ? 2 * cus / units
                  : units <= cus         ? 3
                  : 4 * units <= 7 * cus ? 2
                                         : 1;
    n = std::min<long long>(n, (n_kt + 1) / 2);  // two key tiles each, as the kernel does
    return n > 1 && units <= kPrefillCounters && units * n * kWavesP <= kPrefillStates ? (int)n : 1;
}

int planes_chunks(int n_lb, int n_head_kv, int gqa, int pos0, int n_tok)
{
    const long long units =
        (long long)n_lb * n_head_kv * ((gqa + kWavesP - 1) / kWavesP) * ((n_tok + kQTile - 1) / kQTile);
    return attention_chunks(units, (pos0 + n_tok + kKTile - 1) / kKTile);
}

}  // namespace

bool prefill_shares(bool short_launch, int n_lb, int n_head_kv, int gqa, int pos0, int n_tok)
{
    return (short_launch ? short_shape(n_lb, n_head_kv, gqa, pos0, n_tok).n_ch
                         : planes_chunks(n_lb, n_head_kv, gqa, pos0, n_tok)) > 1;
}

hipError_t launch_prefill_attention(const PrefillParams& p, float* part, int* counters, hipStream_t s)
{
    const int n_ch = planes_chunks(p.n_lb, p.n_head_kv, p.gqa, p.pos0, p.n_tok);
    if (!p.kvp || p.n_ptiles != (p.pos0 + p.n_tok + kKTile - 1) / kKTile || (n_ch > 1 && (!part || !counters)))
        return hipErrorInvalidValue;
    return launch_attention(p, n_ch, part, counters, s);
}

}  // namespace tla
