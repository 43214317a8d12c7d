// What the attention kernels' files share: the geometry of a launch, and the
// prefill attention on the f32 matrix cores as a device function (attn_prefill,
// and attn_prefill_bf16's form for values that its parts cannot hold).
#pragma once

#include "common.h"
#include "kernels.h"

namespace slhip {
namespace {

struct Geo {
    const float* q;
    const float* k_new;
    const float* v_new;
    float* wcache;
    const float* cache;
    float* out;
    float* ws;
    uint32_t heads, kv_heads, seq, head_dim, group;
    uint32_t past_len, chunk, chunks;
    uint64_t batch_stride, layer_offset, parity_stride;  // elements
    float scale;
    const uint32_t* dyn;  // when set, dyn[0] is past_len
    // fused form: rope inputs and the extra outputs (see AttentionArgs)
    const uint32_t* pos;
    double theta;
    uint32_t rope_variant;
    float* merged;
    float* mirror;
    float* q_split;  // fused form: intermediates a later command reads, or null
    float* k_split;
    float* v_split;
    float* q_rot;
    float* k_rot;
    const float* rope_tab;  // fused form: the sine / cosine table, or null
    // paged form (attn_decode<.., PAGED>): key j of row b is slot j % page_size
    // of page block_table[b * pages_per_seq + j / page_size]; a page holds
    // K then V, [2][page_size][kv_heads][head_dim], page_stride elements, and
    // the layer's pages start at wcache + layer_offset; row b has seq_past[b]
    // cached keys before this step
    const uint32_t* block_table;
    const uint32_t* seq_past;
    uint32_t page_size, pages_per_seq;
    uint64_t page_stride;
};

__device__ __forceinline__ uint32_t past_of(const Geo& g) { return g.dyn != nullptr ? g.dyn[0] : g.past_len; }

inline Geo make_geo(const AttentionArgs& a, const Workspace& ws) {
    Geo g{};
    g.q = a.q;
    g.k_new = a.k_new;
    g.v_new = a.v_new;
    g.wcache = a.cache;
    g.cache = a.cache;
    g.out = a.out;
    g.ws = ws.data;
    g.heads = static_cast<uint32_t>(a.heads);
    g.kv_heads = static_cast<uint32_t>(a.kv_heads);
    g.seq = static_cast<uint32_t>(a.seq);
    g.head_dim = static_cast<uint32_t>(a.head_dim);
    g.group = static_cast<uint32_t>(a.heads / a.kv_heads);
    g.past_len = static_cast<uint32_t>(a.past_len);
    g.parity_stride = a.max_seq * a.kv_heads * a.head_dim;
    g.layer_offset = a.layer * 2 * g.parity_stride;
    g.batch_stride = a.layers * 2 * g.parity_stride;
    g.scale = a.scale;
    g.dyn = a.dyn;
    g.pos = a.positions;
    g.theta = static_cast<double>(a.theta);
    g.rope_variant = a.rope_variant;
    g.merged = a.merged;
    g.mirror = a.mirror;
    g.q_split = a.q_split;
    g.k_split = a.k_split;
    g.v_split = a.v_split;
    g.q_rot = a.q_rot;
    g.k_rot = a.k_rot;
    g.rope_tab = a.rope_table;
    if (a.block_table != nullptr) {  // paged cache: a pool of pages, rows at their own lengths
        const uint64_t row = a.kv_heads * a.head_dim;
        g.parity_stride = static_cast<uint64_t>(a.page_size) * row;
        g.page_stride = 2 * g.parity_stride;
        g.layer_offset = a.layer * a.num_pages * g.page_stride;
        g.batch_stride = 0;
        g.block_table = a.block_table;
        g.seq_past = a.seq_lens;
        g.page_size = a.page_size;
        g.pages_per_seq = a.pages_per_seq;
    }
    return g;
}

// ---- prefill: the f32 matrix cores ----
//
// A block owns 64 queries of one head (query wave w: queries 16 w .. 16 w +
// 15 of the block's range) and streams the keys 32 at a time; with KH = 2
// two waves serve each query wave, one per 16-key half of every tile, and
// their softmax states are combined through LDS at the end. Each
// tile of K and V rows goes to LDS (row stride D + 4 floats, so a wave's
// 16-byte K reads and 4-byte V reads hit 64 distinct banks) while the next
// tile's rows wait in registers. Per tile a wave forms S^T = K Q^T (keys x
// its 16 queries) and O^T += V^T P^T (dims x queries) with
// v_mfma_f32_16x16x4_f32: f32 products and f32 sums, like the VALU form.
// The accumulator layout puts rows 4 (l / 16) + i, column l % 16 in lane l,
// so every value a lane holds of S^T and O^T belongs to query l % 16: the
// online-softmax state (m, l) is per lane, a query's reductions span lanes
// l % 16 + 16 r (two lane swaps), and P^T is S^T's registers used as the B
// operand of the second product (the keys of its step i are 4 (l / 16) + i).
// The reduction over d is taken in a permuted order, the same for both
// operands: of each 16 dims, step s takes d = 4 (l / 16) + s, so a lane's
// operands of four steps are one float4 of K in LDS and of Q in registers.
// A block runs two query tiles one after the other, the last and the first,
// the second-to-last and the second, ..., so every block's causal key ranges
// add up to about the same work.
typedef float v4f_t __attribute__((ext_vector_type(4)));
constexpr int kPfQ = 64;  // queries per block
constexpr int kPfK = 32;  // keys per tile

// The next tile's K/V rows wait in registers while a tile is computed; they
// travel by value (PfRows). Filled through references into arrays, they were
// kept in scratch memory (at 128 registers per lane) or in LDS slots (at
// more), stored as soon as each load returned, so the loads never
// overlapped a tile's products. 8B layer at 1024 tokens, attn_prefill<128,
// 2>: 154.3 us in scratch, 129.1 in LDS slots, 106.0 in registers at two
// waves per SIMD (144 registers, one block per CU), 108.9 at four (128
// registers, two blocks per CU).
template <int N>
struct PfRows {
    float4 k[N], v[N];
};

template <int D, int KH>
__device__ __forceinline__ void prefill_f32(const Geo& g, uint32_t qtiles, float* __restrict__ ks,
                                            float* __restrict__ vs, float* __restrict__ xs) {
    constexpr int NT = 256 * KH;             // threads
    constexpr int LS = D + 4;                // LDS row stride (floats)
    constexpr int D16 = D / 16;              // float4 of Q per lane, and 16-dim output tiles
    constexpr int F4 = kPfK * D / 4 / NT;    // float4 of K (and of V) per thread per tile
    constexpr int NS = 2 / KH;               // 16-key halves of a tile per wave
    static_assert(F4 >= 1 && KH >= 1 && KH <= 2, "tile split");
    // ks, vs: kPfK * LS floats each
    // KH == 2: the second key half's softmax state (m, l, o) per lane of
    // each query wave, field-major, in xs ((2 + D / 4) * 256 floats)
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int qw = wave % 4;                 // query wave: queries 16 qw .. of the tile
    const int half = KH == 2 ? wave / 4 : 0; // KH == 2: keys 16 half .. 16 half + 15 of each tile
    const int c = lane % 16, kk = lane / 16;
    const uint32_t h = blockIdx.y;
    const uint64_t b = blockIdx.z;
    const uint32_t kvh = h / g.group;
    const uint32_t past = past_of(g);
    // query tiles qtiles - 1 - x, then x (the causal key ranges of the two
    // add up to about the same for every block)
    for (uint32_t pass = 0; pass < 2; ++pass) {
    const uint32_t qt = pass == 0 ? qtiles - 1 - blockIdx.x : blockIdx.x;
    if (pass == 1 && qt >= qtiles - 1 - blockIdx.x) break;  // block-uniform
    const uint32_t q0 = qt * kPfQ + qw * 16;    // the wave's first query
    const uint32_t t = q0 + c;                  // this lane's query
    const uint32_t tq = min(t, g.seq - 1);      // lanes past the end compute on the last query, unstored
    const uint32_t block_keys = past + min(g.seq, (qt + 1) * kPfQ);
    const uint32_t wave_keys = q0 < g.seq ? past + min(g.seq - 1, q0 + 15) + 1 : 0;
    const uint32_t my_keys = past + t + 1;

    float4 qv[D16];
    const float4* qrow = reinterpret_cast<const float4*>(g.q + ((b * g.heads + h) * g.seq + tq) * D);
#pragma unroll
    for (int j = 0; j < D16; ++j) qv[j] = qrow[4 * j + kk];
    v4f_t o[D16];
#pragma unroll
    for (int j = 0; j < D16; ++j) o[j] = v4f_t{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, lsum = 0.f;

    const uint64_t time_stride = static_cast<uint64_t>(g.kv_heads) * D;
    const float* kbase = g.cache + b * g.batch_stride + g.layer_offset + kvh * D;
    const float* vbase = kbase + g.parity_stride;
    // rows past the block's keys re-read its last key (their scores are
    // masked); the rows travel by value (an array the lambda filled through a
    // reference would be kept in memory, stored as soon as it arrived)
    auto load = [&](uint32_t kt) -> PfRows<F4> {
        PfRows<F4> n;
#pragma unroll
        for (int u = 0; u < F4; ++u) {
            const uint32_t e = tid + NT * u, row = e / (D / 4), col = e % (D / 4);
            const uint64_t j = min(kt + row, block_keys - 1);
            n.k[u] = reinterpret_cast<const float4*>(kbase + j * time_stride)[col];
            n.v[u] = reinterpret_cast<const float4*>(vbase + j * time_stride)[col];
        }
        return n;
    };
    PfRows<F4> nx = load(0);
    for (uint32_t kt = 0; kt < block_keys; kt += kPfK) {
        __syncthreads();  // every wave is done reading the previous tile
#pragma unroll
        for (int u = 0; u < F4; ++u) {
            const uint32_t e = tid + NT * u, row = e / (D / 4), col = e % (D / 4);
            *reinterpret_cast<float4*>(ks + row * LS + 4 * col) = nx.k[u];
            *reinterpret_cast<float4*>(vs + row * LS + 4 * col) = nx.v[u];
        }
        __syncthreads();
        // the next tile's rows, waiting in registers while this tile is computed
        nx = load(kt + kPfK);
        // wave-uniform: no key of the wave's part of the tile is visible to it
        if (kt + 16 * half >= wave_keys) continue;
        // S^T: keys 16 sub + 4 kk + i of the tile, query c
        v4f_t st[NS];
#pragma unroll
        for (int si = 0; si < NS; ++si) {
            const int sub = KH == 2 ? half : si;
            st[si] = v4f_t{0.f, 0.f, 0.f, 0.f};
            const float* krow = ks + (sub * 16 + c) * LS + 4 * kk;
#pragma unroll
            for (int j = 0; j < D16; ++j) {
                const float4 k4 = *reinterpret_cast<const float4*>(krow + 16 * j);
                st[si] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.x, qv[j].x, st[si], 0, 0, 0);
                st[si] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.y, qv[j].y, st[si], 0, 0, 0);
                st[si] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.z, qv[j].z, st[si], 0, 0, 0);
                st[si] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.w, qv[j].w, st[si], 0, 0, 0);
            }
        }
        float p[NS][4];
        float tmax = -INFINITY;
#pragma unroll
        for (int si = 0; si < NS; ++si)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int sub = KH == 2 ? half : si;
                const uint32_t key = kt + 16 * sub + 4 * kk + i;
                p[si][i] = key < my_keys ? st[si][i] * g.scale : -INFINITY;
                tmax = fmaxf(tmax, p[si][i]);
            }
        tmax = fmaxf(tmax, lane_xor16(tmax));
        tmax = fmaxf(tmax, lane_xor32(tmax));
        // With one key half per wave a query can see none of a tile's keys
        // (m_new == -inf): the guards keep corr and every weight 0, not NaN.
        // (With both halves key 0 is visible to every query, so m is finite
        // from the first tile on.)
        const float m_new = fmaxf(m, tmax);
        const float corr = m == -INFINITY ? 0.f : expf(m - m_new);
        float psum = 0.f;
#pragma unroll
        for (int si = 0; si < NS; ++si)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[si][i] = p[si][i] == -INFINITY ? 0.f : expf(p[si][i] - m_new);
                psum += p[si][i];
            }
        psum += lane_xor16(psum);
        psum += lane_xor32(psum);
        lsum = lsum * corr + psum;
        m = m_new;
        // O^T += V^T P^T: dims 16 j + c (A), keys 16 sub + 4 kk + i (k), query c (B)
#pragma unroll
        for (int j = 0; j < D16; ++j) {
            o[j] *= corr;
#pragma unroll
            for (int si = 0; si < NS; ++si)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int sub = KH == 2 ? half : si;
                    o[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vs[(16 * sub + 4 * kk + i) * LS + 16 * j + c],
                                                                 p[si][i], o[j], 0, 0, 0);
                }
        }
    }
    if constexpr (KH == 2) {
        // the second half's state through LDS; the first half's waves merge
        const int x = qw * kWave + lane;
        if (half == 1) {
            xs[x] = m;
            xs[256 + x] = lsum;
#pragma unroll
            for (int j = 0; j < D16; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) xs[(2 + 4 * j + e) * 256 + x] = o[j][e];
        }
        __syncthreads();
        if (half == 1) continue;
        const float m1 = xs[x], l1 = xs[256 + x];
        const float mm = fmaxf(m, m1);
        const float c0 = m == -INFINITY ? 0.f : expf(m - mm), c1 = m1 == -INFINITY ? 0.f : expf(m1 - mm);
        lsum = lsum * c0 + l1 * c1;
#pragma unroll
        for (int j = 0; j < D16; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[j][e] = o[j][e] * c0 + xs[(2 + 4 * j + e) * 256 + x] * c1;
    }
    if (t < g.seq) {
        const float inv = 1.0f / lsum;
        // [B, H, S, D], and MergeHeads' [B, S, H * D] (fused form)
        float* orow = g.out != nullptr ? g.out + ((b * g.heads + h) * g.seq + t) * D + 4 * kk : nullptr;
        float* mrow = g.merged != nullptr ? g.merged + ((b * g.seq + t) * g.heads + h) * D + 4 * kk : nullptr;
#pragma unroll
        for (int j = 0; j < D16; ++j) {
            const float4 v = make_float4(o[j][0] * inv, o[j][1] * inv, o[j][2] * inv, o[j][3] * inv);
            if (orow != nullptr) *reinterpret_cast<float4*>(orow + 16 * j) = v;
            if (mrow != nullptr) *reinterpret_cast<float4*>(mrow + 16 * j) = v;
        }
    }
    }
}

}  // namespace
}  // namespace slhip
