// Prefill attention on the bf16 matrix cores (reference/attention.rs:129-219).
//
// In a file of its own, so that the decode kernels of attention.hip keep their
// places in that file's code object: with these four kernels among them 8B INT4
// decode ran 0.6% slower on the same instructions.
//
// The f32 matrix cores do 1,024 multiply-adds in 32 cycles, the bf16 ones 8,192
// in 16. A float is exactly three bf16 parts (8 + 8 + 8 significant bits),
// x = h + m + l; of the nine products of two such splits the six down to 2^-16
// (hh, hm, mh, hl, lh, mm) are kept, smallest first, so a product is off by
// about 2^-24 of itself, like a rounded f32 one: 6 x 16 cycles for 32 x 16 x 16
// multiply-adds against 8 x 32. Vector instructions do not overlap with
// either, so the splits are made once per layer and not once per query tile:
// attn_planes writes every 32-key tile of K and V as parts in operand order
// (K: per 16 keys and 32 dims, lane l holds key l % 16, dims 8 (l / 16) ..; V:
// per 16 dims, lane l holds dim l % 16 and the keys 4 (l / 16) .., 16 + 4 (l /
// 16) .. - the keys whose weights the same lane holds after S^T), and
// attn_prefill_bf16 copies tiles to LDS and reads them 16 bytes per lane,
// without bank conflicts. The softmax is attn_prefill's on unscaled scores, in base
// 2 (so a negative scale, whose maximum is their minimum, is left to that form);
// each product's sum starts from zero and joins O^T with the rescale's multiply-add.
//
// Values whose parts or partial products could leave the range (NaN, infinity,
// 2^56 and above, below 2^-100) are found by attn_planes per tile (`flags`) and
// in q per block; a block that sees one does its query tiles as attn_prefill.
//
// Per layer with the planes (f32 form before): 1024 rows, 32 heads of 128: 117 ->
// 94 us; 3001 rows, 32 heads of 64: 519 -> 305; 2 x 256 rows after 640, heads of
// 128: 146 -> 121. Bound by vector and matrix instructions (D = 128, per 32 keys
// of a wave: 96 MFMA, 1,536 cycles, and about 300 vector instructions, 1,200) and,
// with one block of 8 waves per CU at D = 128, the waits between them; D = 64 has
// room for two.
#include "attention_geo.h"
#include "common.h"
#include "kernels.h"

namespace slhip {
namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bool out_of_range(float v) {
    constexpr uint32_t lo = 27u << 23, hi = 183u << 23;  // 2^-100, 2^56
    const uint32_t bits = __float_as_uint(v) & 0x7fffffffu;
    return bits != 0 && bits - lo >= hi - lo;
}

template <int D>
constexpr uint32_t plane_words() {  // 16-byte words of one 32-key tile's parts of K and V
    return (2 * (D / 32) + D / 16) * 3 * 64;
}

__device__ __forceinline__ void split3(const float (&x)[8], v8bf& h, v8bf& m, v8bf& l) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        h[i] = static_cast<__bf16>(x[i]);
        const float r = x[i] - static_cast<float>(h[i]);
        m[i] = static_cast<__bf16>(r);
        l[i] = static_cast<__bf16>(r - static_cast<float>(m[i]));
    }
}

// A grid of (blocks, kv_heads, batch); each block takes every gridDim.x-th tile.
template <int D>
__global__ __launch_bounds__(256) void attn_planes(Geo g, u32x4* __restrict__ planes, uint32_t* __restrict__ flags,
                                                   uint32_t tiles_max) {
    prefetch_kernarg<arg_bytes<Geo, u32x4*, uint32_t*, uint32_t>()>();
    const uint32_t tid = threadIdx.x, kvh = blockIdx.y;
    const uint64_t b = blockIdx.z, head = b * g.kv_heads + kvh;
    const uint32_t keys = past_of(g) + g.seq, tiles = (keys + 31) / 32;
    const uint64_t time_stride = static_cast<uint64_t>(g.kv_heads) * D;
    const float* kbase = g.cache + b * g.batch_stride + g.layer_offset + kvh * D;
    const float* vbase = kbase + g.parity_stride;
    const auto put = [](u32x4* at, uint32_t frag, uint32_t lane, const float (&x)[8]) {
        v8bf p[3];
        split3(x, p[0], p[1], p[2]);
#pragma unroll
        for (int q = 0; q < 3; ++q) at[(frag * 3 + q) * 64 + lane] = __builtin_bit_cast(u32x4, p[q]);
    };
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        u32x4* const at = planes + (head * tiles_max + tile) * plane_words<D>();
        const uint32_t k0 = tile * 32;
        bool bad = false;
        const auto see = [&](float v) { bad |= out_of_range(v); };
        for (uint32_t u = tid; u < 32 * (D / 8); u += 256) {
            const uint32_t key = u / (D / 8), d8 = u % (D / 8);
            float x[8] = {};
            if (k0 + key < keys) {
                const float4* row = reinterpret_cast<const float4*>(kbase + (k0 + key) * time_stride) + 2 * d8;
                const float4 lo = row[0], hi = row[1];
                x[0] = lo.x, x[1] = lo.y, x[2] = lo.z, x[3] = lo.w, x[4] = hi.x, x[5] = hi.y, x[6] = hi.z, x[7] = hi.w;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) see(x[i]);
            put(at, key / 16 * (D / 32) + d8 / 4, key % 16 + 16 * (d8 % 4), x);
        }
        for (uint32_t u = tid; u < 4 * D / 2; u += 256) {
            const uint32_t grp = u / (D / 2), d = u % (D / 2) * 2;
            float x[8] = {}, y[8] = {};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t key = k0 + 16 * (i / 4) + 4 * grp + i % 4;
                if (key < keys) {
                    const float2 v = *reinterpret_cast<const float2*>(vbase + key * time_stride + d);
                    x[i] = v.x;
                    y[i] = v.y;
                }
                see(x[i]);
                see(y[i]);
            }
            const uint32_t frag = 2 * (D / 32) + d / 16;
            put(at, frag, d % 16 + 16 * grp, x);
            put(at, frag, d % 16 + 1 + 16 * grp, y);
        }
        const int any = __syncthreads_or(bad);
        if (tid == 0) flags[head * tiles_max + tile] = any ? 1u : 0u;
    }
}

template <int D>
__global__ __launch_bounds__(512, D == 64 ? 4 : 2) void attn_prefill_bf16(
    Geo g, uint32_t qtiles, const u32x4* __restrict__ planes, const uint32_t* __restrict__ flags, uint32_t tiles_max) {
    prefetch_kernarg<arg_bytes<Geo, uint32_t, const u32x4*, const uint32_t*, uint32_t>()>();
    constexpr int KT = D / 32, DT = D / 16;            // 32-dim steps, 16-dim output tiles
    constexpr uint32_t PW = plane_words<D>();          // 16-byte words of a tile
    constexpr int NL = 2 * PW / 512;                   // words of a 64-key stage per thread
    constexpr int XF = 2 + D / 4;
    __shared__ u32x4 ts[2 * PW];
    __shared__ float xs[XF * 256];  // the second key half's softmax state, field-major
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int qw = wave % 4, half = wave / 4;  // queries 16 qw ..; tile `half` of each stage
    const int c = lane % 16, kk = lane / 16;
    const uint32_t h = blockIdx.y;
    const uint64_t b = blockIdx.z, head = b * g.kv_heads + h / g.group;
    const uint32_t past = past_of(g);
    {
        bool bad = false;
        const uint32_t keys = past + min(g.seq, (qtiles - blockIdx.x) * kPfQ);  // of the later of its query tiles
        for (uint32_t x = tid; x < (keys + 31) / 32; x += 512) bad |= flags[head * tiles_max + x] != 0;
        const float4* const q4 = reinterpret_cast<const float4*>(g.q + (b * g.heads + h) * g.seq * D);
        for (uint32_t pass = 0; pass < 2; ++pass) {
            const uint32_t from = (pass == 0 ? qtiles - 1 - blockIdx.x : blockIdx.x) * kPfQ;
            const uint32_t words = min(kPfQ, g.seq - from) * (D / 4);
            for (uint32_t x = tid; x < words; x += 512) {
                const float4 v = q4[from * (D / 4) + x];
                bad |= out_of_range(v.x) || out_of_range(v.y) || out_of_range(v.z) || out_of_range(v.w);
            }
        }
        if (__syncthreads_or(bad)) {
            float* const f = reinterpret_cast<float*>(ts);
            static_assert(sizeof(ts) >= 2 * kPfK * (D + 4) * sizeof(float), "K and V of the f32 form");
            prefill_f32<D, 2>(g, qtiles, f, f + kPfK * (D + 4), xs);
            return;
        }
    }
    const float c2 = static_cast<float>(g.scale * 1.4426950408889634);
    const u32x4* const base = planes + head * tiles_max * PW;
    for (uint32_t pass = 0; pass < 2; ++pass) {
        const uint32_t qt = pass == 0 ? qtiles - 1 - blockIdx.x : blockIdx.x;
        if (pass == 1 && qt >= qtiles - 1 - blockIdx.x) break;  // block-uniform
        const uint32_t q0 = qt * kPfQ + qw * 16;
        const uint32_t t = q0 + c;              // this lane's query
        const uint32_t tq = min(t, g.seq - 1);  // lanes past the end compute on the last query, unstored
        const uint32_t block_keys = past + min(g.seq, (qt + 1) * kPfQ);
        const uint32_t wave_keys = q0 < g.seq ? past + min(g.seq - 1, q0 + 15) + 1 : 0;
        const uint32_t my_keys = past + t + 1;
        const uint32_t last_stage = (block_keys - 1) / 64;

        v8bf qp[KT][3];
        {
            const float4* qrow = reinterpret_cast<const float4*>(g.q + ((b * g.heads + h) * g.seq + tq) * D);
#pragma unroll
            for (int j = 0; j < KT; ++j) {
                const float4 lo = qrow[8 * j + 2 * kk], hi = qrow[8 * j + 2 * kk + 1];
                const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                split3(x, qp[j][0], qp[j][1], qp[j][2]);
            }
        }
        v4f_t o[DT];
#pragma unroll
        for (int j = 0; j < DT; ++j) o[j] = v4f_t{0.f, 0.f, 0.f, 0.f};
        float m = -INFINITY, lsum = 0.f;
        // (an odd last tile's stage reads the tile after it, which the planes
        // have room for and no wave uses)
        u32x4 nx[NL];
#pragma unroll
        for (int u = 0; u < NL; ++u) nx[u] = base[tid + 512 * u];
        for (uint32_t stage = 0; stage <= last_stage; ++stage) {
            __syncthreads();  // every wave is done reading the previous stage
#pragma unroll
            for (int u = 0; u < NL; ++u) ts[tid + 512 * u] = nx[u];
            __syncthreads();
            const u32x4* const next = base + static_cast<uint64_t>(min(stage + 1, last_stage)) * 2 * PW;
#pragma unroll
            for (int u = 0; u < NL; ++u) nx[u] = next[tid + 512 * u];
            const uint32_t kt = 64 * stage + 32 * half;
            // wave-uniform: no key of the wave's tile is visible to it
            if (kt >= wave_keys) continue;
            const u32x4* const tile = ts + half * PW + lane;
            const auto frag = [&](int f, int q) -> v8bf { return __builtin_bit_cast(v8bf, tile[(f * 3 + q) * 64]); };
            const v4f_t zero = {0.f, 0.f, 0.f, 0.f};
#define SL_BF16(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0)
            // S^T: keys 16 s + 4 kk + i, query c; the leading products apart
            // from the small ones, so that a large sum rounds once per step
            v4f_t st[2];
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
                v4f_t hi = zero, lo = zero;
#pragma unroll
                for (int j = 0; j < KT; ++j) {
                    const v8bf k0 = frag(s2 * KT + j, 0), k1 = frag(s2 * KT + j, 1), k2 = frag(s2 * KT + j, 2);
                    lo = SL_BF16(k2, qp[j][0], lo);
                    lo = SL_BF16(k0, qp[j][2], lo);
                    lo = SL_BF16(k1, qp[j][1], lo);
                    lo = SL_BF16(k1, qp[j][0], lo);
                    lo = SL_BF16(k0, qp[j][1], lo);
                    hi = SL_BF16(k0, qp[j][0], hi);
                }
                st[s2] = hi + lo;
            }
            // exp(x scale - max(x scale)) is exp2((x - max(x)) c) for c >= 0:
            // exactly 1 for the largest score, however large (a rounded x c
            // differs from the exact one by more than 128 from 2^31 on, and
            // its power of two overflows); only a tile with keys past the
            // wave's first query is masked (wave-uniform)
            const bool edge = kt + 32 > past + q0 + 1;
            float p[8];
            float tmax = -INFINITY;
#pragma unroll
            for (int i = 0; i < 8; ++i) p[i] = st[i / 4][i % 4];
            if (edge) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (kt + 16 * (i / 4) + 4 * kk + i % 4 >= my_keys) p[i] = -INFINITY;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) tmax = fmaxf(tmax, p[i]);
            tmax = fmaxf(tmax, lane_xor16(tmax));
            tmax = fmaxf(tmax, lane_xor32(tmax));
            // A query can see none of the tile's keys (m_new == -inf): the
            // guards keep corr and every weight 0, not NaN.
            const float m_new = fmaxf(m, tmax);
            const float corr = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - m_new) * c2);
            float psum = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) p[i] = __builtin_amdgcn_exp2f((p[i] - m_new) * c2);
            if (edge) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (kt + 16 * (i / 4) + 4 * kk + i % 4 >= my_keys) p[i] = 0.f;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) psum += p[i];
            psum += lane_xor16(psum);
            psum += lane_xor32(psum);
            lsum = lsum * corr + psum;
            m = m_new;
            v8bf p0, p1, p2;
            split3(p, p0, p1, p2);
            // O^T += V^T P^T: dims 16 j + 4 kk + e, query c
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                const v8bf v0 = frag(2 * KT + j, 0), v1 = frag(2 * KT + j, 1), v2 = frag(2 * KT + j, 2);
                v4f_t r = SL_BF16(v2, p0, zero);
                r = SL_BF16(v0, p2, r);
                r = SL_BF16(v1, p1, r);
                r = SL_BF16(v1, p0, r);
                r = SL_BF16(v0, p1, r);
                r = SL_BF16(v0, p0, r);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[j][e] = fmaf(o[j][e], corr, r[e]);
            }
#undef SL_BF16
        }
        // the second half's state through LDS; the first half's waves merge
        const int x = qw * kWave + lane;
        if (half == 1) {
            xs[x] = m;
            xs[256 + x] = lsum;
#pragma unroll
            for (int j = 0; j < DT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) xs[(2 + 4 * j + e) * 256 + x] = o[j][e];
        }
        __syncthreads();
        if (half == 1) continue;
        const float m1 = xs[x], l1 = xs[256 + x];
        const float mm = fmaxf(m, m1);
        const float c0 = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - mm) * c2);
        const float c1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m1 - mm) * c2);
        lsum = lsum * c0 + l1 * c1;
        if (t < g.seq) {
            const float inv = 1.0f / lsum;
            // [B, H, S, D], and MergeHeads' [B, S, H * D] (fused form)
            float* orow = g.out != nullptr ? g.out + ((b * g.heads + h) * g.seq + t) * D + 4 * kk : nullptr;
            float* mrow = g.merged != nullptr ? g.merged + ((b * g.seq + t) * g.heads + h) * D + 4 * kk : nullptr;
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                float w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) w[e] = (o[j][e] * c0 + xs[(2 + 4 * j + e) * 256 + x] * c1) * inv;
                const float4 v = make_float4(w[0], w[1], w[2], w[3]);
                if (orow != nullptr) *reinterpret_cast<float4*>(orow + 16 * j) = v;
                if (mrow != nullptr) *reinterpret_cast<float4*>(mrow + 16 * j) = v;
            }
        }
    }
}

}  // namespace

// The parts and flags go to the end of the workspace, past the first `keep`
// floats; without that room, or for short chunks, hipErrorNotSupported (the f32
// form). The line between the two depends on the chunk only, not on the keys before
// it, so that a replayed submission takes the form it was recorded with: at these
// lengths they are even without earlier keys (one op with KvAppend, 32 heads on 8
// K/V heads, us, bf16 / f32: head_dim 64, 512 rows 51 / 50, 768 61 / 66; head_dim
// 128, 256 rows 52 / 51, 512 68 / 76, 1024 98 / 125) and earlier keys favour bf16
// (256 rows after 768: 64 89 / 113, 128 125 / 182).
hipError_t launch_attention_prefill_bf16(const AttentionArgs& a, const float* q, const Workspace& ws, uint64_t keep,
                                         hipStream_t s) {
    const bool wide = a.head_dim == 128;
    const uint64_t tiles = (a.max_seq + 63) / 64 * 2;  // an even count: stages are two tiles
    const uint64_t words = a.batch * a.kv_heads * tiles * (wide ? plane_words<128>() : plane_words<64>());
    const uint64_t flag_floats = (a.batch * a.kv_heads * tiles + 63) / 64 * 64, floats = flag_floats + 4 * words;
    if (!(wide || a.head_dim == 64) || a.seq < (wide ? 256 : 512) || !(a.scale >= 0.f && a.scale <= 32.f) ||
        tiles > 0xffffffull || ws.shared || keep + floats + 64 > ws.floats)
        return hipErrorNotSupported;
    Geo g = make_geo(a, ws);
    g.q = q;
    const uint64_t at = (ws.floats - floats) / 64 * 64;
    uint32_t* const flags = reinterpret_cast<uint32_t*>(ws.data + at);
    u32x4* const planes = reinterpret_cast<u32x4*>(ws.data + at + flag_floats);
    const uint32_t qtiles = static_cast<uint32_t>((a.seq + kPfQ - 1) / kPfQ), tm = static_cast<uint32_t>(tiles);
    const dim3 grid((qtiles + 1) / 2, g.heads, static_cast<unsigned>(a.batch));
    const dim3 pgrid(tm < 64 ? tm : 64, g.kv_heads, static_cast<unsigned>(a.batch));
    if (wide) {
        attn_planes<128><<<pgrid, 256, 0, s>>>(g, planes, flags, tm);
        attn_prefill_bf16<128><<<grid, 512, 0, s>>>(g, qtiles, planes, flags, tm);
    } else {
        attn_planes<64><<<pgrid, 256, 0, s>>>(g, planes, flags, tm);
        attn_prefill_bf16<64><<<grid, 512, 0, s>>>(g, qtiles, planes, flags, tm);
    }
    return hipGetLastError();
}

// Loads this file's code object now: HIP loads one at the first use of
// any of its kernels, which otherwise lands inside the first submission
// that needs it (about 1-2 ms each, more for large objects).
hipError_t load_code_attention_bf16() {
    hipFuncAttributes attr;
    return hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&attn_planes<64>));
}

}  // namespace slhip
