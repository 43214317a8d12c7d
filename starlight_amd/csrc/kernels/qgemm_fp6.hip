// Group-quantized MatMulNT for many activation rows (prefill) with INT4
// weights, on the block-scaled 6-bit matrix cores:
// out[m, n] = sum_k a[m, k] * (q[n, k] * s[n, k / G]), G a multiple of 128.
//
// Exactness plan. E2M3, the 6-bit float of v_mfma_scale_f32_16x16x128_f8f6f4,
// holds every integer of magnitude at most 16 exactly (as n / 8, with the
// sign-magnitude code n itself), so an INT4 code is one E2M3 value. Of every
// activation row, each 32 elements that one lane feeds to a product share an
// exponent E (|a| < 2^E) and become integers X = rint(a * 2^(24 - E)), cut
// into five signed base-32 digits, X = sum_j d_j 32^j with |d_j| <= 16, each
// one E2M3 value as well: 24 significant bits below the block's largest
// element. The products d_j * q are exact, and the instruction's block scales
// carry 2^E (relative to the row's largest exponent) and 32^j. A product's sum
// over its 128 k is exact where the blocks' exponents are close, but adding
// it to a larger sum rounds down by up to 2^-23 of that: chained over all five
// digits, the errors of a whole model's logits grew 1.2 to 2.4 times. So the
// three low digits and the two high ones are summed apart (the high sum needs
// 19 bits plus the exponents' spread), added in f32, multiplied by the
// group's scale, added to the f32 result, and that is scaled back by the
// row's exponent at the end. Error against float64 as the fp16 split's
// (qgemm_mfma.hip) or below: [4096 x 14336] at M = 1024 1.5e-7 against 1.7e-7,
// [28672 x 4096] 1.3e-7 against 1.4e-7; whole models the same.
//
// Rate. Register-resident loops on MI355X reach 8.43 PFLOP/s with 6-bit
// operands and 2.17 PFLOP/s with fp16 ones: five 6-bit products per multiply
// allow 1.69 PFLOP/s of f32 result, two fp16 ones 1.08. With the split, against
// the fp16 route: [28672 x 4096] M = 1024 358 us against 525 (673 TFLOP/s of
// f32 result), M = 77 58 against 89; [4096 x 14336] M = 1024 212 against 304,
// M = 512 117 against 186, M = 77 41 against 159; [4096 x 4096] M = 77 24
// against 56. What bounds it now: vector and matrix instructions of a SIMD's
// waves do not overlap here, and a 64 x 256 tile's pass has 80 products (1,280
// cycles) and about 160 vector instructions (640) per wave, two waves per
// SIMD: 3,840 of about 6,000 cycles measured; LDS is busy a third of the time.
// Deeper operand prefetch and wave priorities changed nothing, and gathering
// the records in operand order from memory (no LDS conflicts, scattered
// 64-byte loads) was slower.
//
// Kernels
//  * repack_fp6 (bind): the codes as E2M3 in operand order, per 16-row tile
//    and 128-k superblock 64 lanes x 16 bytes, then 64 lanes x 8 bytes. Lane
//    l holds row l % 16 and the elements k = 16 (i / 4) + 4 (l / 16) + i % 4,
//    i < 32, of the superblock (the order in which a quad of threads reads
//    whole float4 of the activations);
//  * split_fp6: one block per row: row maximum, block exponents, digits. A
//    record of 512 bytes per row and superblock: five digit planes of 4 lanes
//    x 16 then 4 x 8 bytes, and the four block scales;
//  * qgemm_fp6: records staged through LDS in rows of 528 bytes (the 16 rows
//    of one operand read fall on disjoint groups of 4 banks), shared by the
//    block's waves; weights straight from memory into registers, one
//    superblock ahead.
#include "common.h"
#include "kernels.h"
#include "qgemm_act.h"
#include "qgemm_plan.h"
#include "starlight_hip.h"

namespace slhip {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kDigits = 5, kLowDigits = 3;
constexpr uint32_t kRecord = 512;     // bytes per row and superblock
constexpr uint32_t kPlane = 96;       // bytes of one digit of a record
constexpr uint32_t kScalesAt = kDigits * kPlane;
constexpr uint32_t kLdsRow = kRecord + 16;
constexpr uint32_t kTileBytes = 1536;           // one 16-row weight tile of one superblock
constexpr int kOne = 127;                       // E8M0 of 1.0

// Sign and magnitude of d, |d| <= 16: the E2M3 code of d / 8.
__device__ __forceinline__ uint32_t e2m3(int d) {
    return static_cast<uint32_t>(max(d, -d)) | (static_cast<uint32_t>(d >> 26) & 32u);
}

// Element i of lane l within a superblock.
__device__ __forceinline__ uint32_t lane_k(uint32_t l, uint32_t i) { return 16 * (i / 4) + 4 * (l / 16) + i % 4; }

// One thread per 16 elements (half a lane) of the 6-bit copy.
__global__ __launch_bounds__(256) void repack_fp6(const uint8_t* __restrict__ payload, uint32_t* __restrict__ tiles,
                                                  uint64_t n, uint64_t k, uint64_t units) {
    const uint64_t sb_total = k / 128;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t u = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; u < units; u += stride) {
        const uint32_t h = u % 2, lane = u / 2 % kWave;
        const uint64_t t = u / (2 * kWave), row = t / sb_total * 16 + lane % 16, sb = t % sb_total;
        uint32_t w[3] = {0u, 0u, 0u};
        if (row < n) {
            for (uint32_t i = 0; i < 16; ++i) {
                const uint64_t e = row * k + sb * 128 + lane_k(lane, 16 * h + i);  // k is even: rows are whole bytes
                const int nib = payload[e / 2] >> (4 * (e % 2)) & 15;
                const uint32_t code = e2m3(nib < 8 ? nib : nib - 16);
                w[6 * i / 32] |= code << (6 * i % 32);
                if (6 * i % 32 > 26) w[6 * i / 32 + 1] |= code >> (32 - 6 * i % 32);
            }
        }
        uint32_t* const dst = tiles + t * (kTileBytes / 4);
        if (h == 0) {
            for (int q = 0; q < 3; ++q) dst[4 * lane + q] = w[q];
        } else {
            dst[4 * lane + 3] = w[0];
            dst[256 + 2 * lane] = w[1];
            dst[256 + 2 * lane + 1] = w[2];
        }
    }
}

__device__ __forceinline__ uint32_t block_max_u32(uint32_t v, uint32_t* scratch) {
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    v = wave_max_u32(v);
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    return max(max(scratch[0], scratch[1]), max(scratch[2], scratch[3]));
}

// |v| as bits, ordered like the magnitudes (infinities and NaN on top)
__device__ __forceinline__ uint32_t mag4(float4 v) {
    constexpr uint32_t kMag = 0x7fffffffu;
    return max(max(__float_as_uint(v.x) & kMag, __float_as_uint(v.y) & kMag),
               max(__float_as_uint(v.z) & kMag, __float_as_uint(v.w) & kMag));
}

// E with |v| < 2^E of a finite magnitude (0 for zero); 128 otherwise.
__device__ __forceinline__ int mag_exp(uint32_t mag) {
    if (mag >= 0x7f800000u) return 128;
    int e = 0;
    if (mag != 0) frexpf(__uint_as_float(mag), &e);
    return e;
}

// Row r's records. Thread t holds units t + 256 j, j < NP (k <= 4096 NP): unit
// u is half h = u % 2 (elements 16 h ..) of lane block b = u / 2 % 4 of
// superblock u / 8. With gamma (NP <= 2), of RMSNorm(a) * gamma; NP == 0 reads
// the row twice instead of holding it. Bound by the vector unit's work on the
// digits and by its reads; M = 1024, k = 4096: see qgemm_fp6.
template <int NP>
__global__ __launch_bounds__(256) void split_fp6(const float* __restrict__ a, const float* __restrict__ u,
                                                 uint8_t* __restrict__ records, int* __restrict__ row_exp, uint32_t k,
                                                 const float* __restrict__ gamma, float eps) {
    __shared__ float scratch[4];
    __shared__ uint32_t scratch_u[4];
    const uint64_t r = blockIdx.x;
    const float4* row = reinterpret_cast<const float4*>(a + r * k);
    const float4* urow = u != nullptr ? reinterpret_cast<const float4*>(u + r * k) : nullptr;
    const uint32_t k4 = k / 4, units = k / 16;
    // float4 q of unit w
    auto at = [](uint32_t w, uint32_t q) -> uint32_t { return w / 8 * 32 + 4 * (4 * (w % 2) + q) + w / 2 % 4; };
    float4 keep[NP > 0 ? NP : 1][4];
    uint32_t mx = 0;
    if constexpr (NP > 0) {
        if (NP <= 2 && gamma != nullptr) {
            // RMSNorm first. Its sum of squares runs in the standalone
            // kernel's order (rms_norm_vec: thread t over float4 columns t +
            // 256 i, ascending, then block_sum), from a second set of loads
            // of the row, so the normalised values are bit-identical to that
            // kernel's output. Every load is unconditional (clamped indices;
            // columns past the row count as zeros, which leave the sum
            // unchanged) and issued before any of them is used.
            const float4* g4 = reinterpret_cast<const float4*>(gamma);
            float4 xv[4 * NP], gv[NP][4];
#pragma unroll
            for (int j = 0; j < NP; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t i = at(min(threadIdx.x + 256u * j, units - 1), q);
                    keep[j][q] = row[i];
                    gv[j][q] = g4[i];
                }
#pragma unroll
            for (int i = 0; i < 4 * NP; ++i) xv[i] = row[min(threadIdx.x + 256u * i, k4 - 1)];
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < 4 * NP; ++i) {
                const float4 v = threadIdx.x + 256u * i < k4 ? xv[i] : make_float4(0.f, 0.f, 0.f, 0.f);
                ss = fmaf(v.x, v.x, ss);
                ss = fmaf(v.y, v.y, ss);
                ss = fmaf(v.z, v.z, ss);
                ss = fmaf(v.w, v.w, ss);
            }
            ss = block_sum(ss, scratch);
            const float inv = 1.0f / sqrtf(ss / static_cast<float>(k) + eps);
#pragma unroll
            for (int j = 0; j < NP; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float4& v = keep[j][q];
                    v.x = (v.x * inv) * gv[j][q].x;
                    v.y = (v.y * inv) * gv[j][q].y;
                    v.z = (v.z * inv) * gv[j][q].z;
                    v.w = (v.w * inv) * gv[j][q].w;
                }
        } else {
#pragma unroll
            for (int j = 0; j < NP; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    keep[j][q] = act4(row, urow, at(min(threadIdx.x + 256u * j, units - 1), q));
        }
        // (units past the row repeat its last one: the maximum is unchanged)
#pragma unroll
        for (int j = 0; j < NP; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) mx = max(mx, mag4(keep[j][q]));
    } else {
        for (uint32_t i = threadIdx.x; i < k4; i += 256) mx = max(mx, mag4(act4(row, urow, i)));
    }
    const int er = mag_exp(block_max_u32(mx, scratch_u));
    if (threadIdx.x == 0) row_exp[r] = er;
    uint8_t* const rec = records + r * (k / 128) * kRecord;
    // Unit w's digits; its lane block's other half is in the neighbouring thread.
    auto put = [&](uint32_t w, const float4 (&v)[4]) {
        uint32_t m = max(max(mag4(v[0]), mag4(v[1])), max(mag4(v[2]), mag4(v[3])));
        m = max(m, static_cast<uint32_t>(dpp_i<kDppXor1>(static_cast<int>(m))));
        if (w >= units) return;
        // (a block of zeros takes the row's exponent: 0 would lie 127 and more
        // above that of a row of denormals, where the scale's byte is NaN's)
        const int e = m != 0 ? mag_exp(m) : er;
        const bool finite = m < 0x7f800000u;
        const bool held = finite && kOne + e - er >= 0;  // else below what a block scale can say: zero digits
        const uint32_t b = w / 2 % 4;
        uint8_t* const dst = rec + static_cast<uint64_t>(w / 8) * kRecord;
        constexpr int kBias = 16 * (1 + 32 + 1024 + 32768 + 1048576);  // makes every digit d + 16 >= 0
        int x[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float f[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) x[4 * q + i] = held ? __float2int_rn(ldexpf(f[i], 24 - e)) + kBias : kBias;
        }
#pragma unroll
        for (int j = 0; j < kDigits; ++j) {
            uint32_t c[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) c[i] = e2m3((j == kDigits - 1 ? x[i] >> 20 : (x[i] >> (5 * j)) & 31) - 16);
            const uint32_t w0 = c[0] | c[1] << 6 | c[2] << 12 | c[3] << 18 | c[4] << 24 | c[5] << 30;
            const uint32_t w1 = c[5] >> 2 | c[6] << 4 | c[7] << 10 | c[8] << 16 | c[9] << 22 | c[10] << 28;
            const uint32_t w2 = c[10] >> 4 | c[11] << 2 | c[12] << 8 | c[13] << 14 | c[14] << 20 | c[15] << 26;
            uint32_t* const hi = reinterpret_cast<uint32_t*>(dst + j * kPlane) + 4 * b;
            if (w % 2 == 0) {
                hi[0] = w0;
                hi[1] = w1;
                hi[2] = w2;
            } else {
                hi[3] = w0;
                *reinterpret_cast<uint2*>(dst + j * kPlane + 64 + 8 * b) = make_uint2(w1, w2);
            }
        }
        // the block's power of two against the row's; 255 (NaN) where the
        // block holds an infinity or NaN: its row's results are NaN then, as
        // infinity minus its own high part is in an fp16 split
        if (w % 2 == 0) dst[kScalesAt + b] = finite ? static_cast<uint8_t>(max(kOne + e - er, 0)) : 255u;
    };
    if constexpr (NP > 0) {
#pragma unroll
        for (int j = 0; j < NP; ++j) put(threadIdx.x + 256u * j, keep[j]);
    } else {
        // (whole waves: both halves of a lane block take every pass together)
        for (uint32_t w0 = 0; w0 < units; w0 += 256) {
            const uint32_t w = w0 + threadIdx.x, wc = min(w, units - 1);
            const float4 v[4] = {act4(row, urow, at(wc, 0)), act4(row, urow, at(wc, 1)), act4(row, urow, at(wc, 2)),
                                 act4(row, urow, at(wc, 3))};
            put(w, v);
        }
    }
}

struct Fp6Seg {
    const uint8_t* tiles;  // 6-bit copy
    const float* scales;   // [tile][superblock][16]
    float* out;
    const float* resid;  // with out2: out2 = resid + out (a residual Add), else null
    float* out2;
    uint32_t n, block0;  // first column block
};

struct Fp6Args {
    const uint8_t* records;
    const int* row_exp;
    Fp6Seg seg[kFusedMaxSegs];
    uint32_t nseg, m, sb_total, rows, cols;  // rows, cols: row and column blocks
    uint32_t slices;                         // k cut into this many slices of whole superblocks
    // slices > 1: slice z's sums at partial + z slice_floats, the weights'
    // m x n one after the other
    float* partial;
    uint64_t slice_floats;
};

// A load of 4, 8 or 16 bytes at a global address.
template <typename T>
__device__ __forceinline__ T load_at(__attribute__((address_space(1))) const uint8_t* p) {
    typedef uint32_t words __attribute__((ext_vector_type(sizeof(T) / 4)));
    const words v = *(__attribute__((address_space(1))) const words*)p;
    return __builtin_bit_cast(T, v);
}

// A block's waves are WM x WN, each 16 MT rows by 16 NT columns. At most 256
// registers a wave (two per SIMD): with more allowed, the compiler keeps the
// digit sums in accumulation registers and moves each out before the vector
// unit can add it, 128 moves in a 64 x 256 tile's pass (396 -> 360 us).
template <int MT, int NT, int WM, int WN>
__global__ __launch_bounds__(kWave* WM* WN) __attribute__((amdgpu_waves_per_eu(2))) void qgemm_fp6(Fp6Args p) {
    constexpr int T = kWave * WM * WN;
    constexpr uint32_t BM = 16 * MT * WM, BN = 16 * NT * WN;
    constexpr int NL = BM * 32 / T;  // 16-byte pieces of a stage per thread
    static_assert(NL * T == BM * 32, "whole pieces per thread");
    prefetch_kernarg<arg_bytes<Fp6Args>()>();
    __shared__ __align__(16) uint8_t as[2][BM * kLdsRow];
    const uint32_t tid = threadIdx.x, lane = tid % kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), wm = wave / WN, wn = wave % WN;
    // Blocks go to the 8 XCDs round robin; each XCD takes a contiguous run of
    // column blocks, row blocks innermost, so that its L2 reads a weight once
    // for all the row blocks it runs together.
    const uint32_t total = gridDim.x, xcd = blockIdx.x % 8, per = total / 8, rem = total % 8;
    const uint32_t lin = xcd * per + min(xcd, rem) + blockIdx.x / 8;
    // (run-time divisions leave their results in vector registers)
    const auto uniform = [](uint32_t v) -> uint32_t { return __builtin_amdgcn_readfirstlane(v); };
    const uint32_t by = uniform(lin % p.rows), bxz = uniform(lin / p.rows);
    const uint32_t bx = uniform(bxz % p.cols), bz = uniform(bxz / p.cols);
    const uint32_t si = (p.nseg > 1 && bx >= p.seg[1].block0 ? 1u : 0u) + (p.nseg > 2 && bx >= p.seg[2].block0 ? 1u : 0u);
#define SL_GSEG(f) (si == 0 ? p.seg[0].f : si == 1 ? p.seg[1].f : p.seg[2].f)
    const uint32_t n = SL_GSEG(n), n_tiles = (n + 15) / 16;
    const uint32_t m0 = by * BM, n0 = (bx - SL_GSEG(block0)) * BN;
    const uint32_t beg = uniform(bz * p.sb_total / p.slices), end = uniform((bz + 1) * p.sb_total / p.slices);

    struct Stage {
        uint4 v[NL];
    };
    struct Weights {
        uint4 lo[NT];
        uint2 hi[NT];
        float s[NT];
    };
    uint32_t src[NL];  // byte offsets of this thread's pieces: piece tid % 32 of rows tid / 32 + T / 32 i
#pragma unroll
    for (int i = 0; i < NL; ++i)
        src[i] = (min(m0 + tid / 32 + T / 32 * i, p.m - 1) * p.sb_total * (kRecord / 16) + tid % 32) * 16;
    // A uniform base that stays in scalar registers plus a 32-bit lane offset
    // per load: left to itself the compiler keeps one 64-bit vector address
    // per load.
    typedef __attribute__((address_space(1))) const uint8_t global_u8;
    const auto scalar = [](const void* q) -> global_u8* {
        global_u8* r = (global_u8*)q;
        asm volatile("" : "+s"(r));
        return r;
    };
    const uint8_t* wt[NT];
    const float* ws[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const uint64_t t = static_cast<uint64_t>(min(n0 / 16 + wn * NT + j, n_tiles - 1)) * p.sb_total;
        wt[j] = SL_GSEG(tiles) + t * kTileBytes;
        ws[j] = SL_GSEG(scales) + t * 16;
    }
    const uint32_t lane16 = lane * 16, lane8 = lane * 8, col4 = lane % 16 * 4;
    auto load_stage = [&](uint32_t sb) -> Stage {
        Stage r;
        global_u8* const base = scalar(p.records + static_cast<uint64_t>(sb) * kRecord);
#pragma unroll
        for (int i = 0; i < NL; ++i) r.v[i] = load_at<uint4>(base + src[i]);
        return r;
    };
    auto load_weights = [&](uint32_t sb) -> Weights {
        Weights r;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            global_u8* const base = scalar(wt[j] + static_cast<uint64_t>(sb) * kTileBytes);
            r.lo[j] = load_at<uint4>(base + lane16);
            r.hi[j] = load_at<uint2>(base + 1024 + lane8);
            r.s[j] = load_at<float>(scalar(ws[j] + static_cast<uint64_t>(sb) * 16) + col4);
        }
        return r;
    };
    struct Digit {
        uint4 lo;
        uint2 hi;
    };
    auto row_of = [&](uint32_t buf, int i) -> const uint8_t* {
        return &as[buf][(16 * (wm * MT + i) + lane % 16) * kLdsRow];
    };
    auto read_digit = [&](uint32_t buf, int q) -> Digit {  // digit q % kDigits of row tile q / kDigits
        const uint8_t* const at = row_of(buf, q / kDigits) + q % kDigits * kPlane;
        return Digit{*reinterpret_cast<const uint4*>(at + 16 * (lane / 16)),
                     *reinterpret_cast<const uint2*>(at + 64 + 8 * (lane / 16))};
    };
    auto read_scale = [&](uint32_t buf, int i) -> int { return row_of(buf, i)[kScalesAt + lane / 16]; };
    constexpr int kArithmetic = 0xF, kAhead = 1;
    auto store_stage = [&](uint32_t buf, const Stage r) {
#pragma unroll
        for (int i = 0; i < NL; ++i)
            *reinterpret_cast<uint4*>(&as[buf][(tid / 32 + T / 32 * i) * kLdsRow + tid % 32 * 16]) = r.v[i];
    };

    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    // One superblock with weights w; returns the next one's.
    auto pass = [&](uint32_t sb, const Weights w) -> Weights {
        const uint32_t buf = (sb - beg) & 1;
        // past the end the last superblock again: every pass issues the same loads
        const uint32_t nx = min(sb + 1, end - 1);
        const Stage st = load_stage(nx);
        const Weights wx = load_weights(nx);
        // Digits are read kAhead steps before their products. (The barriers
        // let arithmetic pass and hold memory operations: left alone, the
        // compiler sinks every load to just before its use.)
        __builtin_amdgcn_sched_barrier(kArithmetic);
        Digit ring[kAhead + 1];
        int scale[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) scale[i] = read_scale(buf, i);
#pragma unroll
        for (int q = 0; q < kAhead; ++q) ring[q] = read_digit(buf, q);
        v4f lo[NT], hi[NT];
#pragma unroll
        for (int q = 0; q < MT * kDigits; ++q) {
            if (q + kAhead < MT * kDigits) ring[(q + kAhead) % (kAhead + 1)] = read_digit(buf, q + kAhead);
            __builtin_amdgcn_sched_barrier(kArithmetic);
            const int i = q / kDigits, d = q % kDigits;
            const Digit x = ring[q % (kAhead + 1)];
            const v8i av = {static_cast<int>(x.lo.x), static_cast<int>(x.lo.y), static_cast<int>(x.lo.z),
                            static_cast<int>(x.lo.w), static_cast<int>(x.hi.x), static_cast<int>(x.hi.y), 0, 0};
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const v8i bv = {static_cast<int>(w.lo[j].x), static_cast<int>(w.lo[j].y),
                                static_cast<int>(w.lo[j].z), static_cast<int>(w.lo[j].w),
                                static_cast<int>(w.hi[j].x), static_cast<int>(w.hi[j].y), 0, 0};
                v4f& t = d < kLowDigits ? lo[j] : hi[j];
                const v4f c = d == 0 || d == kLowDigits ? v4f{0.f, 0.f, 0.f, 0.f} : t;
                t = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 2, 2, 0, scale[i], 0,
                                                                     kOne + 5 * (d - (kDigits - 1)));
            }
            if (d == kDigits - 1)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j][e] = fmaf(hi[j][e] + lo[j][e], w.s[j], acc[i][j][e]);
        }
        store_stage(buf ^ 1, st);
        __syncthreads();
        return wx;
    };
    Weights w0 = load_weights(beg);
    store_stage(0, load_stage(beg));
    __syncthreads();
    // two passes per iteration: the weights' registers alternate, not moved
    uint32_t sb = beg;
    for (; sb + 1 < end; sb += 2) {
        const Weights w1 = pass(sb, w0);
        w0 = pass(sb + 1, w1);
    }
    if (sb < end) pass(sb, w0);

    // accumulator value e of lane l: row 4 (l / 16) + e, column l % 16 of its
    // tile; (d / 8) (q / 8) 2^(E - Erow) 32^(j - 4) against d q 32^j 2^(E - 24)
    float* const out = SL_GSEG(out);
    const float* const resid = SL_GSEG(resid);
    float* const out2 = SL_GSEG(out2);
    const uint64_t before = si == 0 ? 0 : p.seg[0].n + (si == 1 ? 0 : p.seg[1].n);  // columns of earlier weights
    float* const part = p.slices > 1 ? p.partial + bz * p.slice_floats + before * p.m : nullptr;
#undef SL_GSEG
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t row = m0 + 16 * (wm * MT + i) + 4 * (lane / 16) + e;
            if (row >= p.m) continue;
            const int sh = p.row_exp[row] + 2;
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const uint32_t col = n0 + 16 * (wn * NT + j) + lane % 16;
                if (col >= n) continue;
                const uint64_t o = static_cast<uint64_t>(row) * n + col;
                const float val = ldexpf(acc[i][j][e], sh);
                if (p.slices > 1) {
                    part[o] = val;
                    continue;
                }
                if (out != nullptr) out[o] = val;
                if (out2 != nullptr) out2[o] = resid[o] + val;
            }
        }
}

struct RecordLayout {
    uint64_t exp_at, floats;
};
RecordLayout record_layout(uint64_t m, uint64_t k) {
    const uint64_t exp_at = m * (k / 128) * (kRecord / 4);
    return {exp_at, exp_at + m};
}

template <int MT, int NT, int WM, int WN>
hipError_t run_gemm(Fp6Args& p, hipStream_t s) {
    constexpr uint32_t BM = 16 * MT * WM, BN = 16 * NT * WN;
    p.rows = (p.m + BM - 1) / BM;
    p.cols = 0;
    for (uint32_t i = 0; i < p.nseg; ++i) {
        p.seg[i].block0 = p.cols;
        p.cols += (p.seg[i].n + BN - 1) / BN;
    }
    qgemm_fp6<MT, NT, WM, WN><<<p.rows * p.cols * p.slices, kWave * WM * WN, 0, s>>>(p);
    return hipGetLastError();
}

// Measured with [28672 x 4096], [4096 x 14336] and [4096 x 4096] at M = 20 to
// 1024. Larger tiles read the activations' digits and the weights less often
// per product (0.74 us per 32 x 256 outputs in 128 x 256 tiles, 0.81, 0.86 and
// 1.04 in the others); smaller ones reach every CU with fewer rows.
// [4096 x 14336] at M = 77: 39 us in 32 x 128 tiles and 8 slices, 204 in 64 x
// 256 ones and one; at M = 1024 225 us in 64 x 256 and 4 slices, 201 in 128 x
// 256 and 2; [4096 x 4096] at M = 512 48 us in 64 x 256 and 4 slices, 96 in 128
// x 256 and one.
constexpr GemmShape kShapes[] = {{128, 256, 1, {2.95f}},
                                 {64, 256, 2, {1.8f, 2.9f}},
                                 {32, 256, 2, {1.1f, 1.72f}},
                                 {32, 128, 4, {0.7f, 1.1f, 1.6f, 2.07f}}};

}  // namespace

uint64_t quant_fp6_bytes(uint32_t format, uint64_t n, uint64_t k, uint32_t group, QuantLayout layout) {
    if (layout != QuantLayout::Mfma || format != SL_QFORMAT_INT4 || group % 128 != 0) return 0;
    return (n + 15) / 16 * (k / 128) * kTileBytes;
}

hipError_t launch_fp6_repack(const uint8_t* payload, uint8_t* tiles, uint64_t n, uint64_t k, hipStream_t s) {
    const uint64_t units = (n + 15) / 16 * (k / 128) * 2 * kWave;
    if (units == 0) return hipSuccess;
    repack_fp6<<<grid_for(units, 256, 256 * 64), 256, 0, s>>>(payload, reinterpret_cast<uint32_t*>(tiles), n, k, units);
    return hipGetLastError();
}

bool qgemm_fp6_takes(const float* a, const QuantWeight* const* w, uint32_t nseg, uint64_t m, const Workspace& ws) {
    if (nseg == 0 || nseg > kFusedMaxSegs || !aligned16(a) || m == 0 || m > 0xffffffull) return false;
    uint64_t n = 0;
    for (uint32_t i = 0; i < nseg; ++i) {
        const QuantWeight& x = *w[i];
        if (x.fp6 == nullptr || x.tile_scales == nullptr || x.k != w[0]->k || x.k > 0xffffffull || x.n == 0 ||
            x.n > 0xffffffull)
            return false;
        n += x.n;
    }
    // byte offsets of the records in 32 bits
    return m * (w[0]->k / 128) * kRecord <= 0xffffffffull && m * n <= 0xffffffffffull &&
           record_layout(m, w[0]->k).floats <= ws.floats;
}

hipError_t launch_qgemm_fp6(const float* a, const QuantWeight* const* w, float* const* out, uint32_t nseg, uint64_t m,
                            const Workspace& ws, hipStream_t s, const float* u, const float* const* resid,
                            float* const* out2, const float* gamma, float eps) {
    if (!qgemm_fp6_takes(a, w, nseg, m, ws)) return hipErrorNotSupported;
    const uint64_t k = w[0]->k;
    if (gamma != nullptr && (u != nullptr || !qgemm_norm_takes(k, gamma))) return hipErrorNotSupported;
    const RecordLayout lay = record_layout(m, k);
    uint8_t* const records = reinterpret_cast<uint8_t*>(ws.data);
    int* const row_exp = reinterpret_cast<int*>(ws.data + lay.exp_at);
    const uint32_t kk = static_cast<uint32_t>(k);
    const unsigned rows = static_cast<unsigned>(m);
    if (k <= 4096) split_fp6<1><<<rows, 256, 0, s>>>(a, u, records, row_exp, kk, gamma, eps);
    else if (k <= 8192) split_fp6<2><<<rows, 256, 0, s>>>(a, u, records, row_exp, kk, gamma, eps);
    else if (k <= 16384) split_fp6<4><<<rows, 256, 0, s>>>(a, u, records, row_exp, kk, nullptr, 0.f);
    else split_fp6<0><<<rows, 256, 0, s>>>(a, u, records, row_exp, kk, nullptr, 0.f);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    Fp6Args p{};
    p.records = records;
    p.row_exp = row_exp;
    p.nseg = nseg;
    p.m = static_cast<uint32_t>(m);
    p.sb_total = kk / 128;
    uint64_t n_total = 0, n[kFusedMaxSegs] = {};
    for (uint32_t i = 0; i < nseg; ++i) {
        const bool res = resid != nullptr && out2 != nullptr && out2[i] != nullptr;
        p.seg[i] = Fp6Seg{w[i]->fp6, w[i]->tile_scales, out[i], res ? resid[i] : nullptr, res ? out2[i] : nullptr,
                          static_cast<uint32_t>(w[i]->n), 0u};
        n[i] = w[i]->n;
        n_total += n[i];
    }
    const uint64_t part_at = (lay.floats + 63) / 64 * 64;
    const GemmChoice best =
        choose_gemm(kShapes, n, nseg, m, p.sb_total, part_at < ws.floats ? ws.floats - part_at : 0,
                    [](uint32_t) { return true; });
    const size_t shape = best.shape;
    p.slices = best.slices;
    p.partial = p.slices > 1 ? ws.data + part_at : nullptr;
    p.slice_floats = m * n_total;
    if (shape == 0) e = run_gemm<4, 4, 2, 4>(p, s);
    else if (shape == 1) e = run_gemm<4, 4, 1, 4>(p, s);
    else if (shape == 2) e = run_gemm<2, 4, 1, 4>(p, s);
    else e = run_gemm<2, 2, 1, 4>(p, s);
    if (e != hipSuccess || p.slices == 1) return e;
    SliceSum sum{};
    sum.partial = p.partial;
    sum.slice_floats = p.slice_floats;
    sum.m = m;
    sum.slices = p.slices;
    for (uint32_t i = 0; i < nseg; ++i)
        sum.seg[i] = SliceSeg{w[i]->n, p.seg[i].out, p.seg[i].resid, p.seg[i].out2};
    return launch_slices_sum(sum, s);
}

// Loads this file's code object now: HIP loads one at the first use of
// any of its kernels, which otherwise lands inside the first submission
// that needs it (about 1-2 ms each, more for large objects).
hipError_t load_code_qgemm_fp6() {
    hipFuncAttributes attr;
    return hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&split_fp6<0>));
}

}  // namespace slhip
