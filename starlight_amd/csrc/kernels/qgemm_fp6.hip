// Group-quantized MatMulNT for many activation rows (prefill) with INT4
// weights, on the block-scaled 6-bit matrix cores:
// out[m, n] = sum_k a[m, k] * (q[n, k] * s[n, k / G]), G a multiple of 128.
//
// Exactness plan. E2M3, the 6-bit float of v_mfma_scale_f32_16x16x128_f8f6f4,
// holds every integer of magnitude at most 16 exactly (as n / 8, with the
// sign-magnitude code n itself), so an INT4 code is one E2M3 value. Of every
// activation row, each 32 elements that one lane feeds to a product share an
// exponent E (|a| < 2^E) and become integers X = rint(a * 2^(29 - E)), cut
// into six signed base-32 digits, X = sum_j d_j 32^j with |d_j| <= 16, each
// one E2M3 value as well: 29 bits below 2^E. A block most of whose elements
// (17 or more nonzero ones) lie below 2^(E - 8), under an outlier channel for
// instance, gets two more digits, 39 bits. So an element keeps at least the 22
// bits it has as two fp16 parts (qgemm_mfma.hip), or the block's small ones do
// statistically: with five digits a channel at 1,000 times the others, in each
// 32 and under zero codes, left those an error of 2e-5. The products d_j * q
// are exact, and the instruction's block scales carry 2^E (relative to the
// row's largest exponent) and 32^j. A product's sum over its 128 k is exact
// where the blocks' exponents are close, but adding it to a larger sum cuts
// that downwards by up to 2^-23 of it: chained over all digits, the errors of
// a whole model's logits grew 1.2 to 2.4 times. So the four low digits and the
// two high ones are summed apart (the high sum needs 20 bits plus the
// exponents' spread), added in f32, multiplied by the group's scale, added to
// the f32 result, and that is scaled back by the row's exponent at the end.
//
// Error against float64, normwise, fp16 split / this: activations normal, silu
// of a normal times another, Student t with 3 and 2 degrees, cubed Laplace, one
// channel or one in each 32 at 30 to 100,000 times the others with and without
// codes under it: k = 512 1.1e-7 to 1.8e-7 / 4.6e-8 to 7.6e-8, k = 4096 1.3e-7
// to 2.7e-7 / 7.3e-8 to 9.6e-8, k = 14336 1.7e-7 to 3.2e-7 / 9.0e-8 to 1.2e-7.
//
// Rate. Register-resident loops on MI355X reach 8.43 PFLOP/s with 6-bit
// operands and 2.17 PFLOP/s with fp16 ones: six 6-bit products per multiply
// allow 1.41 PFLOP/s of f32 result, two fp16 ones 1.08. With the split, against
// the fp16 route (and five digits): [28672 x 4096] M = 1024 398 us against 525
// (355; 604 TFLOP/s of f32 result), M = 77 65 against 89 (58); [4096 x 14336] M =
// 1024 238 against 304 (213), M = 512 130 against 186 (117), M = 77 46 against
// 159 (41); [4096 x 4096] M = 77 26 against 56 (25). What bounds it now: vector
// and matrix instructions of a SIMD's waves do not overlap here, and a 64 x 256
// tile's pass has 96 products (1,536 cycles) and 178 vector instructions (712)
// per wave, two waves per SIMD: 4,500 of 5,830 cycles measured (at 1.9 GHz); LDS
// is busy for 2,370 of them (reads of the digits, and the stage's writes in the
// middle of the pass: at its end, 1-2% slower; loads straight into LDS the same
// time as through registers). Deeper operand prefetch and wave priorities
// changed nothing, and gathering the records in operand order from memory (no
// LDS conflicts, scattered 64-byte loads) was slower. A sixth digit only for
// blocks that need it costs as much where they are few (the LDS room and the
// branch) and more behind silu(g) * u, where nearly every tile has one.
//
// Kernels
//  * repack_fp6 (bind): the codes as E2M3 in operand order, per 16-row tile
//    and 128-k superblock 64 lanes x 16 bytes, then 64 lanes x 8 bytes. Lane
//    l holds row l % 16 and the elements k = 16 (i / 4) + 4 (l / 16) + i % 4,
//    i < 32, of the superblock (the order in which a quad of threads reads
//    whole float4 of the activations);
//  * split_fp6: one block per row: row maximum, block exponents, digits. A
//    record of 592 bytes per superblock and row: six digit planes of 4 lanes
//    x 16 then 4 x 8 bytes, and four block scales with the flag of further
//    digits, which lie in planes of their own;
//  * qgemm_fp6: a block's rows of a superblock, contiguous, staged through LDS
//    as they are (592 bytes a row: the 16 rows of one operand read begin 20
//    banks apart, no two on the same 4; rows of 640 bytes: 400 -> 480 us), shared
//    by the block's waves; weights straight from memory into registers, one
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

constexpr int kDigits = 6, kLowDigits = 4;    // digits of every element, and of the low sum
constexpr int kMoreDigits = 2;                // of a block whose maximum stands far above most of it
constexpr int kFar = 8;                       // powers of two that is
constexpr uint32_t kPlane = 96;               // bytes of one digit of a row and superblock
constexpr uint32_t kScalesAt = kDigits * kPlane;  // 16 bits per lane: block scale, kFurther
constexpr int kFurther = 256;
constexpr uint32_t kRecord = 592;                 // bytes per row and superblock, also of its row in LDS
constexpr uint32_t kMore = kMoreDigits * kPlane;  // bytes of the further digits of a row and superblock
static_assert(kScalesAt + 8 <= kRecord && kRecord % 16 == 0, "record layout");
constexpr uint32_t kTileBytes = 1536;           // one 16-row weight tile of one superblock
constexpr uint32_t kPad = 128 * kRecord + 8192;  // bytes a block's loads may reach past the last record
constexpr int kOne = 127;                       // E8M0 of 1.0

// Sign and magnitude of d, |d| <= 16: the E2M3 code of d / 8.
__device__ __forceinline__ uint32_t e2m3(int d) {
    return static_cast<uint32_t>(max(d, -d)) | (static_cast<uint32_t>(d >> 26) & 32u);
}

// The same of digit j of x, a sum of 32^j (d_j + 16) with every d_j + 16 < 32
// but the highest's (4 instructions, not 7: digits are most of the split's).
__device__ __forceinline__ uint32_t digit(int x, int j, bool highest) {
    const uint32_t u = static_cast<uint32_t>(x);
    if (highest) return e2m3(static_cast<int>(u >> (5 * j)) - 16);
    const uint32_t sign = j == 0 ? ~u << 1 : ~u >> (5 * j - 1);
    return __builtin_amdgcn_sad_u8(u >> (5 * j) & 31u, 16u, 0u) | (sign & 32u);
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
// digits and by its reads; M = 1024: k = 4096 12.3 us, silu(a) * u at k = 14336
// 53 (174 MB read and written, 3.3 TB/s, with two waves per SIMD).
template <int NP>
__global__ __launch_bounds__(256) void split_fp6(const float* __restrict__ a, const float* __restrict__ u,
                                                 uint8_t* __restrict__ records, uint8_t* __restrict__ more,
                                                 int* __restrict__ row_exp, uint32_t k,
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
    const uint64_t m = gridDim.x;
    // The records a last block reads past the last superblock's (up to 127, in
    // kPad) hold what was there before: without further digits, or they would
    // choose how the rows beside them are summed.
    if (r == m - 1 && threadIdx.x < 128)
        *reinterpret_cast<uint2*>(records + (k / 128 * m + threadIdx.x) * kRecord + kScalesAt) = make_uint2(0u, 0u);
    // One plane of 16 elements' codes: half h of lane block b.
    const auto store = [](uint8_t* plane, uint32_t h, uint32_t b, const uint32_t (&c)[16]) {
        const uint32_t w0 = c[0] | c[1] << 6 | c[2] << 12 | c[3] << 18 | c[4] << 24 | c[5] << 30;
        const uint32_t w1 = c[5] >> 2 | c[6] << 4 | c[7] << 10 | c[8] << 16 | c[9] << 22 | c[10] << 28;
        const uint32_t w2 = c[10] >> 4 | c[11] << 2 | c[12] << 8 | c[13] << 14 | c[14] << 20 | c[15] << 26;
        uint32_t* const hi = reinterpret_cast<uint32_t*>(plane) + 4 * b;
        if (h == 0) {
            hi[0] = w0;
            hi[1] = w1;
            hi[2] = w2;
        } else {
            hi[3] = w0;
            *reinterpret_cast<uint2*>(plane + 64 + 8 * b) = make_uint2(w1, w2);
        }
    };
    // Unit w's digits; its lane block's other half is in the neighbouring thread.
    auto put = [&](uint32_t w, const float4 (&v)[4]) {
        uint32_t mx32 = max(max(mag4(v[0]), mag4(v[1])), max(mag4(v[2]), mag4(v[3])));
        mx32 = max(mx32, static_cast<uint32_t>(dpp_i<kDppXor1>(static_cast<int>(mx32))));
        // (a block of zeros takes the row's exponent: 0 would lie 127 and more
        // above that of a row of denormals, where the scale's byte is NaN's)
        const int e = mx32 != 0 ? mag_exp(mx32) : er;
        const bool finite = mx32 < 0x7f800000u;
        float f[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) f[4 * q] = v[q].x, f[4 * q + 1] = v[q].y, f[4 * q + 2] = v[q].z, f[4 * q + 3] = v[q].w;
        // (of its 32 elements, 17 or more nonzero and below 2^(e - kFar))
        const uint32_t least = max(__float_as_uint(ldexpf(1.0f, e - kFar)), 1u) - 1u;
        int small = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) small += (__float_as_uint(f[i]) & 0x7fffffffu) - 1u < least ? 1 : 0;
        small += dpp_i<kDppXor1>(small);
        if (w >= units) return;
        const bool held = finite && kOne + e - er >= 0;  // else below what a block scale can say: zero digits
        const bool further = held && small > 16;
        const uint32_t h = w % 2, b = w / 2 % 4;
        const uint64_t at = w / 8 * m + r;
        uint8_t* const dst = records + at * kRecord;
        constexpr int kBias = 16 * (1 + 32 + 1024 + 32768 + 1048576 + 33554432);  // makes every digit d + 16 >= 0
        int x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = held ? __float2int_rn(ldexpf(f[i], 29 - e)) + kBias : kBias;
#pragma unroll
        for (int j = 0; j < kDigits; ++j) {
            uint32_t c[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) c[i] = digit(x[i], j, j == kDigits - 1);
            store(dst + j * kPlane, h, b, c);
        }
        // the block's power of two against the row's; 255 (NaN) where the
        // block holds an infinity or NaN: its row's results are NaN then, as
        // infinity minus its own high part is in an fp16 split
        if (h == 0)
            reinterpret_cast<uint16_t*>(dst + kScalesAt)[b] =
                static_cast<uint16_t>((finite ? max(kOne + e - er, 0) : 255) | (further ? kFurther : 0));
        if (further) {
            // what the digits leave, at most half a unit (exact: a value
            // of 2^24 units or more is whole), in 1024ths of it: |.| <= 512
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float t = ldexpf(f[i], 29 - e);
                x[i] = __float2int_rn((t - rintf(t)) * 1024.0f) + 16 * (1 + 32);
            }
#pragma unroll
            for (int j = 0; j < kMoreDigits; ++j) {
                uint32_t c[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) c[i] = e2m3((j == kMoreDigits - 1 ? x[i] >> 5 : x[i] & 31) - 16);
                store(more + at * kMore + j * kPlane, h, b, c);
            }
        }
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
    const uint8_t* records;  // [superblock][row]
    const uint8_t* more;     // the same, written where a block has further digits
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
__global__ __launch_bounds__(kWave* WM* WN) __attribute__((amdgpu_waves_per_eu(MT * NT <= 4 ? 4 : 2))) void qgemm_fp6(Fp6Args p) {
    constexpr int T = kWave * WM * WN;
    constexpr uint32_t BM = 16 * MT * WM, BN = 16 * NT * WN;
    // 16-byte pieces of a stage per thread, the last ones past its BM rows (kPad)
    constexpr int NL = (BM * (kRecord / 16) + T - 1) / T;
    static_assert(NL * T * 16 <= kPad, "a whole stage past the last record");
    prefetch_kernarg<arg_bytes<Fp6Args>()>();
    constexpr uint32_t kBuf = NL * T * 16;
    __shared__ __align__(16) uint8_t as[2 * kBuf];
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
    const uint32_t tid16 = tid * 16, lane16 = lane * 16, lane8 = lane * 8, col4 = lane % 16 * 4;
    auto load_stage = [&](uint32_t sb) -> Stage {
        Stage r;
        // (rows past m are the next superblock's, or kPad: computed, not stored)
        const uint8_t* const rec = p.records + (static_cast<uint64_t>(sb) * p.m + m0) * kRecord;
#pragma unroll
        for (int i = 0; i < NL; ++i) r.v[i] = load_at<uint4>(scalar(rec + T * 16 * i) + tid16);
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
    const auto operand = [](const Digit x) -> v8i {
        return v8i{static_cast<int>(x.lo.x), static_cast<int>(x.lo.y), static_cast<int>(x.lo.z),
                   static_cast<int>(x.lo.w), static_cast<int>(x.hi.x), static_cast<int>(x.hi.y), 0, 0};
    };
    // LDS addresses: one register per use that the pass's buffer is added to,
    // the rest as the instructions' 16-bit offsets (both buffers' addresses as
    // constants do not fit those and took 34 registers more than there are)
    const auto opaque = [](uint32_t v) -> uint32_t {
        asm volatile("" : "+v"(v));
        return v;
    };
    const uint32_t row0 = (16 * wm * MT + lane % 16) * kRecord;
    auto read_plane = [&](uint32_t at16, uint32_t at8, int i, int plane) -> Digit {  // of row tile i
        const uint32_t o = i * 16 * kRecord + plane * kPlane;
        return Digit{*reinterpret_cast<const uint4*>(as + at16 + o), *reinterpret_cast<const uint2*>(as + at8 + o)};
    };
    constexpr int kArithmetic = 0xF, kAhead = 1;
    auto store_piece = [&](uint32_t at, const Stage& r, int i) { *reinterpret_cast<uint4*>(as + at + T * 16 * i) = r.v[i]; };

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
        const uint32_t row = row0 + buf * kBuf, at16 = opaque(row + 16 * (lane / 16)),
                       at8 = opaque(row + 64 + 8 * (lane / 16)), at2 = row + kScalesAt + 2 * (lane / 16);
#pragma unroll
        for (int i = 0; i < MT; ++i) scale[i] = *reinterpret_cast<const uint16_t*>(as + at2 + i * 16 * kRecord);
#pragma unroll
        for (int q = 0; q < kAhead; ++q) ring[q] = read_plane(at16, at8, q / kDigits, q % kDigits);
        const auto product = [&](const Digit x, int j, const v4f c, int scale_a, int e) -> v4f {
            return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(operand(x), operand(Digit{w.lo[j], w.hi[j]}), c, 2, 2,
                                                                    0, scale_a, 0, kOne + e);
        };
        const v4f zero = {0.f, 0.f, 0.f, 0.f};
        // With further digits anywhere, the whole pass is left to its end (below)
        // and adds nothing here.
        int flags = scale[0];
#pragma unroll
        for (int i = 1; i < MT; ++i) flags |= scale[i];
        const bool wide = __builtin_amdgcn_ballot_w64(flags >= kFurther) != 0;  // wave-uniform
        float here[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) here[j] = wide ? 0.f : w.s[j];
        const uint32_t to = opaque(tid16 + (buf ^ 1) * kBuf);
        v4f lo[NT], hi[NT];
#pragma unroll
        for (int q = 0; q < MT * kDigits; ++q) {
            // the next stage's pieces, in the middle of the pass
            if (const int a = q - (MT * kDigits - NL) / 2; a >= 0 && a < NL) store_piece(to, st, a);
            if (const int a = q + kAhead; a < MT * kDigits)
                ring[a % (kAhead + 1)] = read_plane(at16, at8, a / kDigits, a % kDigits);
            __builtin_amdgcn_sched_barrier(kArithmetic);
            const int i = q / kDigits, d = q % kDigits;
            const Digit x = ring[q % (kAhead + 1)];
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                v4f& t = d < kLowDigits ? lo[j] : hi[j];
                t = product(x, j, d == 0 || d == kLowDigits ? zero : t, scale[i], 5 * (d - (kDigits - 1)));
            }
            if (d == kDigits - 1)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j][e] = fmaf(hi[j][e] + lo[j][e], here[j], acc[i][j][e]);
        }
        // Further digits: elements of a block 2^8 and more apart. The sum of a
        // plane is still exact or close, the four low planes' together is not, and
        // is cut always downwards (a bias of 5e-7 over 129 superblocks), so each
        // plane starts from zero here and f32 additions, which round to nearest,
        // join them from the lowest on. (A row past m may show a row's flag of
        // the next superblock: it reads row m - 1's further digits and stores
        // nothing.)
        if (wide) {
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                v4f sum[NT];
#pragma unroll
                for (int j = 0; j < NT; ++j) sum[j] = zero;
#pragma unroll 1
                for (int d = -kMoreDigits; d < kDigits; ++d) {
                    Digit x{make_uint4(0u, 0u, 0u, 0u), make_uint2(0u, 0u)};
                    if (d >= 0) {
                        x = read_plane(at16, at8, i, d);
                    } else if (scale[i] >= kFurther) {
                        const uint32_t l = opaque(lane);  // addresses made here, not kept over the loop
                        const uint32_t r = min(m0 + 16 * (wm * MT + i) + l % 16, p.m - 1);
                        const uint8_t* const at = p.more + (static_cast<uint64_t>(sb) * p.m + r) * kMore +
                                                  (d + kMoreDigits) * kPlane + 8 * (l / 16);
                        x = Digit{*reinterpret_cast<const uint4*>(at + 8 * (l / 16)),
                                  *reinterpret_cast<const uint2*>(at + 64)};
                    }
#pragma unroll
                    for (int j = 0; j < NT; ++j) sum[j] += product(x, j, zero, scale[i], 5 * (d - (kDigits - 1)));
                }
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j][e] = fmaf(sum[j][e], w.s[j], acc[i][j][e]);
            }
        }
        __syncthreads();
        return wx;
    };
    Weights w0 = load_weights(beg);
    {
        const Stage st = load_stage(beg);
#pragma unroll
        for (int i = 0; i < NL; ++i) store_piece(tid16, st, i);
    }
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

// Records, then what a last block's loads read past them, the further
// digits, and the row exponents, in the workspace.
struct RecordLayout {
    uint64_t more_at, exp_at, floats;
};
RecordLayout record_layout(uint64_t m, uint64_t k) {
    const uint64_t records = m * (k / 128);
    const uint64_t more_at = (records * kRecord + kPad) / 4, exp_at = more_at + records * (kMore / 4);
    return {more_at, exp_at, exp_at + m};
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

// Measured at k = 8192 with 1 to `most` blocks on every CU (3.75, 2.27 / 3.40,
// 1.32 / 1.79, 0.88 / 1.16 / 1.76 / 2.22 us); the large tiles' full figures a
// little lower, as whole products show them ([28672 x 4096] at M = 512 and 1024:
// 3.2 and 2.94 us of two 64 x 256 blocks). Larger tiles read the activations'
// digits and the weights less often per product; smaller ones reach every CU
// with fewer rows. [4096 x 14336] at M = 200: 70 us in 32 x 256 tiles and 4
// slices, 76 in 64 x 256 and 8; [4096 x 4096] at M = 200 33 us in 32 x 256 and 4,
// 38 in 32 x 128 and one.
constexpr GemmShape kShapes[] = {{128, 256, 1, {3.6f}},
                                 {64, 256, 2, {2.27f, 3.3f}},
                                 {32, 256, 2, {1.32f, 1.79f}},
                                 {32, 128, 4, {0.88f, 1.16f, 1.76f, 2.22f}}};

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
    return m * n <= 0xffffffffffull &&
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
    uint8_t* const more = reinterpret_cast<uint8_t*>(ws.data + lay.more_at);
    int* const row_exp = reinterpret_cast<int*>(ws.data + lay.exp_at);
    const uint32_t kk = static_cast<uint32_t>(k);
    const unsigned rows = static_cast<unsigned>(m);
    if (k <= 4096) split_fp6<1><<<rows, 256, 0, s>>>(a, u, records, more, row_exp, kk, gamma, eps);
    else if (k <= 8192) split_fp6<2><<<rows, 256, 0, s>>>(a, u, records, more, row_exp, kk, gamma, eps);
    else if (k <= 16384) split_fp6<4><<<rows, 256, 0, s>>>(a, u, records, more, row_exp, kk, nullptr, 0.f);
    else split_fp6<0><<<rows, 256, 0, s>>>(a, u, records, more, row_exp, kk, nullptr, 0.f);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    Fp6Args p{};
    p.records = records;
    p.more = more;
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
                    [](uint32_t) { return true; }, 64);
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
