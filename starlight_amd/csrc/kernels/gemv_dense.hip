// Dense f32 MatMulNT for few activation rows (decode with unquantized
// weights; reference/matmul.rs:29-59): out[m, n] = sum_k a[m, k] * w[n, k],
// with the fusions of the decode step (up to three weights reading the same
// rows, RMSNorm first, a residual Add or silu(g) * u after).
//
// Bound: HBM, every weight is read once. A 64x64-tile GEMM gives a few rows
// only n / 64 blocks, each walking the whole of k through LDS 16 at a time:
// [2048 x 8192] at M = 1 took 540 us for 67 MB (0.12 TB/s) that way, and takes
// 15.0 us (4.5 TB/s) here; [8192 x 2048] 12.3 us (5.5 TB/s), [2048 x 2048] 5.3,
// [4096 x 4096] at M = 4 15.0, at M = 16 18.7.
//
//  * gemv_dense_rows (M <= 4, m * k <= 16384): the activations sit in LDS
//    (normalised there first when asked), and a wave dots one weight row at
//    a time, 64 lanes x 16 bytes per load. Waves stay resident over several
//    rows, so the prologue is paid once per block. The row's next batch of
//    loads (4 float4 per lane, across rows) is in flight while the current
//    one is multiplied: 16 waves per CU x 8 KB covers the memory latency
//    several times over.
//  * gemv_dense_mfma (m <= 32, or activations larger than that): a block owns
//    16 weight rows and cuts k over its waves; v_mfma_f32_16x16x4_f32 multiplies
//    them with 16 or 32 activation rows, so the vector unit's work does not
//    grow with m. Operands come straight from memory (16 rows x 64 bytes per
//    load, the activations from L2); the waves' sums meet in LDS.
//
// Products and sums are f32: per-lane sums over k, then across lanes (or the
// matrix core's order), a shorter chain of additions than ascending k.
#include "common.h"
#include "kernels.h"

namespace slhip {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kRowsThreads = 512, kRowsWaves = kRowsThreads / kWave;
constexpr uint32_t kRowsMaxFloats = 16384;  // activations in LDS: 64 KB, two blocks per CU
constexpr int kBatch = 4;                   // float4 per lane and weight row in one batch of loads

struct DenseSeg {
    const float* w;
    float* out;
    const float* resid;
    float* out2;
    uint32_t n, unit0;  // rows; first unit (weight row, or 16-row tile) of this weight
};

struct DenseArgs {
    const float* a;
    const float* gamma;
    uint32_t m, k;
    float* normed;
    float eps;
    uint32_t nseg, units;
    DenseSeg seg[kFusedMaxSegs];
};

__device__ __forceinline__ float silu_mul(float g, float u) { return (g * (1.0f / (1.0f + expf(-g)))) * u; }

// M: activation rows (m <= M); AF: float4 of activations per thread; PAIR:
// unit r is row r of both weights, out[0] = silu(g) * u.
template <int M, int AF, bool NORM, bool PAIR>
__global__ __launch_bounds__(kRowsThreads) void gemv_dense_rows(DenseArgs p) {
    prefetch_kernarg<arg_bytes<DenseArgs>()>();
    constexpr int R = PAIR ? 2 : 1;
    extern __shared__ __align__(16) float xs[];  // [m][k]
    __shared__ float runs[AF * kRowsWaves];      // sums of squares of each wave's runs
    const uint32_t tid = threadIdx.x, lane = tid % kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t k4 = p.k / 4, total4 = p.m * k4;

    // activations, then the first batch of weights, then the prologue's work
    const float4* a4 = reinterpret_cast<const float4*>(p.a);
    float4 x[AF], g[NORM ? AF : 1];
#pragma unroll
    for (int i = 0; i < AF; ++i) x[i] = a4[min(tid + kRowsThreads * i, total4 - 1)];
    if constexpr (NORM) {
        const float4* g4 = reinterpret_cast<const float4*>(p.gamma);
#pragma unroll
        for (int i = 0; i < AF; ++i) g[i] = g4[min(tid + kRowsThreads * i, total4 - 1) % k4];
    }

    // This wave's units: first, first + stride, ...; batch b of a unit is
    // float4 columns lane + 64 (kBatch b + j).
    const uint32_t batches = (k4 + kBatch * kWave - 1) / (kBatch * kWave);
    const uint32_t first = blockIdx.x * kRowsWaves + wave, stride = gridDim.x * kRowsWaves;
    struct Regs {
        v4f w[R][kBatch];
    };
    auto seg_of = [&](uint32_t u) -> uint32_t {
        if constexpr (PAIR) return 0u;
        return (p.nseg > 1 && u >= p.seg[1].unit0 ? 1u : 0u) + (p.nseg > 2 && u >= p.seg[2].unit0 ? 1u : 0u);
    };
#define SL_DSEG(s, f) ((s) == 0 ? p.seg[0].f : (s) == 1 ? p.seg[1].f : p.seg[2].f)
    auto load = [&](uint32_t u, uint32_t b) -> Regs {
        Regs r;
        const uint32_t s = seg_of(u);
        const uint64_t row = static_cast<uint64_t>(u - SL_DSEG(s, unit0)) * k4;
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const v4f* w = reinterpret_cast<const v4f*>(PAIR ? p.seg[t].w : SL_DSEG(s, w)) + row;
#pragma unroll
            for (int j = 0; j < kBatch; ++j)
                r.w[t][j] = w[min(lane + kWave * (kBatch * b + j), k4 - 1)];
        }
        return r;
    };
    // (a wave without a unit loads the last one's rows and stores nothing)
    uint32_t u = first, b = 0;
    Regs cur = load(min(u, p.units - 1), 0);

    if constexpr (NORM) {
        // k is a multiple of 256, so a wave's run of 64 float4 lies in one row
#pragma unroll
        for (int i = 0; i < AF; ++i) {
            const float4 v = x[i];
            const float ss = wave_sum(fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, v.w * v.w))));
            if (lane == 0) runs[i * kRowsWaves + wave] = ss;
        }
        __syncthreads();
        const uint32_t per_row = k4 / kWave;
#pragma unroll
        for (int i = 0; i < AF; ++i) {
            const uint32_t run = i * kRowsWaves + wave, row = run / per_row;
            if (row >= p.m) continue;
            float ss = 0.f;
            for (uint32_t q = row * per_row; q < (row + 1) * per_row; ++q) ss += runs[q];
            const float inv = 1.0f / sqrtf(ss / static_cast<float>(p.k) + p.eps);
            float4 v = x[i];
            v.x = (v.x * inv) * g[i].x;
            v.y = (v.y * inv) * g[i].y;
            v.z = (v.z * inv) * g[i].z;
            v.w = (v.w * inv) * g[i].w;
            x[i] = v;
            if (blockIdx.x == 0 && p.normed != nullptr)
                reinterpret_cast<float4*>(p.normed)[tid + kRowsThreads * i] = v;
        }
    }
#pragma unroll
    for (int i = 0; i < AF; ++i)
        if (tid + kRowsThreads * i < total4) reinterpret_cast<float4*>(xs)[tid + kRowsThreads * i] = x[i];
    __syncthreads();

    const v4f* x4 = reinterpret_cast<const v4f*>(xs);
    v4f acc[R][M];
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
        for (int q = 0; q < M; ++q) acc[t][q] = v4f{0.f, 0.f, 0.f, 0.f};
    while (u < p.units) {
        const bool last = b + 1 == batches;
        const uint32_t nu = last ? u + stride : u, nb = last ? 0 : b + 1;
        const Regs next = load(min(nu, p.units - 1), nb);
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const uint32_t c = lane + kWave * (kBatch * b + j);
            if (c < k4) {
#pragma unroll
                for (int q = 0; q < M; ++q) {
                    const v4f xv = x4[min(static_cast<uint32_t>(q), p.m - 1) * k4 + c];
#pragma unroll
                    for (int t = 0; t < R; ++t)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[t][q][e] = fmaf(cur.w[t][j][e], xv[e], acc[t][q][e]);
                }
            }
        }
        if (last) {
            const uint32_t s = seg_of(u);
            const uint32_t row = u - SL_DSEG(s, unit0);
            float val = 0.f;  // lane q: row q's result
#pragma unroll
            for (int q = 0; q < M; ++q) {
                float v[R];
#pragma unroll
                for (int t = 0; t < R; ++t) {
                    v[t] = wave_sum((acc[t][q][0] + acc[t][q][1]) + (acc[t][q][2] + acc[t][q][3]));
                    acc[t][q] = v4f{0.f, 0.f, 0.f, 0.f};
                }
                const float o = PAIR ? silu_mul(v[0], v[R - 1]) : v[0];
                val = lane == static_cast<uint32_t>(q) ? o : val;
            }
            if (lane < p.m) {
                const uint64_t o = static_cast<uint64_t>(lane) * SL_DSEG(s, n) + row;
                SL_DSEG(s, out)[o] = val;
                float* const out2 = SL_DSEG(s, out2);
                if (out2 != nullptr) out2[o] = SL_DSEG(s, resid)[o] + val;
            }
        }
        cur = next;
        u = nu;
        b = nb;
    }
}

// NW waves per block; MT 16-row tiles of activations.
template <int NW, int MT, bool PAIR>
__global__ __launch_bounds__(NW* kWave) void gemv_dense_mfma(DenseArgs p) {
    prefetch_kernarg<arg_bytes<DenseArgs>()>();
    constexpr int R = PAIR ? 2 : 1;
    __shared__ float sums[R][MT][NW][16][17];  // [..][wave][activation row][column]
    const uint32_t tid = threadIdx.x, lane = tid % kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t tile = blockIdx.x;
    const uint32_t s = PAIR ? 0u
                            : (p.nseg > 1 && tile >= p.seg[1].unit0 ? 1u : 0u) +
                                  (p.nseg > 2 && tile >= p.seg[2].unit0 ? 1u : 0u);
    const uint32_t n = SL_DSEG(s, n), col0 = (tile - SL_DSEG(s, unit0)) * 16;
    // 16-k steps of this wave: lane group lane / 16 takes k 4 (lane / 16) .. + 3
    // of a step, so one float4 of each operand feeds four products
    const uint32_t steps = (p.k + 15) / 16, per = (steps + NW - 1) / NW;
    const uint32_t beg = min(wave * per, steps), end = min(beg + per, steps);
    const uint32_t kq = 4 * (lane / 16);
    const float* wrow[R];
#pragma unroll
    for (int t = 0; t < R; ++t)
        wrow[t] = (PAIR ? p.seg[t].w : SL_DSEG(s, w)) + static_cast<uint64_t>(min(col0 + lane % 16, n - 1)) * p.k;
    const float* arow[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) arow[i] = p.a + static_cast<uint64_t>(min(16 * i + lane % 16, p.m - 1)) * p.k;
    struct Regs {
        v4f w[R][kBatch], a[MT][kBatch];
    };
    auto load = [&](uint32_t st) -> Regs {
        Regs r;
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const uint32_t kk = min(16 * (st + j) + kq, p.k - 4);
#pragma unroll
            for (int t = 0; t < R; ++t)
                r.w[t][j] = *reinterpret_cast<const v4f*>(wrow[t] + kk);
#pragma unroll
            for (int i = 0; i < MT; ++i) r.a[i][j] = *reinterpret_cast<const v4f*>(arow[i] + kk);
        }
        return r;
    };
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    v4f acc[R][MT];
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[t][i] = zero;
    Regs cur = load(beg);
    for (uint32_t st = beg; st < end; st += kBatch) {
        const Regs next = load(st + kBatch);
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            // past the slice or the row: both operands zero, so that a stray
            // infinity times zero never forms a NaN
            const bool in = st + j < end && 16 * (st + j) + kq < p.k;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const v4f av = in ? cur.a[i][j] : zero;
#pragma unroll
                for (int t = 0; t < R; ++t) {
                    const v4f wv = in ? cur.w[t][j] : zero;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[e], wv[e], acc[t][i], 0, 0, 0);
                }
            }
        }
        cur = next;
    }
    // accumulator value e of lane l: activation row 4 (l / 16) + e, column l % 16
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) sums[t][i][wave][4 * (lane / 16) + e][lane % 16] = acc[t][i][e];
    __syncthreads();
    for (uint32_t o = tid; o < 256u * MT; o += NW * kWave) {
        const uint32_t i = o / 256, r = o / 16 % 16, c = o % 16, row = 16 * i + r;
        float v[R];
#pragma unroll
        for (int t = 0; t < R; ++t) {
            v[t] = 0.f;
            for (int q = 0; q < NW; ++q) v[t] += sums[t][i][q][r][c];
        }
        if (row >= p.m || col0 + c >= n) continue;
        const float val = PAIR ? silu_mul(v[0], v[R - 1]) : v[0];
        const uint64_t at = static_cast<uint64_t>(row) * n + col0 + c;
        SL_DSEG(s, out)[at] = val;
        float* const out2 = SL_DSEG(s, out2);
        if (out2 != nullptr) out2[at] = SL_DSEG(s, resid)[at] + val;
    }
}
#undef SL_DSEG

bool rows_form(uint64_t m, uint64_t k) { return m <= 4 && m * k <= kRowsMaxFloats; }

template <int M, int AF, bool NORM, bool PAIR>
hipError_t run_rows(const DenseArgs& p, unsigned grid, size_t lds, hipStream_t s) {
    gemv_dense_rows<M, AF, NORM, PAIR><<<grid, kRowsThreads, lds, s>>>(p);
    return hipGetLastError();
}

template <int M, int AF>
hipError_t run_rows_form(const DenseArgs& p, bool norm, bool pair, unsigned grid, size_t lds, hipStream_t s) {
    if (norm) return pair ? run_rows<M, AF, true, true>(p, grid, lds, s) : run_rows<M, AF, true, false>(p, grid, lds, s);
    return pair ? run_rows<M, AF, false, true>(p, grid, lds, s) : run_rows<M, AF, false, false>(p, grid, lds, s);
}

template <int M>
hipError_t run_rows_af(const DenseArgs& p, bool norm, bool pair, unsigned grid, hipStream_t s) {
    const uint32_t f4 = p.m * (p.k / 4);
    const size_t lds = static_cast<size_t>(f4) * 16;
    if (f4 <= kRowsThreads) return run_rows_form<M, 1>(p, norm, pair, grid, lds, s);
    if (f4 <= 2 * kRowsThreads) return run_rows_form<M, 2>(p, norm, pair, grid, lds, s);
    if (f4 <= 4 * kRowsThreads) return run_rows_form<M, 4>(p, norm, pair, grid, lds, s);
    return run_rows_form<M, 8>(p, norm, pair, grid, lds, s);
}

template <int MT>
void run_mfma(const DenseArgs& p, bool pair, hipStream_t s) {
    // Waves per block: the blocks are the 16-row tiles, so few tiles take
    // more waves each (k cut finer) to keep as many loads in flight.
    const bool few = p.units <= 2 * compute_units();
    if (pair) {
        if (few) gemv_dense_mfma<8, MT, true><<<p.units, 8 * kWave, 0, s>>>(p);
        else gemv_dense_mfma<4, MT, true><<<p.units, 4 * kWave, 0, s>>>(p);
    } else {
        if (few) gemv_dense_mfma<16, MT, false><<<p.units, 16 * kWave, 0, s>>>(p);
        else gemv_dense_mfma<4, MT, false><<<p.units, 4 * kWave, 0, s>>>(p);
    }
}

}  // namespace

bool gemv_dense_takes(const GemvDense& f) {
    if (f.nseg == 0 || f.nseg > kFusedMaxSegs || f.m == 0 || f.m > 32 || f.k == 0 || f.k % 4 != 0 ||
        f.k > 0x3fffffffull || !aligned16(f.a))
        return false;
    uint64_t n = 0;
    for (uint32_t i = 0; i < f.nseg; ++i) {
        if (f.n[i] == 0 || !aligned16(f.w[i])) return false;
        n += f.n[i] + 16;
    }
    return n <= 0x7fffffffull;
}

bool gemv_dense_norm_takes(const GemvDense& f) {
    return rows_form(f.m, f.k) && f.k % (4 * kWave) == 0 && aligned16(f.gamma) && aligned16(f.normed);
}

hipError_t launch_gemv_dense(const GemvDense& f, hipStream_t s) {
    const bool norm = f.gamma != nullptr, pair = f.epilogue == kFusedPair;
    if (!gemv_dense_takes(f) || (norm && !gemv_dense_norm_takes(f)) || (pair && (f.nseg != 2 || f.n[0] != f.n[1])))
        return hipErrorNotSupported;
    const bool rows = rows_form(f.m, f.k);
    DenseArgs p{};
    p.a = f.a;
    p.gamma = f.gamma;
    p.normed = f.normed;
    p.eps = f.eps;
    p.m = static_cast<uint32_t>(f.m);
    p.k = static_cast<uint32_t>(f.k);
    p.nseg = f.nseg;
    for (uint32_t i = 0; i < f.nseg; ++i) {
        const bool res = f.epilogue == kFusedResidual;
        p.seg[i] = DenseSeg{f.w[i], f.out[i], res ? f.resid[i] : nullptr, res ? f.out2[i] : nullptr,
                            static_cast<uint32_t>(f.n[i]), pair ? 0u : p.units};
        const uint32_t units = rows ? p.seg[i].n : (p.seg[i].n + 15) / 16;
        p.units = pair ? units : p.units + units;
    }
    if (!rows) {
        if (f.m <= 16) run_mfma<1>(p, pair, s);
        else run_mfma<2>(p, pair, s);
        return hipGetLastError();
    }
    const unsigned grid = grid_for(p.units, kRowsWaves, 2 * compute_units());
    if (f.m == 1) return run_rows_af<1>(p, norm, pair, grid, s);
    if (f.m == 2) return run_rows_af<2>(p, norm, pair, grid, s);
    return run_rows_af<4>(p, norm, pair, grid, s);
}

// Loads this file's code object now: HIP loads one at the first use of
// any of its kernels, which otherwise lands inside the first submission
// that needs it (about 1-2 ms each, more for large objects).
hipError_t load_code_gemv_dense() {
    hipFuncAttributes attr;
    return hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&gemv_dense_mfma<4, 1, false>));
}

}  // namespace slhip
