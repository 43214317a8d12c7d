// Dense f32 MatMulNT for more rows than the GEMV serves (prefill with
// unquantized weights; reference/matmul.rs:29-59), up to three weights
// reading the same rows in one launch, with a residual Add.
//
// Bound: the f32 matrix cores (150 TFLOP/s in a register-resident loop on
// MI355X). A block owns 16 MT rows and 128 columns: its four waves share the
// rows, staged 32 k at a time through LDS, and each reads the weights of its
// own 32 columns straight from memory, 16 rows x 64 bytes per load, one stage
// ahead. v_mfma_f32_16x16x4_f32: lane l supplies A[l % 16][k] and B[k][l % 16];
// lane group g = l / 16 takes k = 4 g + s at step s, so one float4 of each
// operand feeds four products. MT follows the row count (200 rows are two
// blocks of 112, where 128-row tiles would spend a fifth of the products on
// padding), and k is cut into slices where the tiles alone leave CUs idle:
// 128 x 128 tiles gave [2048 x 8192] at 200 rows 32 blocks of 512 k-stages of 16
// each, 766 us; here 88 us (76 TFLOP/s). [2048 x 2048] at 33 rows 192 -> 17 us,
// [4096 x 4096] at 4,096 rows 1,236 -> 1,167 us (118 TFLOP/s).
#include "common.h"
#include "kernels.h"

namespace slhip {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
constexpr int kStage = 32, kRow = kStage + 4;  // k per stage; floats per LDS row
constexpr uint32_t kCols = 128;

struct DenseGemmSeg {
    const float* w;
    SliceSeg s;
    uint32_t n, block0;
};

struct DenseGemmArgs {
    const float* a;
    DenseGemmSeg seg[kFusedMaxSegs];
    uint32_t nseg, m, k, rows, cols, slices, per;  // row and column blocks; stages per slice
    float* partial;  // slices > 1: slice z's sums at partial + z slice_floats
    uint64_t slice_floats;
};

template <int MT>
__global__ __launch_bounds__(256) void gemm_dense(DenseGemmArgs p) {
    prefetch_kernarg<arg_bytes<DenseGemmArgs>()>();
    constexpr int BM = 16 * MT, NL = (BM * kStage / 4 + 255) / 256;  // float4 of a stage per thread
    constexpr bool kWhole = BM * kStage / 4 % 256 == 0;
    __shared__ __align__(16) float as[2][(kWhole ? BM : (BM + 31) / 32 * 32) * kRow];
    const uint32_t tid = threadIdx.x, lane = tid % kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    // (run-time divisions leave their results in vector registers)
    const auto uniform = [](uint32_t v) -> uint32_t { return __builtin_amdgcn_readfirstlane(v); };
    // Blocks go to the 8 XCDs round robin; each XCD takes a contiguous run of
    // column blocks, row blocks innermost, so that its L2 reads a weight once.
    const uint32_t total = gridDim.x, xcd = blockIdx.x % 8, per = total / 8, rem = total % 8;
    const uint32_t lin = xcd * per + min(xcd, rem) + blockIdx.x / 8;
    const uint32_t by = uniform(lin % p.rows), bxz = uniform(lin / p.rows);
    const uint32_t bx = uniform(bxz % p.cols), bz = uniform(bxz / p.cols);
    const uint32_t si = (p.nseg > 1 && bx >= p.seg[1].block0 ? 1u : 0u) + (p.nseg > 2 && bx >= p.seg[2].block0 ? 1u : 0u);
#define SL_GSEG(f) (si == 0 ? p.seg[0].f : si == 1 ? p.seg[1].f : p.seg[2].f)
    const uint32_t n = SL_GSEG(n);
    const uint32_t m0 = by * BM, n0 = (bx - SL_GSEG(block0)) * kCols + 32 * wave;
    const uint32_t stages = (p.k + kStage - 1) / kStage;
    const uint32_t beg = min(bz * p.per, stages), end = min(beg + p.per, stages);

    struct Rows {
        v4f v[NL];
    };
    struct Weights {
        v4f v[2][2];  // [column tile][16-k step]
    };
    const float* const w = SL_GSEG(w);
    const float* wt[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) wt[t] = w + static_cast<uint64_t>(min(n0 + 16 * t + lane % 16, n - 1)) * p.k;
    const uint32_t kq = 4 * (lane / 16);
    auto load_rows = [&](uint32_t st) -> Rows {
        Rows r;
        const uint32_t kk = min(st * kStage + 4 * (tid % 8), p.k - 4);
#pragma unroll
        for (int i = 0; i < NL; ++i)
            r.v[i] = *reinterpret_cast<const v4f*>(p.a + static_cast<uint64_t>(min(m0 + tid / 8 + 32 * i, p.m - 1)) * p.k + kk);
        return r;
    };
    auto load_weights = [&](uint32_t st) -> Weights {
        Weights r;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t kk = min(st * kStage + 16 * q + kq, p.k - 4);
#pragma unroll
            for (int t = 0; t < 2; ++t) r.v[t][q] = *reinterpret_cast<const v4f*>(wt[t] + kk);
        }
        return r;
    };
    // past k both operands are zeros, so that nothing read twice counts twice
    // (and an infinity there meets no zero)
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    auto store_rows = [&](uint32_t buf, uint32_t st, const Rows r) {
        const bool in = st * kStage + 4 * (tid % 8) < p.k;
#pragma unroll
        for (int i = 0; i < NL; ++i)
            *reinterpret_cast<v4f*>(&as[buf][(tid / 8 + 32 * i) * kRow + 4 * (tid % 8)]) = in ? r.v[i] : zero;
    };

    v4f acc[MT][2];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i][0] = acc[i][1] = zero;
    Weights cur = load_weights(beg);
    store_rows(0, beg, load_rows(beg));
    __syncthreads();
    for (uint32_t st = beg; st < end; ++st) {
        const uint32_t buf = (st - beg) & 1, nx = min(st + 1, end - 1);
        const Rows rx = load_rows(nx);
        const Weights wx = load_weights(nx);
        __builtin_amdgcn_sched_barrier(0xF);  // arithmetic may pass; left alone, the compiler sinks the loads
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const bool in = st * kStage + 16 * q + kq < p.k;
            const v4f b0 = in ? cur.v[0][q] : zero, b1 = in ? cur.v[1][q] : zero;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const v4f a = *reinterpret_cast<const v4f*>(&as[buf][(16 * i + lane % 16) * kRow + 16 * q + kq]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b0[e], acc[i][0], 0, 0, 0);
                    acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b1[e], acc[i][1], 0, 0, 0);
                }
            }
        }
        store_rows(buf ^ 1, nx, rx);
        __syncthreads();
        cur = wx;
    }

    const SliceSeg o = SL_GSEG(s);
    const uint64_t before = si == 0 ? 0 : p.seg[0].n + (si == 1 ? 0 : p.seg[1].n);  // columns of earlier weights
#undef SL_GSEG
    float* const part = p.slices > 1 ? p.partial + bz * p.slice_floats + before * p.m : nullptr;
    // accumulator value e of lane l: row 4 (l / 16) + e, column l % 16 of its tile
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t row = m0 + 16 * i + 4 * (lane / 16) + e;
            if (row >= p.m) continue;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const uint32_t col = n0 + 16 * t + lane % 16;
                if (col >= n) continue;
                const uint64_t at = static_cast<uint64_t>(row) * n + col;
                const float val = acc[i][t][e];
                if (part != nullptr) {
                    part[at] = val;
                    continue;
                }
                o.out[at] = val;
                if (o.out2 != nullptr) o.out2[at] = o.resid[at] + val;
            }
        }
}

}  // namespace

bool gemm_dense_takes(const GemvDense& f) {
    if (f.nseg == 0 || f.nseg > kFusedMaxSegs || f.m == 0 || f.m > 0xffffffull || f.k == 0 || f.k % 4 != 0 ||
        f.k > 0x3fffffffull || f.gamma != nullptr || f.epilogue == kFusedPair || !aligned16(f.a))
        return false;
    uint64_t n = 0;
    for (uint32_t i = 0; i < f.nseg; ++i) {
        if (f.n[i] == 0 || !aligned16(f.w[i])) return false;
        n += f.n[i] + kCols;
    }
    return n <= 0xffffffull;
}

hipError_t launch_gemm_dense(const GemvDense& f, const Workspace& ws, hipStream_t s) {
    if (!gemm_dense_takes(f)) return hipErrorNotSupported;
    DenseGemmArgs p{};
    p.a = f.a;
    p.m = static_cast<uint32_t>(f.m);
    p.k = static_cast<uint32_t>(f.k);
    p.nseg = f.nseg;
    for (uint32_t i = 0; i < f.nseg; ++i) {
        const bool res = f.epilogue == kFusedResidual;
        p.seg[i] = DenseGemmSeg{f.w[i], SliceSeg{f.n[i], f.out[i], res ? f.resid[i] : nullptr, res ? f.out2[i] : nullptr},
                                static_cast<uint32_t>(f.n[i]), p.cols};
        p.cols += (p.seg[i].n + kCols - 1) / kCols;
        p.slice_floats += f.m * f.n[i];
    }
    p.rows = (p.m + 127) / 128;
    const uint32_t mt = (p.m + 16 * p.rows - 1) / (16 * p.rows);
    p.rows = (p.m + 16 * mt - 1) / (16 * mt);
    const uint32_t stages = (p.k + kStage - 1) / kStage;
    // Slices with the least estimated time: a stage keeps a CU's matrix cores
    // busy for 0.25 MT us per block, the partial sums are written and read
    // once (4 TB/s) and added by a second launch (3.5 us).
    const uint64_t tiles = static_cast<uint64_t>(p.rows) * p.cols;
    float best = INFINITY;
    for (uint32_t z = 1; z <= 16 && z <= stages; z *= 2) {
        if (z > 1 && (ws.shared || z * p.slice_floats > ws.floats)) break;
        const uint64_t per_cu = (tiles * z + compute_units() - 1) / compute_units();
        float t = static_cast<float>(per_cu * ((stages + z - 1) / z) * mt) * 0.25f;
        if (z > 1) t += 3.5f + static_cast<float>(p.slice_floats * (2 * z + 1)) * 1e-6f;
        if (t < best) {
            best = t;
            p.slices = z;
        }
    }
    if (tiles * p.slices > 0x7fffffffull) return hipErrorNotSupported;
    p.per = (stages + p.slices - 1) / p.slices;
    p.partial = p.slices > 1 ? ws.data : nullptr;
    const unsigned grid = static_cast<unsigned>(tiles * p.slices);
    switch (mt) {
        case 1: gemm_dense<1><<<grid, 256, 0, s>>>(p); break;
        case 2: gemm_dense<2><<<grid, 256, 0, s>>>(p); break;
        case 3: gemm_dense<3><<<grid, 256, 0, s>>>(p); break;
        case 4: gemm_dense<4><<<grid, 256, 0, s>>>(p); break;
        case 5: gemm_dense<5><<<grid, 256, 0, s>>>(p); break;
        case 6: gemm_dense<6><<<grid, 256, 0, s>>>(p); break;
        case 7: gemm_dense<7><<<grid, 256, 0, s>>>(p); break;
        default: gemm_dense<8><<<grid, 256, 0, s>>>(p); break;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.slices == 1) return e;
    SliceSum sum{};
    sum.partial = p.partial;
    sum.slice_floats = p.slice_floats;
    sum.m = f.m;
    sum.slices = p.slices;
    for (uint32_t i = 0; i < f.nseg; ++i) sum.seg[i] = p.seg[i].s;
    return launch_slices_sum(sum, s);
}

// Loads this file's code object now: HIP loads one at the first use of
// any of its kernels, which otherwise lands inside the first submission
// that needs it (about 1-2 ms each, more for large objects).
hipError_t load_code_gemm_dense() {
    hipFuncAttributes attr;
    return hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&gemm_dense<1>));
}

}  // namespace slhip
