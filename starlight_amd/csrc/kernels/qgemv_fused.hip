// Group-quantized GEMV for decode (m <= 16 activation rows, m * k <= 16384)
// with the K reduction kept inside one workgroup, and the fusions a decoder
// layer wants around it.
//
// Arithmetic is the int8-limb MFMA scheme of qgemv_mfma.hip (exact integer
// products, one f32 combination per group; the weight tiles are the same
// QuantLayout::Mfma superblocks). What differs is the work split:
//  * a block of 8 waves owns one 16-row tile (or, for a gate/up pair, one
//    tile of each with 4 waves apiece) and the whole K range; its waves take
//    contiguous, group-aligned runs of superblocks and start their weight
//    loads (4 superblocks, rolling) before the activation prologue, then
//    add their partial sums in LDS in wave order. The group scales come
//    with each superblock's codes, or (long streams at m = 1) are loaded
//    into LDS for all the block's tiles at launch.
//    No split partials in HBM, no second launch, deterministic. Blocks stay
//    resident over several tiles (at most two per CU), so the prologue is
//    paid once per block, and the per-tile LDS sums are double-buffered;
//  * the activations are converted once per block from registers: every
//    thread holds its share of the m x k input as float4; the exponent of
//    each 256-element chunk comes from one wave's DPP max (no block-wide
//    pass), and only the RMSNorm sum of squares goes wave -> LDS -> row;
//  * up to three weights that read the same input run as one launch (q/k/v);
//  * prologue RMSNorm: x = (a * inv) * gamma with inv = 1/sqrt(ss/k + eps)
//    (reference/norm.rs:27-60), block 0 also writes x as the norm's output;
//  * epilogues: plain; residual (out2 = resid + out, reference/add.rs); pair
//    (h = silu(g) * u over a gate and an up tile, reference/swiglu.rs:40-84).
#include "common.h"
#include "kernels.h"
#include "qgemv_kernel.h"
#include "starlight_hip.h"

namespace slhip {
namespace {

// out[i] = the sum of the k slices' partials of element i, in slice order;
// with resid, out2[i] = resid[i] + out[i] (the residual Add's order).
__global__ __launch_bounds__(256) void qgemv_slices_sum(const float* __restrict__ partial, uint32_t slices,
                                                        uint64_t count, float* out, const float* resid,
                                                        float* out2) {
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x; i < count;
         i += static_cast<uint64_t>(gridDim.x) * 256) {
        float v = partial[i];
        for (uint32_t sl = 1; sl < slices; ++sl) v += partial[sl * count + i];
        out[i] = v;
        if (out2 != nullptr) out2[i] = resid[i] + v;
    }
}

}  // namespace

hipError_t launch_qgemv_fused(const QgemvFused& f, hipStream_t s) {
    if (f.nseg == 0 || f.nseg > kFusedMaxSegs || f.m == 0 || f.m > 16) return hipErrorNotSupported;
    const QuantWeight& w0 = *f.w[0];
    const uint64_t k = w0.k;
    if (w0.layout != QuantLayout::Mfma || k % 256 != 0 || w0.group % 64 != 0 || k % w0.group != 0 ||
        !(w0.group == 64 || w0.group == 128 || w0.group % 256 == 0) || !aligned16(f.a) ||
        (f.gamma != nullptr && !aligned16(f.gamma)) || (f.normed != nullptr && !aligned16(f.normed)))
        return hipErrorNotSupported;
    if (f.epilogue == kFusedPair && f.nseg != 2) return hipErrorNotSupported;
    // Activations beyond the LDS (m x k above max_elems(16): the down
    // projection, k = 14336, at batch 8): the grid's y dimension cuts k into
    // slices that fit, each block converting only its slice; the slices'
    // partial sums go to f.partial and a second launch adds them up (and
    // the residual). Single weights without a norm prologue only.
    uint32_t slices = 1;
    if (f.m * k > max_elems(16)) {
        if (f.gamma != nullptr || f.epilogue == kFusedPair || f.nseg != 1 || f.partial == nullptr)
            return hipErrorNotSupported;
        const uint64_t unit = w0.group > 256 ? w0.group : 256;
        while (slices <= 16 && (k % (slices * unit) != 0 || f.m * (k / slices) > max_elems(16))) ++slices;
        if (slices > 16 || slices * f.m * w0.n > f.partial_floats) return hipErrorNotSupported;
    }
    const uint64_t kc = k / slices;
    Args p;
    p.normed = f.normed;
    p.eps = f.eps;
    p.nseg = f.nseg;
    p.m = static_cast<uint32_t>(f.m);
    p.k = static_cast<uint32_t>(kc);
    p.group = w0.group;
    p.sb_total = p.k / 128;
    p.groups_total = p.k / p.group;
    p.unit = p.group < 256 ? p.group : 256;
    p.epilogue = slices > 1 ? kFusedPlain : f.epilogue;
    uint32_t tiles = 0;
    for (uint32_t i = 0; i < f.nseg; ++i) {
        const QuantWeight& w = *f.w[i];
        if (w.layout != QuantLayout::Mfma || w.tile_scales == nullptr || w.k != k || w.group != w0.group ||
            w.format != w0.format || w.n > 0xffffffffull)
            return hipErrorNotSupported;
        if (f.epilogue == kFusedPair && w.n != w0.n) return hipErrorNotSupported;
        p.seg[i] = Seg{w.tiles, w.tile_scales, slices > 1 ? f.partial : f.out[i], f.resid[i], f.out2[i],
                       static_cast<uint32_t>(w.n), tiles};
        if (f.epilogue != kFusedPair) tiles += static_cast<uint32_t>((w.n + 15) / 16);
    }
    if (f.epilogue == kFusedPair) tiles = static_cast<uint32_t>((w0.n + 15) / 16);
    p.tiles_total = tiles;
    const bool int4 = w0.format == SL_QFORMAT_INT4, pair = f.epilogue == kFusedPair, lr = p.m <= 4;
    // Waves per block: 16 for long k (the down projection, k = 14336), which
    // doubles the weight loads in flight per CU and halves each thread's
    // share of the activation prologue, and for a single weight above 24 MB
    // whose tiles one round of 16-wave blocks holds (one block per CU
    // instead of two converting the same activations): [14336 x 4096] 7.95-
    // 8.04 -> 7.74-7.83 us. 8 otherwise: with 16, lm_head [128256 x 4096]
    // 47.0 -> 48.1 us, q/k/v and o-proj [4096 x 4096] 0.8 us slower together.
    const uint64_t weight_bytes = static_cast<uint64_t>(tiles) * p.sb_total * (int4 ? 1024 : 2048) * (pair ? 2 : 1);
    const bool wide = !pair && p.m == 1 && p.k >= 4096 && weight_bytes > (24ull << 20) &&
                      tiles <= 4 * compute_units();
    const int waves = p.k >= 8192 || p.m * p.k > max_elems(8) || wide || slices > 1 ? 16 : 8;
    const uint32_t threads = static_cast<uint32_t>(waves) * kWave;
    const uint32_t wpt = f.epilogue == kFusedPair ? waves / 2 : waves;
    const uint32_t sb_per_group = p.group >= 128 ? p.group / 128 : 1;
    uint32_t per = (p.sb_total + wpt - 1) / wpt;
    per = (per + sb_per_group - 1) / sb_per_group * sb_per_group;
    p.sb_per_wave = per;
    // Resident blocks: every block converts the activations once for all
    // its tiles; the results of a block's tiles wait in LDS (at most 16 KB).
    // Weights of up to 24 MB take one block per CU, the tiles dealt round
    // robin (some blocks one more): the prologue, repeated by every block,
    // is then paid once per CU. Larger ones take up to two per CU, with
    // even shares, for more loads in flight. (Measured on MI355X, M = 1:
    // the q/k/v launch [6144 x 4096] gains 1 us from one block per CU, the
    // gate/up pair [2 x 14336 x 4096] loses 0.5 us.)
    uint32_t blocks, per_block;
    const uint32_t per_cap = 4096 / (16 * p.m);
    if (slices > 1) {
        // about one block per CU over all slices: each block converts its
        // slice's activations once for several tiles
        blocks = (compute_units() + slices - 1) / slices;
        if (blocks > tiles) blocks = tiles;
        per_block = (tiles + blocks - 1) / blocks;
    } else if (weight_bytes <= (24ull << 20)) {
        blocks = tiles < compute_units() ? tiles : compute_units();
        per_block = (tiles + blocks - 1) / blocks;
    } else {
        const uint32_t max_blocks = (waves == 16 ? 1 : 2) * compute_units();
        per_block = (tiles + max_blocks - 1) / max_blocks;
        blocks = 0;
    }
    // Float4 of activations per thread, a compile-time count: the prologue
    // is straight-line code run once per wave, fetched cold by every CU at
    // each launch, so its length shows in the launch time (about 1 us for
    // the RMSNorm prologue at 8 float4 per thread against 2).
    const uint32_t f4 = (p.m * p.k / 4 + threads - 1) / threads;
    // Scales in LDS (LS) for one activation row, k >= 4096 and more
    // superblocks per wave than the window holds. Measured on MI355X
    // against scales loaded with each superblock: [14336 x 4096] 8.61 ->
    // 8.45 us, [4096 x 14336] 9.24 -> 9.00 us, the gate/up pair [2 x 14336
    // x 4096] 13.62 -> 13.32 us; but [2048 x 8192] (4 superblocks per
    // wave) 5.80 -> 6.34 us, and M = 8 [14336 x 4096] 13.73 -> 14.38 us.
    const bool ls = p.m == 1 && slices == 1 && p.k >= 4096 && f4 <= 4 && per_block * per > kWindow;
    // A stream that fits the first window (every block's tiles times the
    // superblocks per wave; the cap below only lowers per_block) is one
    // round without refills: [2048 x 8192] 5.50 -> 5.20 us, [2048 x 2048]
    // 3.77 -> 3.60 us. Dropping the refills of a longer stream's last round
    // instead makes the compiler's waits cover more than one item:
    // [14336 x 4096] 8.45 -> 8.69 us.
    const bool one_round = !ls && lr && slices == 1 && f4 <= 4 && per_block * per <= kWindow;
    // the per-lane item table holds at most 64 items per wave, and with LS
    // the tiles' scales at most qgemv_scale_slots float4 per thread
    const uint32_t gps = p.group == 64 ? 2 : 1, nt = pair ? 2 : 1;
    uint32_t item_cap = 64 / per;
    if (ls) {
        const uint32_t scale_cap =
            static_cast<uint32_t>(qgemv_scale_slots(nt, gps, int4 ? 4 : 8)) * threads / (nt * p.sb_total * 4 * gps);
        if (scale_cap < item_cap) item_cap = scale_cap;
    }
    const uint32_t cap = per_cap < item_cap ? per_cap : item_cap;
    if (cap == 0) return hipErrorNotSupported;
    if (per_block > cap) per_block = cap;
    if (blocks == 0 || per_block == cap) blocks = (tiles + per_block - 1) / per_block;
    p.tile_slots = per_block;
    p.tiles_base = tiles / blocks;
    p.tiles_rem = tiles % blocks;
    p.len_magic = magic16(per);
    p.m_magic = magic16(p.m);
    p.run4_magic = static_cast<uint32_t>(((1ull << 32) + run4_of(p.sb_total, gps) - 1) / run4_of(p.sb_total, gps));
    const uint32_t mk = p.m | (magic16(p.k / 256) << 5);
    const size_t lds = static_cast<size_t>(3) * p.m * (p.k + kLimbPad) +
                       sizeof(float) * static_cast<size_t>(per_block) * 16 * p.m +
                       (ls ? sizeof(float) * static_cast<size_t>(per_block) * nt * p.sb_total * 16 * gps : 0);
    if (lds + static_lds(waves) > max_lds_per_block()) return hipErrorNotSupported;
    const int spg = p.group == 64 ? 1 : p.group == 128 ? 2 : 0;
    const dim3 grid(blocks, slices);
#define SL_QGEMV_LAUNCH(B, T, G, L, F, W, S) \
    qgemv_fused<B, T, G, L, F, W, false, S><<<grid, threads, lds, s>>>(f.a, f.gamma, mk, p.k, p)
#define SL_QGEMV_FUSED_F(B, T, G, L)                                                                               \
    (waves == 16 ? (f4 <= 2 ? SL_QGEMV_LAUNCH(B, T, G, L, 2, 16, kSmStream)                                             \
                            : f4 <= 4 ? SL_QGEMV_LAUNCH(B, T, G, L, 4, 16, kSmStream) : SL_QGEMV_LAUNCH(B, T, G, L, 8, 16, kSmStream)) \
                 : f4 <= 2 ? SL_QGEMV_LAUNCH(B, T, G, L, 2, 8, kSmStream)                                               \
                           : f4 <= 4 ? SL_QGEMV_LAUNCH(B, T, G, L, 4, 8, kSmStream) : SL_QGEMV_LAUNCH(B, T, G, L, 8, 8, kSmStream))
#define SL_QGEMV_FUSED_SM(B, T, G, S)                                                                               \
    (waves == 16 ? (f4 <= 2 ? SL_QGEMV_LAUNCH(B, T, G, true, 2, 16, S) : SL_QGEMV_LAUNCH(B, T, G, true, 4, 16, S)) \
                 : f4 <= 2 ? SL_QGEMV_LAUNCH(B, T, G, true, 2, 8, S) : SL_QGEMV_LAUNCH(B, T, G, true, 4, 8, S))
#define SL_QGEMV_FUSED(B, T, G) \
    (ls ? SL_QGEMV_FUSED_SM(B, T, G, kSmLds)                                          \
        : one_round ? SL_QGEMV_FUSED_SM(B, T, G, kSmOneRound)                         \
                    : lr ? SL_QGEMV_FUSED_F(B, T, G, true) : SL_QGEMV_FUSED_F(B, T, G, false))
#define SL_QGEMV_FUSED_G(B, T) \
    (spg == 1 ? SL_QGEMV_FUSED(B, T, 1) : spg == 2 ? SL_QGEMV_FUSED(B, T, 2) : SL_QGEMV_FUSED(B, T, 0))
    if (slices > 1) {
        // k slices: 16 waves, 8 float4 per thread. (Up to four rows (one from
        // k = 32768 on, two from 16384) in the form for as many, not on the
        // split-k fallback with its own reduction and Add: INT8 [4096 x 14336]
        // at M = 4, two 8B layers decoding for four sequences 584 -> 519 us
        // over two steps. That form's six kernels are in a file of their own:
        // among these, 8B INT4 decode ran 0.6% slower on the same instructions.)
        if (f4 > 8) return hipErrorNotSupported;
        if (lr) {
            const hipError_t e =
                run_qgemv_sliced_few_rows(int4, spg, grid, threads, lds, f.a, f.gamma, mk, p.k, &p, s);
            if (e != hipSuccess) return e;
        } else {
#define SL_QGEMV_SLICED(B, G) qgemv_fused<B, 1, G, false, 8, 16, true, kSmStream><<<grid, threads, lds, s>>>(f.a, f.gamma, mk, p.k, p)
            if (int4) {
                if (spg == 1) SL_QGEMV_SLICED(4, 1);
                else if (spg == 2) SL_QGEMV_SLICED(4, 2);
                else SL_QGEMV_SLICED(4, 0);
            } else {
                if (spg == 1) SL_QGEMV_SLICED(8, 1);
                else if (spg == 2) SL_QGEMV_SLICED(8, 2);
                else SL_QGEMV_SLICED(8, 0);
            }
#undef SL_QGEMV_SLICED
        }
    } else if (int4) {
        if (pair) SL_QGEMV_FUSED_G(4, 2);
        else SL_QGEMV_FUSED_G(4, 1);
    } else {
        if (pair) SL_QGEMV_FUSED_G(8, 2);
        else SL_QGEMV_FUSED_G(8, 1);
    }
#undef SL_QGEMV_FUSED_G
#undef SL_QGEMV_FUSED
#undef SL_QGEMV_FUSED_SM
#undef SL_QGEMV_FUSED_F
#undef SL_QGEMV_LAUNCH
    if (slices > 1) {
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const uint64_t count = f.m * w0.n;
        const bool residual = f.epilogue == kFusedResidual;
        qgemv_slices_sum<<<grid_for(count, 256, 1024), 256, 0, s>>>(f.partial, slices, count, f.out[0],
                                                                   residual ? f.resid[0] : nullptr,
                                                                   residual ? f.out2[0] : nullptr);
    }
    return hipGetLastError();
}

// Loads this file's code object now: HIP loads one at the first use of
// any of its kernels, which otherwise lands inside the first submission
// that needs it (about 1-2 ms each, more for large objects).
hipError_t load_code_qgemv_fused() {
    hipFuncAttributes attr;
    return hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&qgemv_slices_sum));
}

}  // namespace slhip
