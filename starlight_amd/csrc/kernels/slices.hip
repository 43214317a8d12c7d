// The sum of a GEMM's k slices: up to three outputs of m rows, each slice's
// partial sums one output after the other, added in slice order, with the
// residual Add where an output has one.
#include "common.h"
#include "kernels.h"

namespace slhip {
namespace {

// V: elements per thread and step (4 where every n is a multiple of four and
// the pointers allow it). Bound by the partial sums' reads.
template <int V>
__global__ __launch_bounds__(256) void slices_sum(SliceSum p) {
    prefetch_kernarg<arg_bytes<SliceSum>()>();
    typedef float vec __attribute__((ext_vector_type(V)));
    const uint64_t step = static_cast<uint64_t>(gridDim.x) * 256 * V;
    const uint64_t end0 = p.m * p.seg[0].n, end1 = end0 + p.m * p.seg[1].n;
    for (uint64_t i = (static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x) * V; i < p.slice_floats; i += step) {
        vec v = *reinterpret_cast<const vec*>(p.partial + i);
        for (uint32_t z = 1; z < p.slices; ++z) v += *reinterpret_cast<const vec*>(p.partial + z * p.slice_floats + i);
        const int si = i < end0 ? 0 : i < end1 ? 1 : 2;
        const uint64_t o = i - (si == 0 ? 0 : si == 1 ? end0 : end1);
        float* const out = si == 0 ? p.seg[0].out : si == 1 ? p.seg[1].out : p.seg[2].out;
        float* const out2 = si == 0 ? p.seg[0].out2 : si == 1 ? p.seg[1].out2 : p.seg[2].out2;
        const float* const resid = si == 0 ? p.seg[0].resid : si == 1 ? p.seg[1].resid : p.seg[2].resid;
        if (out != nullptr) *reinterpret_cast<vec*>(out + o) = v;
        if (out2 != nullptr) *reinterpret_cast<vec*>(out2 + o) = *reinterpret_cast<const vec*>(resid + o) + v;
    }
}

}  // namespace

hipError_t launch_slices_sum(const SliceSum& p, hipStream_t s) {
    bool quads = aligned16(p.partial);
    for (const SliceSeg& g : p.seg)
        quads = quads && g.n % 4 == 0 && aligned16(g.out) && aligned16(g.resid) && aligned16(g.out2);
    if (quads) slices_sum<4><<<grid_for(p.slice_floats / 4, 256, 8192), 256, 0, s>>>(p);
    else slices_sum<1><<<grid_for(p.slice_floats, 256, 8192), 256, 0, s>>>(p);
    return hipGetLastError();
}

// Loads this file's code object now: HIP loads one at the first use of
// any of its kernels, which otherwise lands inside the first submission
// that needs it (about 1-2 ms each, more for large objects).
hipError_t load_code_slices() {
    hipFuncAttributes attr;
    return hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&slices_sum<1>));
}

}  // namespace slhip
