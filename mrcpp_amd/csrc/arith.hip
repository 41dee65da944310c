// Sums and products of trees over one batch of output nodes
// (AdditionCalculator::calcNode, src/treebuilders/AdditionCalculator.h:45-70;
// MultiplicationCalculator::calcNode, src/treebuilders/MultiplicationCalculator.h:45-83).
//
// One workgroup per output node.  A sum reads the operands' nodes
// and writes their linear combination.  A product takes each operand's node
// through its reconstruction to the 8 children's scaling blocks and the
// coefficient -> value maps (MWNode::mwTransform(Reconstruction),
// MWNode::cvTransform(Forward), src/trees/MWNode.cpp:448-594) in LDS,
// multiplies the values in registers, then maps back and compresses.  The
// file is compiled without fused multiply-adds: a sum's nodes equal the host
// formation.
#pragma clang fp contract(off)

#include "mw_passes.h"

namespace mwgdev {

namespace {

// coefs_o = 0; coefs_o += c_i coefs_i, operand by operand, and the norms (the
// order of block_norms).  Bound by the reads' latency: every load of a thread's
// values is in flight at once, and as nothing goes through LDS the registers set
// how many workgroups share a CU, eight at orders 3 and 5, five at order 7, two at
// order 9 (one kernel for sums and products held two; 273 order-7 nodes a launch:
// 46 -> 13 us).
template <int N1>
__global__ __launch_bounds__(kThreads) void k_sum(mwg_combine cb, const long long *in_off, const long long *out_off, double *out, double *norms) {
    constexpr int N3 = N1 * N1 * N1, PT = (8 * N3 + kThreads - 1) / kThreads;
    __shared__ double red[8 * (kThreads / 64)];
    const int k = blockIdx.x;
    const auto offs = ro(in_off) + (size_t)k * cb.nin;
    double *dst = out + out_off[k];
    double s[PT];
#pragma unroll
    for (int p = 0; p < PT; p++) s[p] = 0.0;
    for (int i = 0; i < cb.nin; i++) {
        const long long off = offs[i];
        const bool gen = off < 0;
        const double *src = cb.pool[i] + (gen ? -off - 1 : off);
        const double c = cb.c[i];
        double v[PT];
#pragma unroll
        for (int p = 0; p < PT; p++) {
            const int o = threadIdx.x + kThreads * p;
            v[p] = o < (gen ? N3 : 8 * N3) ? src[o] : 0.0;
        }
#pragma unroll
        for (int p = 0; p < PT; p++) s[p] += c * v[p];
    }
    double ss[8];
#pragma unroll
    for (int t = 0; t < 8; t++) ss[t] = 0.0;
#pragma unroll
    for (int p = 0; p < PT; p++) {
        const int o = threadIdx.x + kThreads * p;
        if (o < 8 * N3) {
            dst[o] = s[p];
#pragma unroll
            for (int t = 0; t < 8; t++)
                if (o / N3 == t) ss[t] += s[p] * s[p];
        }
    }
    norms_of_sums(ss, norms + (size_t)k * 9, red);
}

// Products.  Each pass takes its direction's filters and its map between
// coefficients and values, so an operand takes three passes and the way back
// three (before, six each on the vector units: 162 -> 46 us a launch at order 9,
// 43 -> 18 at order 5), and the values are multiplied in the registers the
// third pass leaves them in.  Bound by the chain of loads, passes and barriers of a node.
template <int N1>
__global__ __launch_bounds__(MwShape<N1>::THREADS, MwShape<N1>::OCC) void k_product(mwg_combine cb, const long long *in_off, const int *scale, const long long *out_off,
                                                                  double *out, double *norms) {
    using P = MwShape<N1>;
    constexpr int T = P::T;
    __shared__ double a[P::SIZE], b[P::SIZE];
    __shared__ double cvs[MwMap<N1>::STORE], vcs[MwMap<N1>::STORE], red[8];
    const int k = blockIdx.x;
    const auto offs = ro(in_off) + (size_t)k * cb.nin;
    MwMap<N1> cv, vc;
    cv.load(cb.cvmap, cvs);
    if constexpr (MwMap<N1>::LDS) vc.load(cb.vcmap, vcs);
    const int n = scale[k];
    double sfp = cb.sf[0] * cb.sf[1] * cb.sf[2];
    if (sfp <= kMachineZero) sfp = 1.0;
    const double two_fac = ldexp(1.0, 3 * (n + 1)) / sfp;
    const double fwd = sqrt(two_fac), bwd = sqrt(1.0 / two_fac);
    double val[P::PER][T];
#pragma unroll
    for (int q = 0; q < P::PER; q++)
#pragma unroll
        for (int J = 0; J < T; J++) val[q][J] = 1.0;
    __syncthreads();
    {
        MwMatrix<N1> M;
        M.filters(cb.filters, 4);
        for (int i = 0; i < cb.nin; i++) {
            const long long off = offs[i];
            const bool gen = off < 0; // a generated node: scaling block, zero wavelets
            const double *src = cb.pool[i] + (gen ? -off - 1 : off);
            mw_pass<N1, 0, MW_MAP_AFTER>(
                M, [&](int t, int r, int e) { return gen && t != 0 ? 0.0 : src[t * P::N3 + N1 * r + e]; },
                [&](int, int, int t, int j, int r, double v) { a[P::at_out(t, j, r)] = v; }, cv);
            __syncthreads();
            mw_pass_lds<N1, 1, MW_MAP_AFTER>(b, a, M, cv);
            __syncthreads();
            const double ci = cb.c[i];
            mw_pass<N1, 2, MW_MAP_AFTER>(
                M, [&](int t, int r, int e) { return b[P::at(t, r, e)]; },
                [&](int q, int J, int, int, int, double v) { val[q][J] *= ci * (fwd * v); }, cv);
        }
    }
    if constexpr (!MwMap<N1>::LDS) vc.load(cb.vcmap, vcs);
    // the values (where the third pass left them) to LDS
    mw_own<N1, 2>([&](int q, int J, int t, int j, int r) { a[P::at_out(t, j, r)] = bwd * val[q][J]; });
    __syncthreads();
    mw_values_to_node<N1>(a, b, cb.filters, vc, out + out_off[k], norms + (size_t)k * 9, red);
}

template <int N1> struct CombineL {
    static mwg_status run(const mwg_combine *cb, const long long *in_off, const int *scale, const long long *out_off, double *out, double *norms,
                          int count) {
        ProfileScope prof_(MWG_KERNEL_ARITH);
        if (cb->mode == 0)
            hipLaunchKernelGGL(k_sum<N1>, dim3(count), dim3(kThreads), 0, 0, *cb, in_off, out_off, out, norms);
        else
            hipLaunchKernelGGL(k_product<N1>, dim3(count), dim3(MwShape<N1>::THREADS), 0, 0, *cb, in_off, scale, out_off, out, norms);
        MWG_LAUNCHED();
        return MWG_OK;
    }
};

// One workgroup per node pair: the scaling and wavelet parts of the pair's
// inner product, each thread over a fixed stride, then a fixed-order
// reduction over the workgroup.
template <int N1>
__global__ __launch_bounds__(kThreads) void k_dot_nodes(const double *a, const long long *a_off, const double *b, const long long *b_off,
                                                        const int *root, double *partial) {
    constexpr int N3 = N1 * N1 * N1;
    __shared__ double red[2 * kThreads];
    const int k = blockIdx.x;
    const double *x = a + a_off[k], *y = b + b_off[k];
    double s = 0.0, w = 0.0;
    if (root[k])
        for (int o = threadIdx.x; o < N3; o += kThreads) s += x[o] * y[o];
    for (int o = N3 + threadIdx.x; o < 8 * N3; o += kThreads) w += x[o] * y[o];
    red[threadIdx.x] = s;
    red[kThreads + threadIdx.x] = w;
    __syncthreads();
    for (int h = kThreads / 2; h > 0; h >>= 1) {
        if (threadIdx.x < h) {
            red[threadIdx.x] += red[threadIdx.x + h];
            red[kThreads + threadIdx.x] += red[kThreads + threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        partial[2 * k] = red[0];
        partial[2 * k + 1] = red[kThreads];
    }
}

template <int N1> struct DotL {
    static mwg_status run(const double *a, const long long *a_off, const double *b, const long long *b_off, const int *root, double *partial,
                          int count) {
        ProfileScope prof_(MWG_KERNEL_ARITH);
        hipLaunchKernelGGL(k_dot_nodes<N1>, dim3(count), dim3(kThreads), 0, 0, a, a_off, b, b_off, root, partial);
        MWG_LAUNCHED();
        return MWG_OK;
    }
};

} // namespace

} // namespace mwgdev

using namespace mwgdev;

extern "C" mwg_status mwg_dot_nodes(int kp1, const double *a, const long long *a_off, const double *b, const long long *b_off, const int *root,
                                    double *partial, int count) {
    if (need_init() != MWG_OK) return MWG_ERR_ARG;
    if (count < 0) return fail(MWG_ERR_ARG, "negative node count");
    if (count == 0) return MWG_OK;
    if (!a || !a_off || !b || !b_off || !root || !partial) return fail(MWG_ERR_ARG, "null argument");
    return dispatch<DotL>(kp1, a, a_off, b, b_off, root, partial, count);
}

extern "C" mwg_status mwg_combine_nodes(const mwg_combine *cb, const long long *in_off, const int *scale, const long long *out_off, double *out,
                                        double *norms, int count) {
    if (need_init() != MWG_OK) return MWG_ERR_ARG;
    if (count < 0) return fail(MWG_ERR_ARG, "negative node count");
    if (count == 0) return MWG_OK;
    if (!cb || !in_off || !scale || !out_off || !out || !norms) return fail(MWG_ERR_ARG, "null argument");
    if (cb->mode < 0 || cb->mode > 1) return fail(MWG_ERR_ARG, "combine mode: 0 sum, 1 product");
    if (cb->nin < 1 || cb->nin > MWG_MAX_OPERANDS) return fail(MWG_ERR_ARG, "operand count outside 1..8");
    for (int i = 0; i < cb->nin; i++)
        if (!cb->pool[i]) return fail(MWG_ERR_ARG, "null operand pool");
    if (!cb->filters || (cb->mode == 1 && (!cb->vcmap || !cb->cvmap))) return fail(MWG_ERR_ARG, "incomplete combine description");
    return dispatch<CombineL>(cb->kp1, cb, in_off, scale, out_off, out, norms, count);
}
