// Projection of a sum of Gaussians onto the nodes of one tree level
// (ProjectionCalculator::calcNode, src/treebuilders/ProjectionCalculator.cpp:34-51).
//
// One workgroup per node.  The function is sampled at the
// Gauss-Legendre points of the node's 8 children (MWNode::getExpandedChildPts,
// src/trees/MWNode.cpp:854-925): point (t, i0, i1, i2) sits at
// sf_d 2^-(n+1) (x_{i_d} + 2 l_d + bit_d(t)).  A Gaussian is separable, so per
// node and term the 3 x 2(k+1) one-dimensional factors exp(-alpha_d q^2) are
// formed once in LDS and every point takes (coef e_x e_y) e_z: 6(k+1) exp
// evaluations per term instead of 8(k+1)^3.  Then the value -> coefficient
// map in each direction (MWNode::cvTransform, :448-490), the scaling factor
// sqrt(sf_x sf_y sf_z / 2^(3(n+1))), the compression to the node's scaling and
// wavelet blocks (MWNode::mwTransform(Compression)) and the component norms.
#include "mw_passes.h"

namespace mwgdev {

namespace {

constexpr int kTermsPerRound = 16; // Gaussian terms whose 1D factors share LDS at a time

// The value at a point is sum_g (c_g e_x e_y)(e_z): the points' values are a
// product of a 4 N1^2 x terms matrix, formed as it is read, and a terms x 2 N1
// matrix, in the tiles of a pass (mw_passes.h) and left as a pass in direction z
// leaves them.  A pass takes the value -> coefficient map and the compression
// filters of its direction, three passes in all.  Bound by the exponentials and the chain of
// passes (points one by one on the vector units, maps and filters apart:
// 142 -> 58 us a launch of order 7).
template <int N1>
__global__ __launch_bounds__(MwShape<N1>::THREADS, MwShape<N1>::OCC) void k_project(mwg_projection pj, const int *scale, const int *lv, const long long *off,
                                                                  double *coef, double *norms) {
    using P = MwShape<N1>;
    constexpr int N2 = P::N2, W = 2 * N1, T = P::T, G = kTermsPerRound;
    __shared__ double a[P::SIZE], b[P::SIZE];
    // exp(-alpha_d q^2) at the 2 N1 points of each direction, in the buffer that
    // the passes write first
    static_assert(G * 3 * W <= P::SIZE, "factors fit a pass buffer");
    double(*fac1d)[3][W] = reinterpret_cast<double(*)[3][W]>(b);
    __shared__ double gcoef[G];
    __shared__ double vcs[MwMap<N1>::STORE], red[8];
    __shared__ double sx[N1];
    const int k = blockIdx.x;
    const int n = scale[k];
    const int l[3] = {lv[3 * k], lv[3 * k + 1], lv[3 * k + 2]};
    const double h = ldexp(1.0, -(n + 1));
    for (int i = threadIdx.x; i < N1; i += P::THREADS) sx[i] = pj.nodes[i];
    MwMap<N1> vc;
    if constexpr (MwMap<N1>::LDS) vc.load(pj.vcmap, vcs);

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 3, row = lane & 15, kk = lane >> 4;
    double val[P::PER][T];
#pragma unroll
    for (int q = 0; q < P::PER; q++)
#pragma unroll
        for (int J = 0; J < T; J++) val[q][J] = 0.0;
    for (int g0 = 0; g0 < pj.ngauss; g0 += G) {
        const int ng = min(G, pj.ngauss - g0), steps = (ng + 3) / 4;
        __syncthreads(); // points staged; previous round's factors consumed
        for (int p = threadIdx.x; p < 4 * steps * 3 * W; p += P::THREADS) {
            const int gi = p / (3 * W), rest = p % (3 * W), d = rest / W, hi = rest % W;
            const int half = hi / N1, i = hi % N1;
            double e = 0.0; // terms past the last fill the step with zeros
            if (gi < ng) {
                const mwg_gauss &gs = pj.gauss[g0 + gi];
                const double base = sx[i] + 2.0 * (double)l[d];
                const double r = pj.sf[d] * (h * (half ? base + 1.0 : base));
                const double dq = r - gs.pos[d];
                e = exp(-(gs.alpha[d] * dq * dq));
            }
            fac1d[gi][d][hi] = e;
        }
        for (int gi = threadIdx.x; gi < 4 * steps; gi += P::THREADS) gcoef[gi] = gi < ng ? pj.gauss[g0 + gi].coef : 0.0;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < P::PER; q++) {
            const int item = wave + P::WAVES * q;
            if (P::ITEMS % P::WAVES != 0 && item >= P::ITEMS) break;
            const int ra = 16 * item + row, c = ra / N2, e = ra - c * N2; // row: child bits (x, y), points (i_x, i_y)
            const int ix = (c & 1) * N1 + e % N1, iy = (c >> 1) * N1 + e / N1;
            for (int K = 0; K < steps; K++) {
                const int gi = 4 * K + kk;
                const double xy = gcoef[gi] * (fac1d[gi][0][ix] * fac1d[gi][1][iy]);
#pragma unroll
                for (int J = 0; J < T; J++) val[q][J] = __builtin_amdgcn_mfma_f64_4x4x4f64(fac1d[gi][2][4 * J + col], xy, val[q][J], 0, 0, 0);
            }
        }
    }
    double sfp = pj.sf[0] * pj.sf[1] * pj.sf[2];
    if (sfp <= kMachineZero) sfp = 1.0;
    const double fac = sqrt(1.0 / (ldexp(1.0, 3 * (n + 1)) / sfp));
    if constexpr (!MwMap<N1>::LDS) vc.load(pj.vcmap, vcs);
    mw_own<N1, 2>([&](int q, int J, int t, int j, int r) { a[P::at_out(t, j, r)] = fac * val[q][J]; });
    __syncthreads();
    mw_values_to_node<N1>(a, b, pj.filters, vc, coef + off[k], norms + (size_t)k * 9, red);
}

template <int N1> struct ProjectL {
    static mwg_status run(const mwg_projection *pj, const int *scale, const int *l, const long long *off, double *coef, double *norms, int count) {
        ProfileScope prof_(MWG_KERNEL_PROJECT);
        hipLaunchKernelGGL(k_project<N1>, dim3(count), dim3(MwShape<N1>::THREADS), 0, 0, *pj, scale, l, off, coef, norms);
        MWG_LAUNCHED();
        return MWG_OK;
    }
};

} // namespace

} // namespace mwgdev

using namespace mwgdev;

extern "C" mwg_status mwg_project_nodes(const mwg_projection *pj, const int *scale, const int *l, const long long *off, double *coef, double *norms,
                                        int count) {
    if (need_init() != MWG_OK) return MWG_ERR_ARG;
    if (count < 0) return fail(MWG_ERR_ARG, "negative node count");
    if (count == 0) return MWG_OK;
    if (!pj || !scale || !l || !off || !coef || !norms) return fail(MWG_ERR_ARG, "null argument");
    if (!pj->nodes || !pj->vcmap || !pj->filters || (pj->ngauss > 0 && !pj->gauss) || pj->ngauss < 0)
        return fail(MWG_ERR_ARG, "incomplete projection description");
    return dispatch<ProjectL>(pj->kp1, pj, scale, l, off, coef, norms, count);
}
