// Multiwavelet transforms on the device: generated band nodes, top-down
// reconstruction, bottom-up compression and component norms.  One workgroup per
// node; a node's values go from HBM into the first pass's operands, through LDS
// twice, and from the last pass's results back (passes on the vector units with
// the node staged in LDS: compression 10.3 -> 8.4 us a launch at order 7, 24 ->
// 13 at order 9; generation 16 -> 9 at order 9).  A launch's few nodes leave most
// of that to its latency: the loads, two barriers and the stores of one node.
#include "mw_passes.h"

namespace mwgdev {

namespace {

// The scaling block of child c of node pid (a, b, red: LDS of the workgroup),
// written at offs[k] (recorded in the tree) or at the
// node's own offset, and its norms.
template <int N1>
__device__ __forceinline__ void generate_node(const mwg_ftree &f, const double *filt, int k, int id, int pid, int c, const long long *offs,
                                              long long *coef_off_w, unsigned char *is_gen_w, double *a, double *b, double *red) {
    using P = MwShape<N1>;
    constexpr int N3 = P::N3;
    const double *src = f.coef + f.coef_off[pid];
    const bool gen = f.is_gen[pid]; // generated parents carry the scaling block only
    MwMatrix<N1> M;
    M.filters(filt, 4);
    mw_pass<N1, 0>(
        M, [&](int t, int r, int i) { return gen && t != 0 ? 0.0 : src[t * N3 + N1 * r + i]; },
        [&](int, int, int t, int j, int r, double v) { a[P::at_out(t, j, r)] = v; });
    __syncthreads();
    mw_pass_lds<N1, 1>(b, a, M);
    __syncthreads();
    mw_pass<N1, 2>(
        M, [&](int t, int r, int i) { return b[P::at(t, r, i)]; },
        [&](int, int, int t, int j, int r, double v) {
            if (t == c) a[P::at_out(0, j, r)] = v;
        });
    __syncthreads();
    double *dst = f.coef + (offs ? offs[k] : f.coef_off[id]);
    if (offs && threadIdx.x == 0) {
        coef_off_w[id] = offs[k];
        is_gen_w[id] = 1;
    }
    for (int e = threadIdx.x; e < N3; e += P::THREADS) dst[e] = a[P::at_elem(0, e)];
    // the norm summed by the first kThreads threads in their order (the
    // order of the band screen's other norms)
    if (threadIdx.x < kThreads) {
        double ss = 0.0;
        for (int e = threadIdx.x; e < N3; e += kThreads) {
            const double v = a[P::at_elem(0, e)];
            ss += v * v;
        }
        for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double v = 0.0;
        for (int w = 0; w < kThreads / 64; w++) v += red[w];
        const double n0 = sqrt(v);
        double *nr = f.norms + (size_t)id * 9;
        nr[0] = n0;
        for (int t = 1; t < 8; t++) nr[t] = 0.0;
        nr[8] = n0 * n0;
    }
}

// Scaling block of one child of an existing node (MWNode::threadSafeGenChildren
// + giveChildrenCoefs, src/trees/MWNode.cpp:312-335,410-418).
// With offs given, the node is also recorded in the mirror: coef_off_w[id] =
// offs[k] (where its block goes) and is_gen_w[id] = 1.
template <int N1>
__global__ __launch_bounds__(MwShape<N1>::THREADS, MwShape<N1>::OCC) void k_generate(mwg_ftree f, const double *filt, const int *ids, const int *parent, const int *child,
                                                           const long long *offs, long long *coef_off_w, unsigned char *is_gen_w) {
    __shared__ double a[MwShape<N1>::SIZE], b[MwShape<N1>::SIZE];
    __shared__ double red[kThreads / 64];
    const int k = blockIdx.x;
    generate_node<N1>(f, filt, k, ids[k], parent[k], child[k], offs, coef_off_w, is_gen_w, a, b, red);
}

// The same for nodes of several trees: node k in trees[tree_of[k]].
template <int N1>
__global__ __launch_bounds__(MwShape<N1>::THREADS, MwShape<N1>::OCC) void k_generate_multi(const mwg_gen_tree *trees, const double *filt, const int *tree_of, const int *ids,
                                                                 const int *parent, const int *child, const long long *offs) {
    __shared__ double a[MwShape<N1>::SIZE], b[MwShape<N1>::SIZE];
    __shared__ double red[kThreads / 64];
    const int k = blockIdx.x;
    const mwg_gen_tree &t = trees[tree_of[k]];
    generate_node<N1>(t.f, filt, k, ids[k], parent[k], child[k], offs, t.coef_off_w, t.is_gen_w, a, b, red);
}

template <int N1>
__global__ __launch_bounds__(MwShape<N1>::THREADS, MwShape<N1>::OCC) void k_reconstruct_add(const double *filt, double *coef, const long long *poff,
                                                                                            const long long *coff, long long stride) {
    using P = MwShape<N1>;
    __shared__ double a[P::SIZE], b[P::SIZE];
    const int k = blockIdx.x;
    const double *src = coef + poff[k];
    double *dst = coef + coff[k];
    MwMatrix<N1> M;
    M.filters(filt, 4);
    mw_pass<N1, 0>(
        M, [&](int t, int r, int i) { return src[t * P::N3 + N1 * r + i]; },
        [&](int, int, int t, int j, int r, double v) { a[P::at_out(t, j, r)] = v; });
    // the children's values as they are, in flight during the second pass
    double old[P::PER][P::T];
    mw_own<N1, 2>([&](int q, int J, int t, int j, int r) { old[q][J] = dst[t * stride + j * P::N2 + r]; });
    __syncthreads();
    mw_pass_lds<N1, 1>(b, a, M);
    __syncthreads();
    // the two contributions added one after the other
    mw_pass<N1, 2, MW_APART>(
        M, [&](int t, int r, int i) { return b[P::at(t, r, i)]; },
        [&](int q, int J, int t, int j, int r, double v0, double v1) { dst[t * stride + j * P::N2 + r] = old[q][J] + v0 + v1; });
}

template <int N1>
__global__ __launch_bounds__(MwShape<N1>::THREADS, MwShape<N1>::OCC) void k_compress(const double *filt, double *coef, const long long *poff,
                                                                                     const long long *coff, long long stride) {
    using P = MwShape<N1>;
    __shared__ double a[P::SIZE], b[P::SIZE];
    const int k = blockIdx.x;
    const double *src = coef + coff[k];
    double *dst = coef + poff[k];
    MwMatrix<N1> M;
    M.filters(filt, 0);
    mw_pass<N1, 0>(
        M, [&](int t, int r, int i) { return src[t * stride + N1 * r + i]; },
        [&](int, int, int t, int j, int r, double v) { a[P::at_out(t, j, r)] = v; });
    __syncthreads();
    mw_pass_lds<N1, 1>(b, a, M);
    __syncthreads();
    mw_pass<N1, 2>(
        M, [&](int t, int r, int i) { return b[P::at(t, r, i)]; },
        [&](int, int, int t, int j, int r, double v) { dst[t * P::N3 + j * P::N2 + r] = v; });
}

template <int N1> __global__ __launch_bounds__(kThreads) void k_node_norms(const double *coef, const long long *off, double *norms) {
    __shared__ double red[8 * (kThreads / 64)];
    const int k = blockIdx.x;
    block_norms<N1>(coef + off[k], norms + (size_t)k * 9, red);
}

template <int N1> struct GenerateL {
    static mwg_status run(const mwg_ftree *f, const double *filt, const int *ids, const int *par, const int *ch, int count, const long long *offs,
                          long long *coef_off_w, unsigned char *is_gen_w) {
        ProfileScope prof_(MWG_KERNEL_GENERATE);
        hipLaunchKernelGGL(k_generate<N1>, dim3(count), dim3(MwShape<N1>::THREADS), 0, 0, *f, filt, ids, par, ch, offs, coef_off_w, is_gen_w);
        MWG_LAUNCHED();
        return MWG_OK;
    }
};
template <int N1> struct GenerateMultiL {
    static mwg_status run(const mwg_gen_tree *trees, const double *filt, const int *tree_of, const int *ids, const int *par, const int *ch,
                          const long long *offs, int count) {
        ProfileScope prof_(MWG_KERNEL_GENERATE);
        hipLaunchKernelGGL(k_generate_multi<N1>, dim3(count), dim3(MwShape<N1>::THREADS), 0, 0, trees, filt, tree_of, ids, par, ch, offs);
        MWG_LAUNCHED();
        return MWG_OK;
    }
};
template <int N1> struct ReconL {
    static mwg_status run(const double *filt, double *coef, const long long *po, const long long *co, int count, long long stride) {
        ProfileScope prof_(MWG_KERNEL_RECONSTRUCT);
        hipLaunchKernelGGL(k_reconstruct_add<N1>, dim3(count), dim3(MwShape<N1>::THREADS), 0, 0, filt, coef, po, co, stride);
        MWG_LAUNCHED();
        return MWG_OK;
    }
};
template <int N1> struct CompressL {
    static mwg_status run(const double *filt, double *coef, const long long *po, const long long *co, int count, long long stride) {
        ProfileScope prof_(MWG_KERNEL_COMPRESS);
        hipLaunchKernelGGL(k_compress<N1>, dim3(count), dim3(MwShape<N1>::THREADS), 0, 0, filt, coef, po, co, stride);
        MWG_LAUNCHED();
        return MWG_OK;
    }
};
template <int N1> struct NormsL {
    static mwg_status run(const double *coef, const long long *off, double *norms, int count) {
        ProfileScope prof_(MWG_KERNEL_NORMS);
        hipLaunchKernelGGL(k_node_norms<N1>, dim3(count), dim3(kThreads), 0, 0, coef, off, norms);
        MWG_LAUNCHED();
        return MWG_OK;
    }
};

} // namespace

} // namespace mwgdev

using namespace mwgdev;

extern "C" {

mwg_status mwg_generate_nodes(const mwg_ftree *f, const double *filters, const int *ids, const int *parent, const int *child_idx, int count) {
    if (need_init() != MWG_OK) return MWG_ERR_ARG;
    if (count <= 0) return MWG_OK;
    if (!f || !filters || !ids || !parent || !child_idx) return fail(MWG_ERR_ARG, "null argument");
    return dispatch<GenerateL>(f->kp1, f, filters, ids, parent, child_idx, count, (const long long *)nullptr, (long long *)nullptr,
                               (unsigned char *)nullptr);
}

mwg_status mwg_generate_nodes_recorded(const mwg_ftree *f, const double *filters, const int *ids, const int *parent, const int *child_idx,
                                       const long long *offs, long long *coef_off_w, unsigned char *is_gen_w, int count) {
    if (need_init() != MWG_OK) return MWG_ERR_ARG;
    if (count <= 0) return MWG_OK;
    if (!f || !filters || !ids || !parent || !child_idx || !offs || !coef_off_w || !is_gen_w) return fail(MWG_ERR_ARG, "null argument");
    if (coef_off_w != f->coef_off || is_gen_w != f->is_gen) return fail(MWG_ERR_ARG, "recorded offsets and flags must be the tree's own arrays");
    return dispatch<GenerateL>(f->kp1, f, filters, ids, parent, child_idx, count, offs, coef_off_w, is_gen_w);
}

mwg_status mwg_generate_nodes_multi(int kp1, const mwg_gen_tree *trees, int ntrees, const double *filters, const int *tree_of, const int *ids,
                                    const int *parent, const int *child_idx, const long long *offs, int count) {
    if (need_init() != MWG_OK) return MWG_ERR_ARG;
    if (count <= 0) return MWG_OK;
    if (!trees || ntrees <= 0 || !filters || !tree_of || !ids || !parent || !child_idx || !offs) return fail(MWG_ERR_ARG, "null argument");
    return dispatch<GenerateMultiL>(kp1, trees, filters, tree_of, ids, parent, child_idx, offs, count);
}

mwg_status mwg_reconstruct_add(int kp1, const double *filters, double *coef, const long long *parent_off, const long long *child_off, int count,
                               long long stride) {
    if (need_init() != MWG_OK) return MWG_ERR_ARG;
    if (count <= 0) return MWG_OK;
    if (!filters || !coef || !parent_off || !child_off) return fail(MWG_ERR_ARG, "null argument");
    return dispatch<ReconL>(kp1, filters, coef, parent_off, child_off, count, stride);
}

mwg_status mwg_compress(int kp1, const double *filters, double *coef, const long long *parent_off, const long long *child_off, int count,
                        long long stride) {
    if (need_init() != MWG_OK) return MWG_ERR_ARG;
    if (count <= 0) return MWG_OK;
    if (!filters || !coef || !parent_off || !child_off) return fail(MWG_ERR_ARG, "null argument");
    return dispatch<CompressL>(kp1, filters, coef, parent_off, child_off, count, stride);
}

mwg_status mwg_node_norms(int kp1, const double *coef, const long long *off, double *norms, int count) {
    if (need_init() != MWG_OK) return MWG_ERR_ARG;
    if (count <= 0) return MWG_OK;
    if (!coef || !off || !norms) return fail(MWG_ERR_ARG, "null argument");
    return dispatch<NormsL>(kp1, coef, off, norms, count);
}

} // extern "C"
