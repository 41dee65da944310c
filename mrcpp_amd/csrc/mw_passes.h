// Separable 3D multiwavelet passes on the matrix cores.
//
// A pass contracts, for one direction d, the two children of that direction
// and their N1 functions with a 2 N1 x 2 N1 matrix M:
//   out(b, j) = sum_(c, i) M((b, j), (c, i)) in(c, i)
// for the 4 N1^2 rows that the other two child bits and the other two indices
// make; M is the four filter blocks (H, G of either child) side by side.  The
// sum is one chain of fused multiply-adds in i order per child and the two
// chains' sum (one chain over both loses a quarter of a bit at order 7).  The index
// that was contracted becomes the slowest of a block, so three passes give the
// original order again.
//
// v_mfma_f64_4x4x4, the matrix on the left: its four blocks take 16
// consecutive rows, the outputs go in N1 / 2 tiles of 4, the terms in N1 / 2 steps
// of 4 (at orders 5 and 9 the middle step belongs to both children and is
// taken twice, the other child's terms as zeros); 2 N1 and 4 N1^2 fit without
// padding at every order.  A result tile lies across the lanes as an input
// step does, so a map between values and coefficients (N1 x N1 for either
// child) follows or precedes the filters in registers.  A wave holds M (up to 50
// registers) and takes one or two of the N1^2 / 4 row tiles, reading each input
// value once: on the vector units a pass read one LDS word per multiply-add and
// was bound by that (order 9: 1.3 MB a node and pass; now 64 KB).
#pragma once
#include "device_common.h"

namespace mwgdev {

template <int N1> struct MwShape {
    static constexpr int N2 = N1 * N1, N3 = N2 * N1, T = N1 / 2, ITEMS = N2 / 4;
    // one row tile per wave at orders 3 and 5; two at order 9 (25 tiles) and at
    // order 7, where two workgroups of 8 waves on a CU overlap each other's
    // loads and stores (an order-7 compression launch: 10.8 us with one of 16, 8.4)
    static constexpr int WAVES = N1 == 10 ? 13 : N1 == 8 ? 8 : ITEMS, PER = (ITEMS + WAVES - 1) / WAVES, THREADS = 64 * WAVES;
    // row stride in LDS: the 16 rows and two terms that half a wave reads fall
    // on different banks for strides 6 and 10; 9 leaves a few pairs at order 7
    // but lets two workgroups' buffers into a CU
    static constexpr int S = N1 == 4 ? 6 : N1 == 8 ? 9 : N1, B = N2 * S, SIZE = 8 * B;
    // waves per SIMD for the register budget: one workgroup of 13 waves, two of 8
    // or 9
    static constexpr int OCC = N1 == 6 ? 5 : 4;
    static_assert(THREADS >= kThreads && THREADS <= 1024 && N2 % 4 == 0, "multiwavelet pass shape");
    // element i of row r of a block; element (j, r) as a pass leaves it
    static __device__ __forceinline__ int at(int blk, int r, int i) { return blk * B + r * S + i; }
    static __device__ __forceinline__ int at_out(int blk, int j, int r) { return blk * B + (j * N1 + r / N1) * S + r % N1; }
    static __device__ __forceinline__ int at_elem(int blk, int e) { return blk * B + (e / N1) * S + e % N1; }
};

// At orders 7 and 9 the matrix leaves no registers for addresses kept from one
// pass to the next: each pass forms its own.
template <int N1> __device__ __forceinline__ int mw_lane() {
    int lane = threadIdx.x & 63;
    if constexpr (N1 >= 8) asm volatile("" : "+v"(lane));
    return lane;
}

// M((b, j), (c, i)) for the wave's lanes
template <int N1> struct MwMatrix {
    static constexpr int T = N1 / 2;
    double m[T][T];
    // base 0: compression, 4: reconstruction (the filter array holds
    // H0t, H1t, G0t, G1t, H0, G0, H1, G1)
    __device__ __forceinline__ void filters(const double *filt, int base) {
        const int lane = mw_lane<N1>();
#pragma unroll
        for (int J = 0; J < T; J++)
#pragma unroll
            for (int K = 0; K < T; K++) {
                const int o = 4 * J + (lane & 3), k = 4 * K + (lane >> 4), b = o >= N1, c = k >= N1;
                m[J][K] = filt[(base + 2 * b + c) * (N1 * N1) + N1 * (o - b * N1) + k - c * N1];
            }
    }
};

// the block of the other two child bits (bit DIM clear)
template <int DIM> __device__ __forceinline__ int mw_spread(int combo) {
    return DIM == 0 ? combo << 1 : DIM == 1 ? (combo & 1) | (combo & 2) << 1 : combo;
}

// The maps between values and coefficients (N1 x N1, out j = sum_i in i m[N1 j +
// i]) for both children, a 2 N1 x 2 N1 block-diagonal matrix: in registers but
// at order 9, where it stays in LDS.
template <int N1> constexpr bool mw_map_tile(int J, int K) { // not wholly another child's
    return (4 * J) / N1 <= (4 * K + 3) / N1 && (4 * K) / N1 <= (4 * J + 3) / N1;
}
template <int N1> struct MwMap {
    static constexpr int T = N1 / 2, W = 2 * N1;
    static constexpr bool LDS = N1 == 10;
    static constexpr int STORE = LDS ? W * W : 1; // doubles of LDS
    double m[LDS ? 1 : T][T];
    const double *lds;
    // store: STORE doubles of LDS; a barrier has to follow
    __device__ __forceinline__ void load(const double *map, double *store) {
        lds = store;
        if constexpr (LDS) {
            for (int o = threadIdx.x; o < W * W; o += MwShape<N1>::THREADS) {
                const int b = o / W >= N1, j = o / W - b * N1, c = o % W >= N1, i = o % W - c * N1;
                store[o] = b == c ? map[N1 * j + i] : 0.0;
            }
        } else {
            const int lane = threadIdx.x & 63;
#pragma unroll
            for (int J = 0; J < T; J++)
#pragma unroll
                for (int K = 0; K < T; K++)
                    if (mw_map_tile<N1>(J, K)) {
                        const int o = 4 * J + (lane & 3), k = 4 * K + (lane >> 4), b = o >= N1, c = k >= N1;
                        const double v = map[N1 * (o - b * N1) + k - c * N1];
                        m[J][K] = b == c ? v : 0.0;
                    }
        }
    }
    // output tile J of the map on a
    __device__ __forceinline__ double tile(int J, const double (&a)[T], int lane) const {
        double t = 0.0;
#pragma unroll
        for (int K = 0; K < T; K++)
            if (mw_map_tile<N1>(J, K)) {
                const double f = LDS ? lds[(4 * J + (lane & 3)) * W + 4 * K + (lane >> 4)] : m[LDS ? 0 : J][K];
                t = __builtin_amdgcn_mfma_f64_4x4x4f64(f, a[K], t, 0, 0, 0);
            }
        return t;
    }
};
struct MwNoMap {};

enum MwMapped { MW_NO_MAP, MW_MAP_BEFORE, MW_MAP_AFTER, MW_APART };

// One pass in direction DIM.  in(block, r, i): the input values; out(q, J,
// block, j, r, v): the outputs, q and J counting a lane's own; with MW_APART
// out(q, J, block, j, r, v0, v1), the sums over either child not yet added.
// Every thread of the workgroup calls; barriers are the caller's.
template <int N1, int DIM, MwMapped MAP = MW_NO_MAP, class Map = MwNoMap, class In, class Out>
__device__ __forceinline__ void mw_pass(const MwMatrix<N1> &M, In in, Out out, const Map &map = Map()) {
    using P = MwShape<N1>;
    constexpr int T = P::T, MID = N1 % 4 ? T / 2 : -1; // the step of both children
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = mw_lane<N1>();
    const int row = lane & 15, kk = lane >> 4;
#pragma unroll
    for (int q = 0; q < P::PER; q++) {
        const int item = wave + P::WAVES * q;
        if (P::ITEMS % P::WAVES != 0 && item >= P::ITEMS) break;
        const int g = 16 * item + row, combo = g / P::N2, blk = mw_spread<DIM>(combo), r = g - combo * P::N2;
        double a[T];
#pragma unroll
        for (int K = 0; K < T; K++) {
            const int k = 4 * K + kk, c = k >= N1;
            a[K] = in(blk | c << DIM, r, k - c * N1);
        }
        if constexpr (MAP == MW_MAP_BEFORE) {
            double t[T];
#pragma unroll
            for (int J = 0; J < T; J++) t[J] = map.tile(J, a, lane);
#pragma unroll
            for (int J = 0; J < T; J++) a[J] = t[J];
        }
        double d[T], e[MAP == MW_APART ? T : 1];
#pragma unroll
        for (int J = 0; J < T; J++) {
            double d0 = 0.0, d1 = 0.0;
#pragma unroll
            for (int K = 0; K < T; K++) {
                const double lo = K == MID ? (kk < 2 ? a[K] : 0.0) : a[K], hi = K == MID ? (kk < 2 ? 0.0 : a[K]) : a[K];
                if (4 * K < N1) d0 = __builtin_amdgcn_mfma_f64_4x4x4f64(M.m[J][K], lo, d0, 0, 0, 0);
                if (4 * K + 3 >= N1) d1 = __builtin_amdgcn_mfma_f64_4x4x4f64(M.m[J][K], hi, d1, 0, 0, 0);
            }
            if constexpr (MAP == MW_APART) {
                d[J] = d0;
                e[J] = d1;
            } else {
                d[J] = d0 + d1;
            }
            if constexpr (N1 == 10) __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int J = 0; J < T; J++) {
            const int o = 4 * J + kk, b = o >= N1;
            if constexpr (MAP == MW_APART) {
                out(q, J, blk | b << DIM, o - b * N1, r, d[J], e[J]);
            } else {
                double v = d[J];
                if constexpr (MAP == MW_MAP_AFTER) v = map.tile(J, d, lane);
                out(q, J, blk | b << DIM, o - b * N1, r, v);
            }
        }
    }
}

// What a lane's own outputs of a pass are: own(q, J, block, j, r).
template <int N1, int DIM, class Own> __device__ __forceinline__ void mw_own(Own own) {
    using P = MwShape<N1>;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = mw_lane<N1>();
#pragma unroll
    for (int q = 0; q < P::PER; q++) {
        const int item = wave + P::WAVES * q;
        if (P::ITEMS % P::WAVES != 0 && item >= P::ITEMS) break;
        const int g = 16 * item + (lane & 15), combo = g / P::N2, blk = mw_spread<DIM>(combo), r = g - combo * P::N2;
#pragma unroll
        for (int J = 0; J < P::T; J++) {
            const int o = 4 * J + (lane >> 4), b = o >= N1;
            own(q, J, blk | b << DIM, o - b * N1, r);
        }
    }
}

// from one LDS buffer to another
template <int N1, int DIM, MwMapped MAP = MW_NO_MAP, class Map = MwNoMap>
__device__ __forceinline__ void mw_pass_lds(double *out, const double *in, const MwMatrix<N1> &M, const Map &map = Map()) {
    using P = MwShape<N1>;
    mw_pass<N1, DIM, MAP, Map>(
        M, [&](int t, int r, int i) { return in[P::at(t, r, i)]; },
        [&](int, int, int t, int j, int r, double v) { out[P::at_out(t, j, r)] = v; }, map);
}

// Component norms of a node in LDS to nrm[0..8] (8 norms + square norm): a wave
// per block.  Every thread calls; red: 8 doubles of LDS.
template <int N1> __device__ __forceinline__ void mw_norms(const double *c, double *nrm, double *red) {
    using P = MwShape<N1>;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int t = wave; t < 8; t += P::WAVES) {
        double v = 0.0;
        for (int e = lane; e < P::N3; e += 64) {
            const double x = c[P::at_elem(t, e)];
            v += x * x;
        }
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        if (lane == 0) red[t] = v;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double tot = 0.0;
        for (int t = 0; t < 8; t++) {
            const double nv = sqrt(red[t]);
            nrm[t] = nv;
            tot += nv * nv;
        }
        nrm[8] = tot;
    }
}

// Values in a -> the node's scaling and wavelet blocks at dst, and its norms.
// A barrier has to stand between the caller's last writes (a, the map's store) or
// reads (b) and this.
template <int N1>
__device__ __forceinline__ void mw_values_to_node(double *a, double *b, const double *filt, const MwMap<N1> &vc, double *dst, double *nrm, double *red) {
    using P = MwShape<N1>;
    MwMatrix<N1> M;
    M.filters(filt, 0);
    mw_pass_lds<N1, 0, MW_MAP_BEFORE>(b, a, M, vc);
    __syncthreads();
    mw_pass_lds<N1, 1, MW_MAP_BEFORE>(a, b, M, vc);
    __syncthreads();
    mw_pass_lds<N1, 2, MW_MAP_BEFORE>(b, a, M, vc);
    __syncthreads();
    for (int o = threadIdx.x; o < 8 * P::N3; o += P::THREADS) dst[o] = b[P::at_elem(o / P::N3, o % P::N3)];
    mw_norms<N1>(b, nrm, red);
}

} // namespace mwgdev
