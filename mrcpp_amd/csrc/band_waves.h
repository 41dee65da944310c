// Band sums with one wave per work item (FP64 at every order, FP32 at order 7; long
// levels of order 7 have a kernel of their own, k_band_rows).
//
// A work item is a unit and one column set of its output: the x sweep's output
// columns (gx, j0) are divided into sets of four, and a wave runs all three
// sweeps of a unit's groups for its own set.  Nothing crosses waves, so there
// is no workgroup barrier anywhere: a wave's 16x16x4 (or 4x4x4, four blocks)
// products of one group overlap with its neighbours' LDS and operand latency.
//
// Measured per apply against the kernels before (MI355X; workgroups of four
// waves exchanging T1 and T2 through LDS with one or two barriers a group,
// 16x16x4 products at every order): 16-Gaussian Poisson order 7 1.86 -> 1.58 ms
// (FP64) and 1.48 -> 1.33 (FP32); one Gaussian, order 3 0.236 -> 0.106, order 5
// 0.646 -> 0.36, order 9 (Helmholtz) 5.55 -> 2.35 ms.  Large order-7 launches
// keep the matrix cores 0.69 busy (0.68 before, with 7% more products); with
// the operands in registers and nothing else to do the same products reach 0.9.
// Any register spilled inside the group loop costs more than it saves: its
// reload waits for every operand load in flight (order 9: 4.4 ms with 40 spilled
// words, 2.35 without).
//
// Between the sweeps the data stay in registers wherever the instructions'
// layouts meet.  A result D of a matrix product has its row index in the
// lane's quarter (lane / 16) and register, its column in the low lane bits; an
// operand has the contracted index in the quarter.  A sweep whose D rows are
// the next sweep's contracted index therefore feeds it without a move: that
// holds for y -> z (rows i2), with the y sweep written as [T1 rows] x
// [Oy columns] and the z sweep as [Oz^T rows] x [T2 columns].  x -> y needs one
// transposition, through LDS private to the wave.
//
// Every output element goes through the same products as in k_band_mfma, at order
// 7 in the same order (f64 and f32 products on the matrix cores are one fused
// multiply-add per contracted index, in index order, whichever instruction shape
// forms them), so order 7 gives the same bits with either.  At orders 3, 5 and 9
// the z product of a group that does not fill its mask is formed from zero and
// then added.
//
// Results: a node's first unit is written to the node itself, each further unit
// to a slot in the order of WaveMap, which each wave writes in whole 512-byte
// rows; the reductions add the slots to the node in unit order.  The first of
// several units writes the node in the slots' order too where a workgroup of the
// reduction can put it right in place (orders 3 and 7).
#pragma once

namespace mwgdev {

namespace {

typedef double dvec2 __attribute__((ext_vector_type(2)));
// Pointers formed from record words are marked global: a flat load would also
// count as an LDS access and every LDS wait would wait for it.
template <typename T> using global = __attribute__((address_space(1))) T;

// Column sets of a unit (work items per unit) and values per set and lane.
template <int N1> struct WaveShape {
    static constexpr int N2 = N1 * N1, N3 = N2 * N1;
    static constexpr int SETS = N1 / 2; // of four (gx, j0) columns
    static constexpr int PER_WAVE = N1 == 4 ? 2 : 1;   // sets of one item
    static constexpr int ITEMS = SETS / PER_WAVE;       // items per unit
    static constexpr int VALS = 8 * N3 / (64 * ITEMS);  // result values per lane of an item
};

// Value v (register index) of item `it`: row(it, v), its 64 lanes' place in a
// partial slot, slot[64 row + lane]; out(it, v, lane), a lane's output element
// (gt block, j0, j1, j2).  At order 7 the four (FP64) or eight (FP32) rows that
// hold every j0 and j1 of their outputs lie where those outputs lie in a node, at
// orders 5 and 9 the rows of every j0 follow each other.
template <int N1, int PREC> struct WaveMap {
    using S = WaveShape<N1>;
    static constexpr int TC = N1 / 2; // tiles of four columns or rows of one 2 N1 side
    static constexpr bool IN_PLACE = N1 == 4 || N1 == 8;
    static constexpr int SET = N1 != 8 ? S::ITEMS : PREC == MWG_PREC_FP64 ? 4 : 8; // rows of a workgroup of the reduction
    __device__ static inline int row(int it, int v) {
        if constexpr (N1 != 8) return v * S::ITEMS + it;
        const int gx = it >> 1, half = it & 1, t = v >> 2, r = v & 3;
        if constexpr (PREC == MWG_PREC_FP64) return (gx + 2 * (t & 1) + 4 * (r >> 1)) * 8 + 4 * (r & 1) + 2 * half + (t >> 1);
        return (gx + 2 * t) * 8 + 4 * half + r;
    }
    __device__ static inline int out(int it, int v, int lane) {
        int gx, gy, gz, j0, j1, j2;
        if constexpr (N1 == 8) {
            gx = it >> 1;
            const int r = v & 3, t = v >> 2, q = lane >> 4;
            const int row = PREC == MWG_PREC_FP64 ? q + 4 * r : 4 * q + r;
            gz = row >> 3;
            j2 = row & 7;
            j1 = lane & 7;
            const int h = (lane >> 3) & 1;
            if (PREC == MWG_PREC_FP64) { // t = 2 p + gy, lanes (j0', j1)
                gy = t & 1;
                j0 = 4 * (it & 1) + 2 * (t >> 1) + h;
            } else { // t = j0 within the set, lanes (gy, j1)
                gy = h;
                j0 = 4 * (it & 1) + t;
            }
        } else {
            // lane j + 4 b + 16 i: column 4 tc + j = (gy, j1), row 4 tr + i = (gz, j2), b = 2 gx + (j0 - 2 set)
            const int set = it * S::PER_WAVE + v / (TC * TC), t = v % (TC * TC);
            const int m = 4 * (t % TC) + (lane & 3), n = 4 * (t / TC) + (lane >> 4), b = (lane >> 2) & 3;
            gx = b >> 1;
            j0 = 2 * set + (b & 1);
            gy = m / N1;
            j1 = m % N1;
            gz = n / N1;
            j2 = n % N1;
        }
        return (gx + 2 * gy + 4 * gz) * S::N3 + j0 + N1 * j1 + S::N2 * j2;
    }
};

struct WaveArgs {
    const int2 *group; // group codes and pair indices, level order
    const int4 *pdl;   // of a pair: translation differences, offset of the band node
    const long long *pfo;
    const int *unit; // WaveRecords
    const long long *uscan;
    int L;
};

// One group of an item: gt mask, operand blocks of the three directions, band block.
struct WaveGroup {
    unsigned mask;
    int bx, by, bz;
    const global<double> *f;
};

// The groups of a work unit that touch the wave's columns (bits `want` of
// their gt masks), in order.  64 at a time in registers, lane j holding group
// c0 + j: x block | gt mask << 24, y block | f bits 32-42 << 21, z block | f bits
// 43-53 << 21, f bits 0-31; a block is 2 (b40 + dl) + f bit of its direction (21
// bits), f the offset of the group's band block.  Units are dealt out in turn: one
// shared counter served a small level's waves more slowly than they worked (86 us
// a launch at order 3 against 20).
template <int N1> struct WaveUnit {
    const WaveArgs &a;
    unsigned long long frag, coef; // operand table, coefficient pool
    global<double> *out;           // result: the unit's slot or the output node
    int gi0, ng, c0;
    unsigned want;
    bool direct;
    int4 rec;
    unsigned long long todo;

    __device__ WaveUnit(const WaveArgs &a_, int u, unsigned want_, int lane) : a(a_), c0(0), want(want_ << 24) {
        const auto d = ro(a.unit) + kUnitInts * (size_t)u;
        auto ptr = [](int lo, int hi) { return ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo; };
        frag = ptr(d[0], d[1]);
        coef = ptr(d[2], d[3]);
        out = (global<double> *)ptr(d[4], d[5]);
        gi0 = d[6];
        ng = d[7];
        direct = d[8] != 0;
        load(lane);
    }
    __device__ void load(int lane) {
        rec = int4{0, 0, 0, 0};
        if (c0 + lane < ng) {
            const int2 g = a.group[gi0 + c0 + lane];
            const int4 d = a.pdl[g.y];
            const unsigned code = (unsigned)g.x;
            const int ft = code_ft(code), b = code_block(code);
            const long long f = a.pfo[g.y] + (long long)ft * (N1 * N1 * N1);
            const unsigned fh = (unsigned)(f >> 32);
            rec.x = (int)((unsigned)((b + d.x) * 2 + (ft & 1)) | (code_mask(code) << 24));
            rec.y = (int)((unsigned)((b + d.y) * 2 + ((ft >> 1) & 1)) | (fh << 21));
            rec.z = (int)((unsigned)((b + d.z) * 2 + ((ft >> 2) & 1)) | ((fh >> 11) << 21));
            rec.w = (int)(unsigned)f;
        }
        todo = __ballot(((unsigned)rec.x & want) != 0u);
    }
    __device__ bool next(int lane, WaveGroup &q) {
        while (todo == 0ull) {
            c0 += 64;
            if (c0 >= ng) return false;
            load(lane);
        }
        const int j = __builtin_ctzll(todo);
        todo &= todo - 1ull;
        const unsigned x = (unsigned)__builtin_amdgcn_readlane(rec.x, j), y = (unsigned)__builtin_amdgcn_readlane(rec.y, j),
                       z = (unsigned)__builtin_amdgcn_readlane(rec.z, j), w = (unsigned)__builtin_amdgcn_readlane(rec.w, j);
        q.mask = x >> 24;
        q.bx = (int)(x & 0x1fffffu);
        q.by = (int)(y & 0x1fffffu);
        q.bz = (int)(z & 0x1fffffu);
        const int fh = (int)((y >> 21) | ((z >> 21) << 11)) << 10 >> 10; // 22 bits, signed
        q.f = (const global<double> *)coef + (long long)(((unsigned long long)(unsigned)fh << 32) | w);
        return true;
    }
};

// An item's result values into the unit's slot or the output node, in the node's order (direct) or the slots'.
template <int N1, int PREC, typename V> __device__ inline void wave_store(global<double> *out, bool direct, int it, int lane, V &&value) {
    constexpr int VALS = WaveShape<N1>::VALS;
    asm volatile("" : "+v"(lane)); // the addresses are formed here, not kept in registers over the groups
    if (direct) {
#pragma unroll
        for (int v = 0; v < VALS; v++) out[WaveMap<N1, PREC>::out(it, v, lane)] = value(v);
    } else {
#pragma unroll
        for (int v = 0; v < VALS; v++) out[WaveMap<N1, PREC>::row(it, v) * 64 + lane] = value(v);
    }
}

// Units in turn over the workgroups.  Workgroup b runs on XCD b % 8 (each XCD
// has its own L2): with ITEMS one-wave workgroups to a unit, workgroups b,
// b + 8, ... take the unit's items, so that they read its operands through one L2.
template <int ITEMS> struct WaveTurn {
    int unit, it, step;
    __device__ WaveTurn() {
        const int b = blockIdx.x, k = b >> 3;
        it = k % ITEMS;
        unit = (k / ITEMS) * 8 + (b & 7);
        step = gridDim.x / ITEMS; // the grid is a multiple of 8 ITEMS
    }
};

__device__ inline void wave_fence() { __atomic_signal_fence(__ATOMIC_SEQ_CST); }

__device__ inline double mma4(double a, double b, double c) { return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0); }

// ---------------------------------------------------------------------------
// Order 7, FP64.  Item = (unit, gx, j0 / 4), a workgroup's four waves taking
// the four items of a unit (they read the same operands at about the same time,
// through one L1): a group without gx in its mask is passed over.  x: 64 lines x 4
// columns, eight 4x4x4 products from the band block held in registers; y: per gy,
// j0 pair and i2 tile, 4x4x4 products whose
// result lanes are (j0', j1) x i2 quarter; z: 16x16x4 into [j0 pair][gy].
// T1[j0][i2][i1] in LDS at 84 j0 + 10 i2 + 2 (i1 & 3) + (i1 >> 2): both k
// steps of an operand in one 16-byte read.  The counters still put half of the LDS
// cycles down to bank conflicts (a third at FP32), while the waves wait 0.13 of theirs
// for anything.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256, 4) void k_band_waves8(WaveArgs a) {
    constexpr int SJ = 84, SI = 10;
    __shared__ __align__(16) double sAll[4][4 * SJ];
    const int lane = threadIdx.x & 63, it = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double *const sT1 = sAll[it];
    const int li = lane & 15, lq = lane >> 4;
    const int total = unit_first(ro(a.uscan)[a.L]);
    const int gx = it >> 1, j0b = 4 * (it & 1);
    const int tw = (lane & 3) * SJ + ((lane >> 3) & 1) * SI + 2 * lq + ((lane >> 2) & 1);
    const int tr = ((lane >> 3) & 1) * SJ + (lane & 3) * SI + 2 * lq;
    const int ox = (lane & 3) + 16 * lq, oy = (lane & 7) + 16 * lq;
    struct Ops {
        double x[2], y[2][2], z[2];
    };
    for (int unit = blockIdx.x; unit < total; unit += gridDim.x) {
        WaveUnit<8> w(a, unit, 0x55u << gx, lane);
        dvec4 acc[2][2];
#pragma unroll
        for (int t = 0; t < 4; t++) acc[t >> 1][t & 1] = dvec4{0.0, 0.0, 0.0, 0.0};
        double fa[4][2];
        auto load_f = [&](const global<double> *src) {
#pragma unroll
            for (int b = 0; b < 4; b++)
#pragma unroll
                for (int ks = 0; ks < 2; ks++) fa[b][ks] = src[8 * (16 * b + li) + 4 * ks + lq];
        };
        auto load_ops = [&](const WaveGroup &q, Ops &o) {
            const auto frag = (const global<double> *)w.frag;
            const auto x = frag + (size_t)q.bx * 128 + 8 * gx + j0b, y = frag + (size_t)q.by * 128, z = frag + (size_t)q.bz * 128;
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                o.x[ks] = x[64 * ks + ox];
                o.y[0][ks] = y[64 * ks + oy];
                o.y[1][ks] = y[64 * ks + 8 + oy];
                o.z[ks] = z[64 * ks + lane];
            }
        };
        WaveGroup ga, gb;
        Ops oa, ob;
        auto step = [&](const WaveGroup &q, const Ops &o, WaveGroup &nq, Ops &no) -> bool {
            double d[4];
#pragma unroll
            for (int b = 0; b < 4; b++) d[b] = mma4(fa[b][0], o.x[0], 0.0);
#pragma unroll
            for (int b = 0; b < 4; b++) d[b] = mma4(fa[b][1], o.x[1], d[b]);
            // the group's operands arrive before anything new is requested, so
            // that no wait below queues behind the next group's loads
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                settled(o.y[0][ks]);
                settled(o.y[1][ks]);
                settled(o.z[ks]);
            }
            const bool more = w.next(lane, nq);
            if (more) {
                if (nq.f != q.f) load_f(nq.f);
                load_ops(nq, no);
            }
#pragma unroll
            for (int b = 0; b < 4; b++) sT1[tw + 2 * SI * b] = d[b];
            wave_fence();
            dvec2 t1[2][2]; // [j0 pair][i2 tile], both k steps
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int ti = 0; ti < 2; ti++) t1[p][ti] = *reinterpret_cast<const dvec2 *>(sT1 + tr + 2 * SJ * p + 4 * SI * ti);
            wave_fence();
#pragma unroll
            for (int gy = 0; gy < 2; gy++) {
                const unsigned m2 = q.mask >> (gx + 2 * gy); // bit 0: gz = 0, bit 4: gz = 1
                if (!(m2 & 0x11u)) continue;
                const bool keep = (m2 >> (4 * (li >> 3))) & 1u;
                const double z0 = keep ? o.z[0] : 0.0, z1 = keep ? o.z[1] : 0.0;
                double t2[2][2];
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int ti = 0; ti < 2; ti++) t2[p][ti] = mma4(t1[p][ti].x, o.y[gy][0], 0.0);
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int ti = 0; ti < 2; ti++) t2[p][ti] = mma4(t1[p][ti].y, o.y[gy][1], t2[p][ti]);
#pragma unroll
                for (int p = 0; p < 2; p++) acc[p][gy] = Mfma<double>::mma(z0, t2[p][0], acc[p][gy]);
#pragma unroll
                for (int p = 0; p < 2; p++) acc[p][gy] = Mfma<double>::mma(z1, t2[p][1], acc[p][gy]);
            }
            return more;
        };
        if (w.next(lane, ga)) {
            load_f(ga.f);
            load_ops(ga, oa);
            while (step(ga, oa, gb, ob) && step(gb, ob, ga, oa)) {
            }
        }
        wave_store<8, MWG_PREC_FP64>(w.out, w.direct, it, lane, [&](int v) { return acc[v >> 3][(v >> 2) & 1][v & 3]; });
    }
}

// ---------------------------------------------------------------------------
// Order 7, FP32 operands and products, every group's product added in FP64.
// x: 4x4x1 products, sixteen line tiles at once, a lane holding its line of the
// band block; y: 16x16x4 with the rows (j0', i2) numbered so that register
// ks + 2 j0' of quarter q holds i2 = 4 ks + q, the z sweep's operand; z: 16x16x4
// per j0, rows (gz, j2), columns (gy, j1), the lanes of an unmasked (gy, gz)
// added.  T1[j0][i2][i1] in LDS at 104 j0 + 12 i2 + i1.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256, 4) void k_band_waves8f(WaveArgs a) {
    constexpr int SJ = 104, SI = 12;
    __shared__ __align__(16) float sAll[4][4 * SJ];
    const int lane = threadIdx.x & 63, it = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float *const sT1 = sAll[it];
    const int li = lane & 15, lq = lane >> 4;
    const int total = unit_first(ro(a.uscan)[a.L]);
    const int gx = it >> 1, j0b = 4 * (it & 1);
    const int tw = (lane & 3) * SJ + (lane >> 3) * SI + 4 * ((lane >> 2) & 1);
    const int tr = ((li >> 1) & 1) * SJ + (4 * (li & 1) + (li >> 2)) * SI + lq;
    struct Ops {
        float x[8], y[2], z[2];
    };
    for (int unit = blockIdx.x; unit < total; unit += gridDim.x) {
        WaveUnit<8> w(a, unit, 0x55u << gx, lane);
        dvec4 acc[4];
#pragma unroll
        for (int t = 0; t < 4; t++) acc[t] = dvec4{0.0, 0.0, 0.0, 0.0};
        double fa[8]; // converted as they are used, so that the loads stay in flight
        auto load_f = [&](const global<double> *src) {
            src += 8 * lane;
#pragma unroll
            for (int k = 0; k < 8; k++) fa[k] = src[k];
        };
        auto load_ops = [&](const WaveGroup &q, Ops &o) {
            const auto frag = (const global<float> *)w.frag;
            const auto x = frag + (size_t)q.bx * 128 + 8 * gx + j0b + (lane & 3), y = frag + (size_t)q.by * 128 + lane,
                       z = frag + (size_t)q.bz * 128 + lane;
#pragma unroll
            for (int k = 0; k < 8; k++) o.x[k] = x[64 * (k >> 2) + 16 * (k & 3)];
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                o.y[ks] = y[64 * ks];
                o.z[ks] = z[64 * ks];
            }
        };
        WaveGroup ga, gb;
        Ops oa, ob;
        auto step = [&](const WaveGroup &q, const Ops &o, WaveGroup &nq, Ops &no) -> bool {
            fvec4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < 8; k++) d = __builtin_amdgcn_mfma_f32_4x4x1f32((float)fa[k], o.x[k], d, 0, 0, 0);
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                settled(o.y[ks]);
                settled(o.z[ks]);
            }
            const bool more = w.next(lane, nq);
            if (more) {
                if (nq.f != q.f) load_f(nq.f);
                load_ops(nq, no);
            }
            *reinterpret_cast<fvec4 *>(sT1 + tw) = d;
            wave_fence();
            float t1[2][2];
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int ks = 0; ks < 2; ks++) t1[p][ks] = sT1[tr + 2 * SJ * p + 4 * ks];
            wave_fence();
            const bool keep = (q.mask >> (gx + 2 * (li >> 3) + 4 * (lq >> 1))) & 1u;
            fvec4 t2[2];
#pragma unroll
            for (int p = 0; p < 2; p++) t2[p] = Mfma<float>::mma(t1[p][0], o.y[0], fvec4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
            for (int p = 0; p < 2; p++) t2[p] = Mfma<float>::mma(t1[p][1], o.y[1], t2[p]);
            fvec4 c[4];
#pragma unroll
            for (int t = 0; t < 4; t++) c[t] = Mfma<float>::mma(o.z[0], t2[t >> 1][2 * (t & 1)], fvec4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
            for (int t = 0; t < 4; t++) c[t] = Mfma<float>::mma(o.z[1], t2[t >> 1][2 * (t & 1) + 1], c[t]);
            if (keep)
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[t][r] += (double)c[t][r];
            return more;
        };
        if (w.next(lane, ga)) {
            load_f(ga.f);
            load_ops(ga, oa);
            while (step(ga, oa, gb, ob) && step(gb, ob, ga, oa)) {
            }
        }
        wave_store<8, MWG_PREC_FP32>(w.out, w.direct, it, lane, [&](int v) { return acc[v >> 2][v & 3]; });
    }
}

// ---------------------------------------------------------------------------
// Orders 3, 5 and 9, FP64: 4x4x4 products only.  Four blocks of one instruction
// are the four columns (gx, j0) of a set (j0 = 2 set, 2 set + 1), rows and
// columns go in tiles of four: 2 N1 is a multiple of four at every order, so
// only the contracted index is padded (10 of 12 at order 9, 6 of 8 at order 5)
// where 16x16x4 tiles use 0.46 and 0.42 of their products.
// T1[column][line] in LDS at SJ column + line, line = i1 + N1 i2: positions past
// a line's or the block's end hold other finite values (zero at the start),
// which meet the zero padding of the y and z operands.
// ---------------------------------------------------------------------------
template <int N1> struct WaveLds {
    static constexpr int SJ = N1 == 4 ? 17 : N1 == 6 ? 55 : 123; // few bank conflicts
    static constexpr int WAVES = N1 == 10 ? 2 : 4;                // per SIMD
};

// gt bits that columns (or rows) 4 t .. 4 t + 3 of a 2 N1 side can hold: lo for
// its first N1, hi for the others.
template <int N1> __device__ constexpr unsigned side_mask(int t, unsigned lo, unsigned hi) {
    return (4 * t < N1 ? lo : 0u) | (4 * t + 3 >= N1 ? hi : 0u);
}

template <int N1> __global__ __launch_bounds__(64, WaveLds<N1>::WAVES) void k_band_waves(WaveArgs a) {
    using W = WaveShape<N1>;
    using G = BandGeom<N1, MWG_PREC_FP64>;
    constexpr int N2 = W::N2, N3 = W::N3, PW = W::PER_WAVE;
    constexpr int KS = (N1 + 3) / 4;        // contraction steps (and tiles of i2)
    constexpr int TC = N1 / 2;              // tiles of 2 N1 columns
    constexpr int LB = (N2 + 15) / 16;      // batches of 16 lines
    constexpr int NT = SweepShape<N1>::NT;  // column tiles of the operand table
    constexpr int FRAG = G::KSTEPS * NT * 64;
    constexpr int SJ = WaveLds<N1>::SJ;
    __shared__ double sT1[PW * 4 * SJ];
    // y and z operand blocks at order 9 (60 registers otherwise, more than fit)
    constexpr bool LDS = N1 == 10;
    constexpr int STAGE = LDS ? FRAG / 128 : 1; // 16-byte loads per lane and block
    __shared__ __align__(16) double sOp[LDS ? 2 * FRAG : 2];
    static_assert(16 * LB <= SJ && N1 * (4 * KS - 1) + 4 * KS <= SJ, "every line written and every operand element read lies in its column");
    const int lane = threadIdx.x;
    const int l4 = lane & 3, lb = (lane >> 2) & 3, lq = lane >> 4;
    const int total = unit_first(ro(a.uscan)[a.L]);
    const WaveTurn<W::ITEMS> turn;
    const int it = turn.it;
    for (int i = lane; i < PW * 4 * SJ; i += 64) sT1[i] = 0.0;
    wave_fence();
    const int tw = l4 * SJ + 4 * lb + lq; // column l4, line 16 batch + 4 lb + lq
    // band block elements of a lane: line 16 batch + lane % 16, contracted
    // index 4 ks + lq.  Past N1 they are other elements of the block (the x
    // operand is zero there); the last batch is kept within the block.
    const int fo = N1 * (lane & 15) + lq;
    const int fl = N1 * min(16 * (LB - 1) + (lane & 15), N2 - 1) + lq;
    const int fe = min(fl + 4 * (KS - 1), N3 - 1);
    static_assert(N1 * (16 * (LB - 1) - 1) + 4 * KS - 1 < N3, "the other batches stay within the block");
    static_assert(4 * (KS - 1) <= N1, "only the last step reaches past the line");
    const int tr = lb * SJ + l4 * N1 + lq; // column lb, i2 = 4 tile + l4, i1 = 4 step + lq
    // operand table offset of column n, contracted index 4 ks + lq
    auto at = [&](int n, int ks) { return (ks * NT + (n >> 4)) * 64 + (n & 15) + 16 * lq; };
    for (int unit = turn.unit; unit < total; unit += turn.step) {
        WaveUnit<N1> w(a, unit, 0xffu, lane);
        const auto frag = (const global<double> *)w.frag;
        double acc[PW][TC][TC];
#pragma unroll
        for (int s = 0; s < PW; s++)
#pragma unroll
            for (int t = 0; t < TC * TC; t++) acc[s][t / TC][t % TC] = 0.0;
        double fa[LB][KS], bx[PW][KS], by[LDS ? 1 : TC][KS], az[LDS ? 1 : TC][KS];
        dvec2 stage[2 * STAGE];
        int cx[PW][KS]; // operand columns of the sets: gx N1 + j0
#pragma unroll
        for (int s = 0; s < PW; s++)
#pragma unroll
            for (int ks = 0; ks < KS; ks++) cx[s][ks] = at((l4 >> 1) * N1 + 2 * (it * PW + s) + (l4 & 1), ks);
        auto load_f = [&](const global<double> *src) {
#pragma unroll
            for (int b = 0; b < LB; b++)
#pragma unroll
                for (int ks = 0; ks < KS; ks++)
                    fa[b][ks] = b < LB - 1 ? src[fo + N1 * 16 * b + 4 * ks] : src[ks == KS - 1 ? fe : fl + 4 * ks];
        };
        auto load_x = [&](const WaveGroup &q) {
            const auto x = frag + (size_t)q.bx * FRAG;
#pragma unroll
            for (int s = 0; s < PW; s++)
#pragma unroll
                for (int ks = 0; ks < KS; ks++) bx[s][ks] = x[cx[s][ks]];
        };
        auto load_y = [&](const WaveGroup &q) {
            const auto y = frag + (size_t)q.by * FRAG;
            if constexpr (LDS) {
                const auto z = frag + (size_t)q.bz * FRAG;
#pragma unroll
                for (int k = 0; k < STAGE; k++) stage[k] = ((const global<dvec2> *)y)[64 * k + lane];
#pragma unroll
                for (int k = 0; k < STAGE; k++) stage[STAGE + k] = ((const global<dvec2> *)z)[64 * k + lane];
                return;
            }
#pragma unroll
            for (int t = 0; t < TC; t++)
#pragma unroll
                for (int ks = 0; ks < KS; ks++) by[t][ks] = y[at(4 * t + l4, ks)];
        };
        auto load_z = [&](const WaveGroup &q, int t) {
            if constexpr (LDS) return;
            const auto z = frag + (size_t)q.bz * FRAG;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) az[t][ks] = z[at(4 * t + l4, ks)];
        };
        auto put = [&]() {
            if constexpr (LDS)
#pragma unroll
                for (int k = 0; k < 2 * STAGE; k++) reinterpret_cast<dvec2 *>(sOp)[64 * k + lane] = stage[k];
            wave_fence();
        };
        WaveGroup q, nq;
        bool more = w.next(lane, q);
        if (more) {
            load_f(q.f);
            load_x(q);
            load_y(q);
#pragma unroll
            for (int t = 0; t < TC; t++) load_z(q, t);
            put();
        }
        // Operands have one register set: each is requested again for the next
        // group as soon as this one is done with it (after the last group its
        // own once more, unused, so that every wait is exact).
        while (more) {
            double d[PW][LB];
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
#pragma unroll
                for (int s = 0; s < PW; s++)
#pragma unroll
                    for (int b = 0; b < LB; b++) d[s][b] = mma4(fa[b][ks], bx[s][ks], ks ? d[s][b] : 0.0);
#pragma unroll
            for (int s = 0; s < PW; s++)
#pragma unroll
                for (int b = 0; b < LB; b++) sT1[s * 4 * SJ + tw + 16 * b] = d[s][b];
            wave_fence();
            if constexpr (!LDS)
#pragma unroll
                for (int t = 0; t < TC; t++)
#pragma unroll
                    for (int ks = 0; ks < KS; ks++) {
                        settled(by[t][ks]);
                        settled(az[t][ks]);
                    }
            more = w.next(lane, nq);
            if (!more) nq = q;
            const unsigned gm = q.mask;
            double t2[PW][TC][KS];
#pragma unroll
            for (int s = 0; s < PW; s++) {
                double t1[KS][KS]; // [i2 tile][step]
#pragma unroll
                for (int ti = 0; ti < KS; ti++)
#pragma unroll
                    for (int ks = 0; ks < KS; ks++) t1[ti][ks] = sT1[s * 4 * SJ + tr + 4 * N1 * ti + 4 * ks];
#pragma unroll
                for (int tc = 0; tc < TC; tc++)
                    if (gm & side_mask<N1>(tc, 0x33u, 0xccu))
#pragma unroll
                        for (int ks = 0; ks < KS; ks++) {
                            const double b = LDS ? sOp[at(4 * tc + l4, ks)] : by[LDS ? 0 : tc][ks];
#pragma unroll
                            for (int ti = 0; ti < KS; ti++) t2[s][tc][ti] = mma4(t1[ti][ks], b, ks ? t2[s][tc][ti] : 0.0);
                        }
            }
            wave_fence();
            if (nq.f != q.f) load_f(nq.f);
            load_x(nq);
            load_y(nq);
            auto z_of = [&](int tz, double (&zo)[KS]) {
#pragma unroll
                for (int ti = 0; ti < KS; ti++) zo[ti] = LDS ? sOp[FRAG + at(4 * tz + l4, ti)] : az[LDS ? 0 : tz][ti];
            };
            if (gm == 0xffu) {
#pragma unroll
                for (int tz = 0; tz < TC; tz++) {
                    double zo[KS];
                    z_of(tz, zo);
#pragma unroll
                    for (int ti = 0; ti < KS; ti++)
#pragma unroll
                        for (int s = 0; s < PW; s++)
#pragma unroll
                            for (int tc = 0; tc < TC; tc++) acc[s][tz][tc] = mma4(zo[ti], t2[s][tc][ti], acc[s][tz][tc]);
                    load_z(nq, tz);
                }
            } else {
                // the mask from a lane's gx on, and for tiles across gy or gz
                // from its gy and gz on (formed here, not kept over the groups)
                int l = lane;
                asm volatile("" : "+v"(l));
                unsigned from[2][2];
                from[0][0] = gm >> ((l >> 3) & 1);
                from[1][0] = from[0][0] >> (l & 2);
                from[0][1] = from[0][0] >> ((l >> 3) & 4);
                from[1][1] = from[1][0] >> ((l >> 3) & 4);
#pragma unroll
                for (int tz = 0; tz < TC; tz++) {
                    const bool cz0 = 4 * tz < N1, cz1 = 4 * tz + 3 >= N1;
                    const unsigned zmask = side_mask<N1>(tz, 0x0fu, 0xf0u);
                    double zo[KS];
                    z_of(tz, zo);
                    if (gm & zmask)
#pragma unroll
                        for (int tc = 0; tc < TC; tc++) {
                            const bool cy0 = 4 * tc < N1, cy1 = 4 * tc + 3 >= N1;
                            if (!(gm & zmask & side_mask<N1>(tc, 0x33u, 0xccu))) continue;
                            // the lanes whose (gx, gy, gz) is in the mask
                            const bool keep = from[cy0 && cy1][cz0 && cz1] & (1u << ((!cy0 ? 2 : 0) + (!cz0 ? 4 : 0)));
#pragma unroll
                            for (int s = 0; s < PW; s++) {
                                double c = 0.0;
#pragma unroll
                                for (int ti = 0; ti < KS; ti++) c = mma4(zo[ti], t2[s][tc][ti], c);
                                acc[s][tz][tc] += keep ? c : 0.0;
                            }
                        }
                    load_z(nq, tz);
                }
            }
            put();
            q = nq;
        }
        wave_store<N1, MWG_PREC_FP64>(w.out, w.direct, it, lane, [&](int v) { return acc[v / (TC * TC)][(v % (TC * TC)) / TC][v % TC]; });
    }
}

// Partial slots of a node added to its first unit's value in unit order, eight
// slots' loads in flight: src[j stride] is slot j's value.
__device__ __forceinline__ double slot_sum(double acc, const double *src, int slots, size_t stride) {
    int j = 0;
    for (; j + 8 <= slots; j += 8) {
        double t[8];
#pragma unroll
        for (int q = 0; q < 8; q++) t[q] = src[(size_t)(j + q) * stride];
#pragma unroll
        for (int q = 0; q < 8; q++) acc += t[q];
    }
    for (; j < slots; j++) acc += src[(size_t)j * stride];
    return acc;
}

// Orders 5 and 9: a workgroup takes the same value of every item.
template <int N1>
__global__ __launch_bounds__(64 * WaveShape<N1>::ITEMS) void k_reduce_waves(const mwg_segment *segs, const int *node_seg, const long long *g_off,
                                                                            const long long *uscan, const double *partial) {
    constexpr int N = 8 * WaveShape<N1>::N3;
    const int g = blockIdx.x;
    const long long v = uscan[g];
    const int Ug = unit_first(v);
    const int nu = unit_first(uscan[g + 1]) - Ug;
    if (nu == 1) return; // a single unit wrote the node already
    double *dst = ro(segs)[ro(node_seg)[g]].g_coef + g_off[g] + WaveMap<N1, MWG_PREC_FP64>::out(threadIdx.x >> 6, blockIdx.y, threadIdx.x & 63);
    *dst = nu == 0 ? 0.0 : slot_sum(*dst, partial + (size_t)(Ug - flagged_before(v)) * N + blockIdx.y * blockDim.x + threadIdx.x, nu - 1, N);
}

// Order 7: a workgroup takes the rows that hold every j0 and j1 of their outputs,
// those of one (gx, gy, r) at FP64, of one (gx, r) at FP32, adds them up and puts
// them in place through LDS (written one by one from the slots' order a level's
// nodes are reached in pieces of 16 bytes).  256 or 512 threads a workgroup: an
// application to 32 Gaussians at FP64 takes 1.59 ms of it (1.75 with 1024 and a slot
// for the first unit, 1.56 for k_reduce_units after the kernel by rows).
template <int PREC>
__global__ __launch_bounds__((64 * WaveMap<8, PREC>::SET)) void k_reduce_waves8(const mwg_segment *segs, const int *node_seg, const long long *g_off,
                                                                                const long long *uscan, const double *partial) {
    using M = WaveMap<8, PREC>;
    constexpr bool F64 = PREC == MWG_PREC_FP64;
    __shared__ double c[64 * M::SET];
    const int g = blockIdx.x, y = blockIdx.y, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long long v = uscan[g];
    const int Ug = unit_first(v);
    const int nu = unit_first(uscan[g + 1]) - Ug;
    if (nu == 1) return; // a single unit wrote the node already
    const int r = y & 3, gx = F64 ? y >> 3 : y >> 2;
    const int it = 2 * gx + (F64 ? w >> 1 : w >> 2), val = F64 ? 4 * (2 * (w & 1) + (y >> 2 & 1)) + r : 4 * (w & 3) + r;
    const int e = M::row(it, val) * 64 + lane, o = M::out(it, val, lane);
    double *dst = ro(segs)[ro(node_seg)[g]].g_coef + g_off[g];
    // the row of the workgroup that lies where output o does
    const int at = F64 ? o >> 6 & 3 : (o >> 10 & 3) | (o >> 8 & 1) << 2;
    c[64 * at + (o & 63)] = nu == 0 ? 0.0 : slot_sum(dst[e], partial + (size_t)(Ug - flagged_before(v)) * 4096 + e, nu - 1, 4096);
    __syncthreads();
    dst[e] = c[threadIdx.x];
}

// The same at order 3 with the component norms (block_norms' order) in one
// launch, a workgroup per node and a thread per value: its levels are short, and a
// launch costs more than the 512 values (two launches: 56 us an application,
// one: 47).  At the higher orders a workgroup per node leaves the slots' loads
// too few workgroups (order 7: 289 -> 376 us an application, order 9: 206 -> 381).
__global__ __launch_bounds__(512) void k_reduce_norms(const mwg_segment *segs, const int *node_seg, const long long *g_off, const long long *uscan,
                                                      const double *partial, double *g_norms) {
    using W = WaveShape<4>;
    static_assert(8 * W::N3 == 512, "a thread per value");
    __shared__ double c[512];
    __shared__ double red[8 * (kThreads / 64)];
    const int g = blockIdx.x, e = threadIdx.x;
    const long long v = uscan[g];
    const int Ug = unit_first(v);
    const int nu = unit_first(uscan[g + 1]) - Ug;
    double *dst = ro(segs)[ro(node_seg)[g]].g_coef + g_off[g];
    if (nu == 1) {
        c[e] = dst[e];
    } else {
        const int o = WaveMap<4, MWG_PREC_FP64>::out((e >> 6) % W::ITEMS, (e >> 6) / W::ITEMS, e & 63);
        c[o] = nu == 0 ? 0.0 : slot_sum(dst[e], partial + (size_t)(Ug - flagged_before(v)) * 512 + e, nu - 1, 512);
    }
    __syncthreads();
    if (nu != 1) dst[e] = c[e];
    block_norms<4>(c, g_norms + (size_t)g * 9, red);
}

} // namespace

} // namespace mwgdev
