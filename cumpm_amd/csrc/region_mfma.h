// Matrix-core spread and contraction over regions of the reciprocal grid (device code shared by
// the dipole and quadrupole operators), for v_mfma 16x16x4 in FP32 and FP64.
#ifndef MPM_REGION_MFMA_H
#define MPM_REGION_MFMA_H

#include "mpm_internal.h"

namespace mpm {

template <typename R>
struct C2;
template <>
struct C2<double> {
    using T = double2;
};
template <>
struct C2<float> {
    using T = float2;
};

__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// v of the neighbouring lane (lane ^ 1), by a lane permutation within quads.
__device__ __forceinline__ double swap_lane1(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}

// ---- spread on the matrix cores ----
//
// For a region of RX x (planes) x 16 rows (slab: RX x 16 y over all slab planes;
// full grid: 4 x 8 or 4 y-planes x 16 z, see RegionGeom) and 16 real columns
// q = 2 NC b + 2 c + (0: real, 1: imaginary) of the right-hand sides (NC = 3 dipole
// components, 8 with quadrupoles),
//   grid^T[q][voxel] = sum_k V[k][q] W[k][voxel],
//   W[k][(x, plane, row)] = wx_k(x) wp_k(plane) wr_k(row)
// over the candidate particles k of the region (every particle whose stencil
// footprint meets it, in ascending id order), one 16x16x4 MFMA (FP32 or FP64)
// per four candidates and (x, plane) pair: A = V^T (16 columns x 4 candidates),
// B = W^T (4 candidates x 16 consecutive rows).  The region-local separable weights
// (stencil folding on small grids included) are staged per candidate chunk in
// LDS.  Every voxel is written exactly once, without atomics; the sum order is
// fixed (deterministic).
constexpr int kMfmaRY = 16;    // y voxels per region (the MFMA N dimension)
constexpr int kMfmaKC = 64;    // candidates staged per chunk
// Planes (y) per region on the full grid and candidate blocks of 16 per chunk of
// its contraction: 4 x 8 x 16-voxel regions, about 28 candidates each in a
// packing of volume fraction 0.3 with 9-point stencils on a 256^3 grid.
constexpr int kFullRegionPlanes = 8;
constexpr int kFullContractNB = 2;

typedef float mpm_f32x4 __attribute__((ext_vector_type(4)));
typedef double mpm_f64x4 __attribute__((ext_vector_type(4)));

// 16x16x4 MFMA: lane l holds A[l % 16][l / 16] and B[l / 16][l % 16]; its
// accumulator entry r is D[drow(l / 16, r)][l % 16], with drow = 4 g + r for
// FP32 and g + 4 r for FP64 (measured on gfx950).  rowcol(i) is the real
// column a spread wave feeds into A row i so that accumulator entries (0, 1)
// and (2, 3) of every lane are the real and imaginary parts of one complex
// column: complex column 2 g + h of the wave sits in entries (2 h, 2 h + 1).
template <typename R>
struct Mfma;
template <>
struct Mfma<float> {
    using V4 = mpm_f32x4;
    static __device__ __forceinline__ V4 mac(float a, float b, V4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int drow(int g, int r) { return 4 * g + r; }
    static __device__ __forceinline__ int rowcol(int i) { return i; }
};
template <>
struct Mfma<double> {
    using V4 = mpm_f64x4;
    static __device__ __forceinline__ V4 mac(double a, double b, V4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int drow(int g, int r) { return g + 4 * r; }
    // row i = g + 4 r -> complex column 2 g + r / 2, part r % 2
    static __device__ __forceinline__ int rowcol(int i) { return 2 * (2 * (i & 3) + (i >> 3)) + ((i >> 2) & 1); }
};

// Block shape of spread_mfma_kernel: 4 waves = (CPB / 16 column groups) x
// (plane groups of ZH planes).  CPB = 32 splits the planes over two waves, CPB = 16 over
// four: fewer accumulators per wave, more blocks, and no idle column group when a batch
// has no more than 16 real columns.
template <int ZSB, int CPB>
struct SpreadShape {
    static constexpr int NPG = 4 / (CPB / 16);
    static constexpr int ZH = (ZSB + NPG - 1) / NPG;
};

// Region-local separable weights of a candidate, one LDS row per candidate:
// x weights at [0, RX), slab-plane weights at [4, 4 + ZSB), y weights at
// [4 + ZSB4, 4 + ZSB4 + 16) (ZSB4 = ZSB rounded up to 4), so that 4-wide
// groups start on 16-byte boundaries.  A voxel's weight sums the stencil points
// that land on it (stencils fold onto themselves on grids narrower than the
// stencil).
template <int RX, int ZSB>
struct RegionW {
    static constexpr int ZSB4 = (ZSB + 3) & ~3;
    static constexpr int X = 0, Z = 4, Y = 4 + ZSB4;
    static constexpr int NW = Y + kMfmaRY;
};

// v where c holds, else +0, by a bit mask rather than a select: the compiler turns a
// select of a loaded value into a branch around the load, which then waits for
// the load at the branch's end.
__device__ __forceinline__ float keep_if(float v, bool c) {
    return __uint_as_float(__float_as_uint(v) & (c ? 0xffffffffu : 0u));
}
__device__ __forceinline__ double keep_if(double v, bool c) {
    return __longlong_as_double(__double_as_longlong(v) & (c ? -1LL : 0LL));
}

// Copies the precomputed region-local weight rows of a chunk of cnt <= KC
// candidates into LDS (zero rows past cnt) and ends with a barrier.  Blocks of 256
// threads; every load is issued before the first store (one memory latency per chunk,
// not one per element).
template <typename R, int RX, int ZSB, int KC = kMfmaKC>
__device__ inline void stage_weights(R* s_w, int cnt, const R* __restrict__ regw) {
    using L = RegionW<RX, ZSB>;
    constexpr int T = (KC * L::NW + 255) / 256;
    const int n = cnt * L::NW;
    R v[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int e = (int)threadIdx.x + 256 * t;
        v[t] = e < n ? regw[e] : R(0);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int e = (int)threadIdx.x + 256 * t;
        if (e < KC * L::NW) s_w[e] = v[t];
    }
    __syncthreads();
}

// Plane loop of the matrix-core contractions, software-pipelined over two operand
// buffers: the loads of the next plane are in flight while the current plane's
// products run.  load(p, buf) issues plane p's loads into buf, mma(buf, p)
// consumes them; planes first, first + step, ... below end.  The loop body has no
// branch between a load and its use (a branch would let the compiler sink the
// loads next to their use): the last pair loads its second plane again, and an
// odd plane count ends with one more product.  Scheduling barriers keep each group
// of loads whole and ahead of the other buffer's products, so that the products
// wait only for their own (older) loads.
template <typename Buf, typename LoadF, typename MmaF>
__device__ __forceinline__ void plane_pipeline(int first, int step, int end, Buf& ga, Buf& gb, LoadF&& load,
                                               MmaF&& mma) {
    if (first >= end) return;
    const int n = (end - first + step - 1) / step;
    const int last = first + (n - 1) * step;
    load(first, ga);
    int i = 0, p = first;
    for (; i + 1 < n; i += 2, p += 2 * step) {
        __builtin_amdgcn_sched_barrier(0);
        load(p + step, gb);
        __builtin_amdgcn_sched_barrier(0);
        mma(ga, p);
        __builtin_amdgcn_sched_barrier(0);
        load(min(p + 2 * step, last), ga);
        __builtin_amdgcn_sched_barrier(0);
        mma(gb, p + step);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (i < n) mma(ga, p);
}

// Vector form of the contractions' grid operands: the four voxels a lane feeds into
// the four products of a plane and x are rows 4 r + u (r = lane / 16, u = 0..3) of
// its real column (even lane) or imaginary column (odd lane); the two lanes of a
// complex column load rows (4 r, 4 r + 1) and (4 r + 2, 4 r + 3) as whole complex
// pairs v = (re, im, re, im) and swap halves with a neighbour-lane move, so that one
// 16-byte load per lane reads the 16 rows of eight complex components (one whole
// 128-byte line each for FP32).  g receives rows 4 r + u of this lane's part.
template <typename R, typename V4>
__device__ __forceinline__ void pair_rows(const V4& v, int part, R (&g)[4]) {
    const R s0 = part ? v[0] : v[1], s1 = part ? v[2] : v[3];
    const R t0 = __shfl_xor(s0, 1, 64), t1 = __shfl_xor(s1, 1, 64);
    g[0] = part ? t0 : v[0];
    g[1] = part ? t1 : v[2];
    g[2] = part ? v[1] : t0;
    g[3] = part ? v[3] : t1;
}

// Where the regions sit in a grid buffer.  A region is RX consecutive x, up to
// pblk consecutive planes and 16 consecutive rows, rows contiguous in memory:
// in the slab layout the planes are the occupied z-planes (all in one region)
// and the rows y; on the full grid the planes are y (blocks of pblk) and the
// rows z.  Regions are numbered (x block, plane block, row block), row block
// fastest.  Strides are in complex elements.
struct RegionGeom {
    int nx, nrow, nplane;  // extents along x, rows, planes
    int nrr, npb, pblk;    // row blocks, plane blocks, planes per region
    unsigned xs, ps, cs;   // strides of x, plane, component (b, c)
};

struct RegionAt {
    int x0, plane0, row0, np;  // origin and number of planes present
};

template <int RX>
__device__ inline RegionAt region_at(const RegionGeom& rg, int reg) {
    const int per_x = rg.npb * rg.nrr;
    const int rx = reg / per_x, rem = reg - rx * per_x;
    const int pb = rem / rg.nrr, rr = rem - pb * rg.nrr;
    RegionAt a;
    a.x0 = rx * RX;
    a.plane0 = pb * rg.pblk;
    a.row0 = rr * kMfmaRY;
    a.np = min(rg.pblk, rg.nplane - a.plane0);
    return a;
}

// FP32: held to 128 registers (four waves per SIMD; at the compiler's 140 three, and the
// N = 4000 monolayer's 1272 blocks took 1.7 rounds instead of 1.2: 39.4 against 37.0 us).
//
// CPB = 16 is the form for few blocks (region_spread): there a region's candidates come in
// several chunks and nothing else hides their loads, so the next chunk's values and
// weights are fetched while the current chunk's products run.
// Weights of the spread: with quadrupoles FP64 rows, so that each product is rounded once
// (the reference's stencils hold the rounded product), else the grid's type.
template <typename R, int NC>
using SpreadW = std::conditional_t<NC == 8, double, R>;

template <typename R, int RX, int ZSB, int CPB, int NC>
__global__ __launch_bounds__(256, sizeof(R) == 4 ? (NC == 3 ? 4 : 3) : 2) void spread_mfma_kernel(SlotTable tab, int B, RegionGeom rg,
                                                          const SpreadW<R, NC>* __restrict__ regw,
                                                          const int* __restrict__ reg_start,
                                                          const int* __restrict__ reg_items,
                                                          const int* __restrict__ reg_quads, size_t n3,
                                                          typename C2<R>::T* __restrict__ out) {
    using CT = typename C2<R>::T;
    using M = Mfma<R>;
    using WR = SpreadW<R, NC>;
    using Sh = SpreadShape<ZSB, CPB>;
    constexpr int KC = kMfmaKC, ZH = Sh::ZH;
    constexpr bool PREFETCH = CPB == 16;
    using L = RegionW<RX, ZSB>;
    __shared__ R s_v[KC][CPB + 1];
    __shared__ __align__(16) WR s_w[KC][L::NW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int cg = wave % (CPB / 16), pg = wave / (CPB / 16);
    const int reg = blockIdx.x;
    const RegionAt ra = region_at<RX>(rg, reg);
    const int x0 = ra.x0, y0 = ra.row0;
    const int col_base = blockIdx.y * CPB;
    const int wcol0 = col_base + cg * 16;
    const int ncols = 2 * NC * B;
    const int Zs = ra.np;    // planes of this region
    const int p0 = pg * ZH;  // this wave's planes [p0, p0 + ZH) of the region
    const int k0 = reg_start[reg], k1 = reg_start[reg + 1];

    typename M::V4 acc[RX][ZH];
#pragma unroll
    for (int xi = 0; xi < RX; ++xi)
#pragma unroll
        for (int p = 0; p < ZH; ++p) acc[xi][p] = typename M::V4{R(0), R(0), R(0), R(0)};

    // staged columns of this thread: s_v[q][scol] for q = tid / CPB + (256 / CPB) t
    constexpr int QS = 256 / CPB, TV = KC / QS;
    constexpr int TW = (KC * L::NW + 255) / 256;  // weight-row entries of this thread
    const int scol = tid % CPB, sqc = col_base + scol;
    // columns past the batch, and the gradient columns when no particle has a quadrupole
    // (reg_quads null: the vectors end at n3), read column 0 and stage zeros
    const bool scok = sqc < ncols && (NC == 3 || reg_quads || (sqc >> 1) % NC < 3);
    const int sq = scok ? sqc : 0;
    // vectors of unknowns: 3 components per particle, with quadrupoles (NC = 8) followed
    // after n3 = 3 N values by 5 per quadrupole; a candidate's entry e of this thread's column
    // is item cs e + the column's offset, e its particle or its quadrupole (-1: none)
    const int sc_ = (sq >> 1) % NC;
    const bool squad = NC == 8 && sc_ >= 3;
    const double* xcol = reinterpret_cast<const double*>(tab.x[sq / (2 * NC)]) + (sq & 1) +
                         (squad ? 2 * (n3 + (size_t)(sc_ - 3)) : 2 * (size_t)sc_);
    const size_t cs = squad ? 10 : 6;
    const int* cand = squad ? reg_quads : reg_items;
    auto value = [&](int e, bool take) {
        if constexpr (NC == 8) {
            take = take && e >= 0;
            e = max(e, 0);
        }
        return keep_if((R)xcol[cs * (size_t)e], take);
    };
    // candidate ids of the chunk of cnt candidates at c0 (clamped to the last one past its
    // end), its values (component (b, c), real or imaginary part) and its weight rows (zero
    // past its end): every load of a group is issued before the first use
    auto load_ids = [&](int c0, int cnt, int (&id)[TV]) {
#pragma unroll
        for (int t = 0; t < TV; ++t) id[t] = cand[c0 + min(tid / CPB + QS * t, cnt - 1)];
    };
    auto load_vals = [&](int cnt, const int (&id)[TV], R (&vv)[TV]) {
#pragma unroll
        for (int t = 0; t < TV; ++t)
            vv[t] = value(id[t], scok && tid / CPB + QS * t < cnt);
    };
    auto load_wts = [&](int c0, WR (&ww)[TW]) {
        const int n = min(KC, k1 - c0) * L::NW;
        const WR* w = regw + (size_t)c0 * L::NW;
#pragma unroll
        for (int t = 0; t < TW; ++t) ww[t] = keep_if(w[min(tid + 256 * t, n - 1)], tid + 256 * t < n);
    };
    int id[TV];
    R vv[TV];
    WR ww[TW];
    if (PREFETCH && k0 < k1) {
        load_ids(k0, min(KC, k1 - k0), id);
        load_vals(min(KC, k1 - k0), id, vv);
        load_wts(k0, ww);
        if (k0 + KC < k1) load_ids(k0 + KC, min(KC, k1 - k0 - KC), id);
    }
    for (int c0 = k0; c0 < k1; c0 += KC) {
        const int cnt = min(KC, k1 - c0);
        __syncthreads();
        if constexpr (PREFETCH) {
#pragma unroll
            for (int t = 0; t < TW; ++t)
                if (tid + 256 * t < KC * L::NW) (&s_w[0][0])[tid + 256 * t] = ww[t];
#pragma unroll
            for (int t = 0; t < TV; ++t) s_v[tid / CPB + QS * t][scol] = vv[t];
        } else {
            int idc[TV];
#pragma unroll
            for (int t = 0; t < TV; ++t) idc[t] = cand[c0 + min(tid / CPB + QS * t, cnt - 1)];
            R vc[TV];
#pragma unroll
            for (int t = 0; t < TV; ++t)
                vc[t] = value(idc[t], scok && tid / CPB + QS * t < cnt);
            stage_weights<WR, RX, ZSB>(&s_w[0][0], cnt, regw + (size_t)c0 * L::NW);
#pragma unroll
            for (int t = 0; t < TV; ++t) s_v[tid / CPB + QS * t][scol] = vc[t];
        }
        __syncthreads();
        if (PREFETCH && c0 + KC < k1) {
            load_vals(min(KC, k1 - c0 - KC), id, vv);
            load_wts(c0 + KC, ww);
            if (c0 + 2 * KC < k1) load_ids(c0 + 2 * KC, min(KC, k1 - c0 - 2 * KC), id);
        }
        if (wcol0 < ncols && p0 < Zs) {
            const int i = lane & 15;
            for (int ks = 0; ks < cnt; ks += 4) {
                const int kq = ks + (lane >> 4);  // rows >= cnt hold zeros
                const R a = s_v[kq][cg * 16 + M::rowcol(i)];
                const WR wy = s_w[kq][L::Y + i];
                WR wx[RX], wz[ZH];
#pragma unroll
                for (int xi = 0; xi < RX; ++xi) wx[xi] = s_w[kq][L::X + xi] * wy;
#pragma unroll
                for (int p = 0; p < ZH; ++p) wz[p] = (p0 + p < ZSB) ? s_w[kq][L::Z + p0 + p] : WR(0);
                // planes past Zs carry zero weights: no branch around the accumulators
#pragma unroll
                for (int p = 0; p < ZH; ++p) {
#pragma unroll
                    for (int xi = 0; xi < RX; ++xi) acc[xi][p] = M::mac(a, (R)(wx[xi] * wz[p]), acc[xi][p]);
                }
            }
        }
    }
    // lane holds complex columns 2 (lane >> 4) + h of the wave (entries 2 h, 2 h + 1)
    // at row y0 + (lane & 15)
    const int y = y0 + (lane & 15);
    if (y >= rg.nrow || wcol0 >= ncols) return;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int qc = wcol0 + 4 * (lane >> 4) + 2 * h;
        if (qc >= ncols) continue;
        const int b = qc / (2 * NC), c = (qc >> 1) % NC;
        CT* o = out + ((size_t)b * NC + c) * rg.cs + (size_t)ra.plane0 * rg.ps + y;
#pragma unroll
        for (int xi = 0; xi < RX; ++xi) {
            const int x = x0 + xi;
            if (x >= rg.nx) continue;
#pragma unroll
            for (int p = 0; p < ZH; ++p)
                if (p0 + p < Zs) {
                    CT v;
                    v.x = acc[xi][p][2 * h];
                    v.y = acc[xi][p][2 * h + 1];
                    o[(size_t)(p0 + p) * rg.ps + (size_t)x * rg.xs] = v;
                }
        }
    }
}

// ---- contraction on the matrix cores ----
//
// The transpose of spread_mfma_kernel over the same regions: for the candidate
// particles k of a region and 16 real columns q,
//   D[k][q] = sum_{voxels v of the region} W[k][v] G[v][q],
// one 16x16x4 MFMA per four voxels and 16 candidates (A = W, B = G), every
// loaded operand feeding all candidate blocks.  Each wave reads its B operands
// straight from the grid: lane (j, u) loads column j at row 4 u + (lane >> 4),
// so the four loads of a 16-voxel row consume whole cache lines, or with VEC
// (pair_rows) one 16-byte complex pair per lane and x; waves run without
// barriers after the one weight-staging step.  D goes to the particle's
// slot of the region (the CSR position of the pair); the per-particle sum over
// its regions happens in the finish step, in a fixed order.  GR is the grid's real type, R
// that of the weights, products and sums: FP64 over an FP32 grid where the per-particle
// gather, which sums in FP64 past each lane's few terms, is the alternative.
template <typename R, int RX, int ZSB, int NB, bool VEC, int NC, typename GR>
__global__ __launch_bounds__(256, sizeof(R) == 4 ? 3 : 2) void contract_mfma_kernel(int B, RegionGeom rg,
                                                                                    const R* __restrict__ regw,
                                                            const int* __restrict__ reg_start,
                                                            const typename C2<GR>::T* __restrict__ grid,
                                                            R* __restrict__ partial, int ncg) {
    using M = Mfma<R>;
    using V4 = typename M::V4;
    constexpr int KC = 16 * NB;  // candidates per chunk, in NB blocks of 16
    using L = RegionW<RX, ZSB>;
    __shared__ __align__(16) R s_w[KC][L::NW];
    __shared__ V4 s_red[4][NB][64];  // per-wave partial accumulators
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // 4 waves = ncg column groups x (4 / ncg) plane groups
    const int npg = 4 / ncg, cg = wave % ncg, pg = wave / ncg;
    const int reg = blockIdx.x;
    const RegionAt ra = region_at<RX>(rg, reg);
    const int x0 = ra.x0, y0 = ra.row0;
    const int wcol0 = (blockIdx.y * ncg + cg) * 16;
    const int ncols = 2 * NC * B;
    const bool active = wcol0 < ncols;
    const int Zs = ra.np;  // planes of this region
    const unsigned plane = rg.ps;
    const int k0 = reg_start[reg], k1 = reg_start[reg + 1];

    // this lane's B-operand column and its rows of the region, as 32-bit offsets
    // (in R) from the uniform grid base: the launch keeps 6 B x (complex per
    // component) below 2^32
    const GR* gf = reinterpret_cast<const GR*>(grid);
    const int qc = wcol0 + (lane & 15);
    const bool cvalid = qc < ncols;
    // column offset at the region origin (cbase, an in-grid voxel of every plane of the
    // region) and at this lane's row; bit 4 xi + u of vmask: (x0 + xi, y0 + 4 u + lane / 16)
    // inside the grid.  VEC (pair_rows): the lane's complex pair at rows y0 + 4 r + 2 part
    // and the next, bit xi of vmask: (x0 + xi, y0 + 4 r + 2 part) inside; even rows keep
    // both rows of a pair inside together.
    const int r = lane >> 4, part = lane & 1;
    unsigned cbase = 0, coff = 0, vmask = 0;
    if (cvalid) {
        const int b = qc / (2 * NC), c = (qc >> 1) % NC;
        cbase = 2u * (unsigned)(b * NC + c) * rg.cs + (VEC ? 0u : (unsigned)(qc & 1)) +
                2u * ((unsigned)ra.plane0 * rg.ps + (unsigned)x0 * rg.xs + (unsigned)y0);
        if (VEC) {
            coff = cbase + 2u * (unsigned)(4 * r + 2 * part);
#pragma unroll
            for (int xi = 0; xi < RX; ++xi)
                if (x0 + xi < rg.nx && y0 + 4 * r + 2 * part < rg.nrow) vmask |= 1u << xi;
        } else {
            coff = cbase + 2u * (unsigned)(lane >> 4);
#pragma unroll
            for (int xi = 0; xi < RX; ++xi)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (x0 + xi < rg.nx && y0 + 4 * u + (lane >> 4) < rg.nrow) vmask |= 1u << (4 * xi + u);
        }
    }
    const unsigned xstep = 2u * rg.xs;

    for (int c0 = k0; c0 < k1; c0 += KC) {
        const int cnt = min(KC, k1 - c0);
        __syncthreads();
        stage_weights<R, RX, ZSB, KC>(&s_w[0][0], cnt, regw + (size_t)c0 * L::NW);
        V4 acc[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[nb] = V4{R(0), R(0), R(0), R(0)};
        if (active) {
            // per-lane weights: candidate k = 16 nb + (lane & 15) at x = x0 + xi and rows
            // y0 + 4 u + r (VEC: y0 + 4 r + u)
            R wyl[NB][4], wxl[NB][RX];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const int k = nb * 16 + (lane & 15);
#pragma unroll
                for (int u = 0; u < 4; ++u) wyl[nb][u] = s_w[k][L::Y + (VEC ? 4 * r + u : 4 * u + r)];
#pragma unroll
                for (int xi = 0; xi < RX; ++xi) wxl[nb][xi] = s_w[k][L::X + xi];
            }
            if constexpr (VEC) {
                struct PlaneBuf {
                    typename Mfma<GR>::V4 g[RX];
                };
                auto load_plane = [&](int p, PlaneBuf& dst) {
                    const unsigned poff = coff + 2u * (unsigned)p * plane, pin = cbase + 2u * (unsigned)p * plane;
#pragma unroll
                    for (int xi = 0; xi < RX; ++xi) {
                        const bool in = (vmask >> xi) & 1u;
                        dst.g[xi] = *reinterpret_cast<const typename Mfma<GR>::V4*>(gf + (in ? poff + xi * xstep : pin));
                    }
                };
                auto mma = [&](PlaneBuf& pb, int p) {
                    R wz[NB];
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) wz[nb] = s_w[nb * 16 + (lane & 15)][L::Z + p];
#pragma unroll
                    for (int xi = 0; xi < RX; ++xi) {
                        GR gv[4];
                        pair_rows<GR>(pb.g[xi], part, gv);
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb) {
                            const R wxz = wxl[nb][xi] * wz[nb];
#pragma unroll
                            for (int u = 0; u < 4; ++u) acc[nb] = M::mac(wyl[nb][u] * wxz, (R)gv[u], acc[nb]);
                        }
                    }
                };
                PlaneBuf ga, gb;
                plane_pipeline(pg, npg, Zs, ga, gb, load_plane, mma);
            } else {
            // the next plane's operands are loaded while this plane's products run
            auto load_plane = [&](int p, GR (&dst)[RX][4]) {
                const unsigned poff = coff + 2u * (unsigned)p * plane, pin = cbase + 2u * (unsigned)p * plane;
#pragma unroll
                for (int xi = 0; xi < RX; ++xi)
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        // lanes outside the grid read the region's origin instead, which
                        // meets a zero weight (the weight rows are zero past the grid's
                        // edges): no branch around the load and no use of it before the
                        // products
                        const bool in = (vmask >> (4 * xi + u)) & 1u;
                        dst[xi][u] = gf[in ? poff + xi * xstep + 8u * u : pin];
                    }
            };
            auto mma = [&](GR (&gv)[RX][4], int p) {
                R wz[NB];
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) wz[nb] = s_w[nb * 16 + (lane & 15)][L::Z + p];
                // every candidate block, filled or not (rows past cnt hold zero weights):
                // a branch here would make the compiler copy the accumulators around it
#pragma unroll
                for (int xi = 0; xi < RX; ++xi)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) {
                        const R wxz = wxl[nb][xi] * wz[nb];
#pragma unroll
                        for (int u = 0; u < 4; ++u) acc[nb] = M::mac(wyl[nb][u] * wxz, (R)gv[xi][u], acc[nb]);
                    }
            };
            GR ga[RX][4], gb[RX][4];
            plane_pipeline(pg, npg, Zs, ga, gb, load_plane, mma);
            }
        }
        // plane groups of one column group are summed in plane-group order
        if (npg > 1) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) s_red[wave][nb][lane] = acc[nb];
            __syncthreads();
            if (pg == 0) {
                for (int q = 1; q < npg; ++q)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) acc[nb] += s_red[q * ncg + cg][nb][lane];
            }
        }
        // lane holds D[16 nb + drow(lane >> 4, r)][lane & 15]
        if (pg == 0 && cvalid) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int k = nb * 16 + M::drow(lane >> 4, q);
                    if (k < cnt) partial[(size_t)(c0 + k) * ncols + qc] = acc[nb][q];
                }
        }
    }
}

// Narrow-batch variant of the contraction: a block is one column group of 16
// and four waves, one per block of 16 candidates, so a wave holds few registers
// and, when only one or two column groups exist, the region's candidates still
// spread over four waves; the next plane's operands are loaded while the
// current plane's products run.
template <typename R, int RX, int ZSB, bool VEC, int NC, typename GR>
__global__ __launch_bounds__(256) void contract_nb_mfma_kernel(int B, RegionGeom rg, const R* __restrict__ regw,
                                                               const int* __restrict__ reg_start,
                                                               const typename C2<GR>::T* __restrict__ grid,
                                                               R* __restrict__ partial) {
    using M = Mfma<R>;
    using V4 = typename M::V4;
    constexpr int KC = kMfmaKC;
    using L = RegionW<RX, ZSB>;
    __shared__ __align__(16) R s_w[KC][L::NW];
    const int tid = threadIdx.x, lane = tid & 63, nb = tid >> 6;  // candidate block of this wave
    const int reg = blockIdx.x;
    const RegionAt ra = region_at<RX>(rg, reg);
    const int x0 = ra.x0, y0 = ra.row0;
    const int wcol0 = blockIdx.y * 16;
    const int ncols = 2 * NC * B;
    const int Zs = ra.np;  // planes of this region
    const unsigned plane = rg.ps;
    const int k0 = reg_start[reg], k1 = reg_start[reg + 1];
    const GR* gf = reinterpret_cast<const GR*>(grid);
    const int qc = wcol0 + (lane & 15);
    const bool cvalid = qc < ncols;
    // column offset at the region origin (cbase, an in-grid voxel of every plane of the
    // region) and at this lane's row; bit 4 xi + u of vmask: (x0 + xi, y0 + 4 u + lane / 16)
    // inside the grid.  VEC (pair_rows): the lane's complex pair at rows y0 + 4 r + 2 part
    // and the next, bit xi of vmask: (x0 + xi, y0 + 4 r + 2 part) inside.
    const int r = lane >> 4, part = lane & 1;
    unsigned cbase = 0, coff = 0, vmask = 0;
    if (cvalid) {
        const int b = qc / (2 * NC), c = (qc >> 1) % NC;
        cbase = 2u * (unsigned)(b * NC + c) * rg.cs + (VEC ? 0u : (unsigned)(qc & 1)) +
                2u * ((unsigned)ra.plane0 * rg.ps + (unsigned)x0 * rg.xs + (unsigned)y0);
        if (VEC) {
            coff = cbase + 2u * (unsigned)(4 * r + 2 * part);
#pragma unroll
            for (int xi = 0; xi < RX; ++xi)
                if (x0 + xi < rg.nx && y0 + 4 * r + 2 * part < rg.nrow) vmask |= 1u << xi;
        } else {
            coff = cbase + 2u * (unsigned)(lane >> 4);
#pragma unroll
            for (int xi = 0; xi < RX; ++xi)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (x0 + xi < rg.nx && y0 + 4 * u + (lane >> 4) < rg.nrow) vmask |= 1u << (4 * xi + u);
        }
    }
    const unsigned xstep = 2u * rg.xs;
    for (int c0 = k0; c0 < k1; c0 += KC) {
        const int cnt = min(KC, k1 - c0);
        __syncthreads();
        stage_weights<R, RX, ZSB>(&s_w[0][0], cnt, regw + (size_t)c0 * L::NW);
        if (nb * 16 >= cnt) continue;  // no candidates for this wave (no barrier follows in this chunk)
        const int k = nb * 16 + (lane & 15);
        R wyl[4], wxl[RX];
#pragma unroll
        for (int u = 0; u < 4; ++u) wyl[u] = s_w[k][L::Y + (VEC ? 4 * r + u : 4 * u + r)];
#pragma unroll
        for (int xi = 0; xi < RX; ++xi) wxl[xi] = s_w[k][L::X + xi];
        V4 acc = V4{R(0), R(0), R(0), R(0)};
        if constexpr (VEC) {
            struct PlaneBuf {
                typename Mfma<GR>::V4 g[RX];
            };
            auto load_plane = [&](int p, PlaneBuf& dst) {
                const unsigned poff = coff + 2u * (unsigned)p * plane, pin = cbase + 2u * (unsigned)p * plane;
#pragma unroll
                for (int xi = 0; xi < RX; ++xi) {
                    const bool in = (vmask >> xi) & 1u;
                    dst.g[xi] = *reinterpret_cast<const typename Mfma<GR>::V4*>(gf + (in ? poff + xi * xstep : pin));
                }
            };
            auto mma = [&](PlaneBuf& pb, int p) {
                const R wz = s_w[k][L::Z + p];
#pragma unroll
                for (int xi = 0; xi < RX; ++xi) {
                    GR gv[4];
                    pair_rows<GR>(pb.g[xi], part, gv);
                    const R wxz = wxl[xi] * wz;
#pragma unroll
                    for (int u = 0; u < 4; ++u) acc = M::mac(wyl[u] * wxz, (R)gv[u], acc);
                }
            };
            PlaneBuf ga, gb;
            plane_pipeline(0, 1, Zs, ga, gb, load_plane, mma);
        } else {
            auto load_plane = [&](int p, GR (&dst)[RX][4]) {
                const unsigned poff = coff + 2u * (unsigned)p * plane, pin = cbase + 2u * (unsigned)p * plane;
#pragma unroll
                for (int xi = 0; xi < RX; ++xi)
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        // lanes outside the grid read the region's origin, which meets a zero weight
                        const bool in = (vmask >> (4 * xi + u)) & 1u;
                        dst[xi][u] = gf[in ? poff + xi * xstep + 8u * u : pin];
                    }
            };
            auto mma = [&](GR (&gv)[RX][4], int p) {
                const R wz = s_w[k][L::Z + p];
#pragma unroll
                for (int xi = 0; xi < RX; ++xi) {
                    const R wxz = wxl[xi] * wz;
#pragma unroll
                    for (int u = 0; u < 4; ++u) acc = M::mac(wyl[u] * wxz, (R)gv[xi][u], acc);
                }
            };
            GR ga[RX][4], gb[RX][4];
            plane_pipeline(0, 1, Zs, ga, gb, load_plane, mma);
        }
        // lane holds D[16 nb + drow(lane >> 4, q)][lane & 15]
        if (cvalid) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int kk = nb * 16 + M::drow(lane >> 4, q);
                if (kk < cnt) partial[(size_t)(c0 + kk) * ncols + qc] = acc[q];
            }
        }
    }
}

// Full-grid contraction on the matrix cores: the products of contract_mfma_kernel
// over RX x PB x 16-voxel regions (x, y planes, z rows), one wave per (region,
// column group of 16), work item = region x column groups + group, so that the
// groups of a region run in neighbouring waves and share its weights in the caches.
// Waves are independent (no LDS, no barriers).
//
// Memory access is in whole 16-byte vectors: the four voxels a lane feeds into the
// four products of a plane and x are rows 4 r + u (r = lane / 16, u = 0..3), and the
// two lanes of a complex column pair (real part j even, imaginary part j + 1) load
// rows (4 r, 4 r + 1) and (4 r + 2, 4 r + 3) as complex pairs, then swap halves with
// a neighbour-lane move; so one load instruction per x and plane reads the 16 rows
// of eight complex components, one whole 128-byte line each.  The candidates'
// weights come the same way, a vector each for x, the planes and the lane's rows.
// Needs an even number of rows (z) and 16-byte aligned grid and weight rows.
// The next plane's operands are loaded while the current plane's products run.
template <typename R, int RX, int PB, int NB, int NC, typename GR>
__global__ __launch_bounds__(256) void contract_full_mfma_kernel(int B, RegionGeom rg, const R* __restrict__ regw,
                                                                 const int* __restrict__ reg_start, int nitems,
                                                                 int ngrp, const typename C2<GR>::T* __restrict__ grid,
                                                                 R* __restrict__ partial) {
    using M = Mfma<R>;
    using V4 = typename M::V4;  // four R: a complex pair of the grid, or four weights
    using L = RegionW<RX, PB>;
    static_assert(RX == 4 && PB == 8, "one weight vector for x, two for the planes");
    static_assert(L::Z == 4 && L::Y == 12 && L::NW == 28, "weight row: x at 0, planes at 4, rows at 12");
    constexpr int KC = 16 * NB;
    const int lane = threadIdx.x & 63;
    const int item = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (item >= nitems) return;  // the whole wave leaves: nothing below synchronises
    const int reg = item / ngrp;
    const RegionAt ra = region_at<RX>(rg, reg);
    const int x0 = ra.x0, y0 = ra.row0, np = ra.np;
    const int ncols = 2 * NC * B;
    const int r = lane >> 4, part = lane & 1;
    const int qc = (item - reg * ngrp) * 16 + (lane & 15);
    const bool cvalid = qc < ncols;
    const GR* gf = reinterpret_cast<const GR*>(grid);
    // 32-bit offsets in R from the uniform grid base (the launch keeps them below 2^32):
    // cbase = the component's voxel (x0, plane0, y0), an in-grid pair of rows of every
    // plane; this lane loads rows y0 + 4 r + 2 part and the next (vmask bit xi: inside)
    unsigned cbase = 2u * ((unsigned)ra.plane0 * rg.ps + (unsigned)x0 * rg.xs + (unsigned)y0), coff = cbase,
             vmask = 0;
    if (cvalid) {
        const int b = qc / (2 * NC), c = (qc >> 1) % NC;
        cbase += 2u * (unsigned)(b * NC + c) * rg.cs;
        coff = cbase + 2u * (unsigned)(4 * r + 2 * part);
#pragma unroll
        for (int xi = 0; xi < RX; ++xi)
            if (x0 + xi < rg.nx && y0 + 4 * r + 2 * part < rg.nrow) vmask |= 1u << xi;
    }
    const unsigned xstep = 2u * rg.xs, pstep = 2u * rg.ps;
    const int k0 = reg_start[reg], k1 = reg_start[reg + 1];
    struct PlaneBuf {
        typename Mfma<GR>::V4 g[RX];
    };
    for (int c0 = k0; c0 < k1; c0 += KC) {
        const int cnt = min(KC, k1 - c0);
        // this lane's candidates k = 16 nb + (lane & 15): x weights, plane weights (zero
        // past the region's planes and for candidates past cnt) and rows 4 r .. 4 r + 3
        R wyl[NB][4], wxl[NB][RX], wzl[NB][PB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int k = nb * 16 + (lane & 15);
            const bool kin = k < cnt;
            const V4* wr = reinterpret_cast<const V4*>(regw + (size_t)(c0 + (kin ? k : 0)) * L::NW);
            const V4 wx = wr[0], wz0 = wr[1], wz1 = wr[2], wy = wr[3 + r];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                wxl[nb][q] = wx[q];
                wzl[nb][q] = keep_if(wz0[q], kin && q < np);
                wzl[nb][4 + q] = keep_if(wz1[q], kin && 4 + q < np);
                wyl[nb][q] = wy[q];
            }
        }
        // an opaque zero, redefined per chunk: keeps the compiler from hoisting all eight
        // planes' loads out of the chunk loop (128 registers, no overlap with the products)
        unsigned salt = 0;
        asm volatile("" : "+v"(salt));
        auto load_plane = [&](int p, PlaneBuf& dst) {
            const int pc = min(p, np - 1);  // planes past the region's reload its last one
            const unsigned poff = coff + salt + (unsigned)pc * pstep, pin = cbase + salt + (unsigned)pc * pstep;
#pragma unroll
            for (int xi = 0; xi < RX; ++xi) {
                const bool in = (vmask >> xi) & 1u;
                dst.g[xi] = *reinterpret_cast<const typename Mfma<GR>::V4*>(gf + (in ? poff + xi * xstep : pin));
            }
        };
        V4 acc[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[nb] = V4{R(0), R(0), R(0), R(0)};
        auto mma = [&](PlaneBuf& pb, int p) {
#pragma unroll
            for (int xi = 0; xi < RX; ++xi) {
                GR gv[4];
                pair_rows<GR>(pb.g[xi], part, gv);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const R wxz = wxl[nb][xi] * wzl[nb][p];
#pragma unroll
                    for (int u = 0; u < 4; ++u) acc[nb] = M::mac(wyl[nb][u] * wxz, (R)gv[u], acc[nb]);
                }
            }
        };
        PlaneBuf ga, gb;
        load_plane(0, ga);
#pragma unroll
        for (int p = 0; p < PB; p += 2) {
            __builtin_amdgcn_sched_barrier(0);
            load_plane(p + 1, gb);
            __builtin_amdgcn_sched_barrier(0);
            mma(ga, p);
            __builtin_amdgcn_sched_barrier(0);
            if (p + 2 < PB) load_plane(p + 2, ga);
            __builtin_amdgcn_sched_barrier(0);
            mma(gb, p + 1);
        }
        // lane holds D[16 nb + drow(lane >> 4, r)][lane & 15]
        if (cvalid) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int k = nb * 16 + M::drow(lane >> 4, q);
                    if (k < cnt) partial[(size_t)(c0 + k) * ncols + qc] = acc[nb][q];
                }
        }
    }
}

// ---- launches ----

// The regions of the current frame: layout, planes compiled for (slab: bucket of Zs; full
// grid: planes per region), number of regions and of (region, candidate) slots, the candidates
// (CSR) and their quadrupoles (-1: none; read with NC = 8 only, null when no particle has one).
struct RegionSet {
    bool slab;
    int zsb, nreg, slots;
    const int *start, *items, *quads;
};

// NC = 8 takes slabs of at most this many planes (the quadrupole plane coupling's registers)
constexpr int kQuadSlabPlanes = 10;

template <typename R, int NC>
inline void region_spread(ProfScope& ps, hipStream_t s, const RegionSet& rs, const RegionGeom& rg, const SlotTable& t,
                          int B, const SpreadW<R, NC>* regw, size_t n3, typename C2<R>::T* grid) {
    // 32 columns per block, or 16 where a batch has no more, and on the full grid while those
    // blocks are fewer than eight per CU (7001 particles on 47 x 47 x 48, 5 right-hand sides:
    // 36.2 -> 28.8 us; the slab's regions hold about one chunk of candidates, which leaves
    // nothing to prefetch)
    const int ncols = 2 * NC * B;
    const int cpb = ncols <= 16 || (!rs.slab && (long long)rs.nreg * ((ncols + 31) / 32) < 2048) ? 16 : 32;
    const dim3 gs((unsigned)rs.nreg, (unsigned)((ncols + cpb - 1) / cpb));
#define MPM_SM1(RXV, ZSV, CPBV)                                                                                   \
    do {                                                                                                          \
        ps.kernel("spread_mfma_kernel", {type_name<R>(), #RXV, #ZSV, #CPBV, NC});                             \
        hipLaunchKernelGGL((spread_mfma_kernel<R, RXV, ZSV, CPBV, NC>), gs, dim3(256), 0, s, t, B, rg, regw,      \
                           rs.start, rs.items, rs.quads, n3, grid);                                           \
        MPM_HIP(hipGetLastError());                                                                               \
        return;                                                                                                   \
    } while (0)
#define MPM_SM(RXV, ZSV)                               \
    case ZSV:                                          \
        if constexpr (NC == 3 || ZSV <= kQuadSlabPlanes) { \
            if (cpb == 16)                             \
                MPM_SM1(RXV, ZSV, 16);                 \
            else                                       \
                MPM_SM1(RXV, ZSV, 32);                 \
        }                                              \
        break;
    switch (rs.zsb) {
        MPM_SM(4, 4)
        MPM_SM(4, 6)
        MPM_SM(4, 8)
        MPM_SM(4, 10)
        MPM_SM(2, 12)
        MPM_SM(2, 14)
        MPM_SM(2, 16)
        default:
            break;
    }
#undef MPM_SM
#undef MPM_SM1
    throw Error(MPM_ERR_RUNTIME, "slab size out of range");
}

// full grid with more than 32 candidates per region on average: four waves per region
// and column group take a candidate block each (30,000 particles, 4 right-hand sides:
// an apply 814 us, 839 with contract_full_mfma_kernel, 984 with contract_mfma_kernel)
inline bool dense_regions(const RegionSet& rs) {
    return !rs.slab && (rs.zsb == 4 || rs.slots > 32ll * rs.nreg);
}

template <typename R, int NC, typename GR>
inline void region_contract(ProfScope& ps, hipStream_t s, const RegionSet& rs, const RegionGeom& rg, bool vec, int B,
                            const R* regw, const typename C2<GR>::T* grid, R* pbuf) {
    // column groups of 16 per block: 4 when there are enough right-hand sides,
    // else fewer, with the region's planes split over the remaining waves; slab
    // with one or two column groups: one wave per candidate block instead
    const int ngrp = (2 * NC * B + 15) / 16;
    const int ncg = ngrp >= 4 ? 4 : (ngrp >= 2 ? 2 : 1);
    const dim3 gs((unsigned)rs.nreg, (unsigned)((ngrp + ncg - 1) / ncg));
    const dim3 gn((unsigned)rs.nreg, (unsigned)ngrp);
#define MPM_NB1(RXV, ZSV, VECV)                                                                               \
    do {                                                                                                      \
        ps.kernel("contract_nb_mfma_kernel", {type_name<R>(), #RXV, #ZSV, #VECV, NC, type_name<GR>()});       \
        hipLaunchKernelGGL((contract_nb_mfma_kernel<R, RXV, ZSV, VECV, NC, GR>), gn, dim3(256), 0, s, B, rg,      \
                           regw, rs.start, grid, pbuf);                                                       \
    } while (0)
#define MPM_CM1(RXV, ZSV, NBV, VECV)                                                                          \
    do {                                                                                                      \
        ps.kernel("contract_mfma_kernel", {type_name<R>(), #RXV, #ZSV, NBV, #VECV, NC, type_name<GR>()});     \
        hipLaunchKernelGGL((contract_mfma_kernel<R, RXV, ZSV, NBV, VECV, NC, GR>), gs, dim3(256), 0, s, B, rg,    \
                           regw, rs.start, grid, pbuf, ncg);                                                  \
    } while (0)
    if (dense_regions(rs)) {
        if (rs.zsb == 4) {
            if (vec) MPM_NB1(4, 4, true);
            else MPM_NB1(4, 4, false);
        } else {
            if (vec) MPM_NB1(4, 8, true);
            else MPM_NB1(4, 8, false);
        }
    } else if (!rs.slab && vec) {
        ps.kernel("contract_full_mfma_kernel",
                  {type_name<R>(), "4", kFullRegionPlanes, kFullContractNB, NC, type_name<GR>()});
        const int nitems = rs.nreg * ngrp;
        hipLaunchKernelGGL((contract_full_mfma_kernel<R, 4, kFullRegionPlanes, kFullContractNB, NC, GR>),
                           dim3((unsigned)((nitems + 3) / 4)), dim3(256), 0, s, B, rg, regw, rs.start, nitems, ngrp,
                           grid, pbuf);
    } else if (!rs.slab) {
        MPM_CM1(4, 8, kFullContractNB, false);
    } else if constexpr (NC == 8 || std::is_same<R, GR>::value) {  // dipole slabs sum in the grid's type
#define MPM_CM(RXV, ZSV)                                   \
    case ZSV:                                              \
        if constexpr (NC == 3 || ZSV <= kQuadSlabPlanes) { \
            if (ngrp <= 2) {                               \
                if (vec) MPM_NB1(RXV, ZSV, true);          \
                else MPM_NB1(RXV, ZSV, false);             \
            } else if (vec) {                              \
                MPM_CM1(RXV, ZSV, 4, true);                \
            } else {                                       \
                MPM_CM1(RXV, ZSV, 4, false);               \
            }                                              \
        }                                                  \
        break;
        switch (rs.zsb) {
            MPM_CM(4, 4)
            MPM_CM(4, 6)
            MPM_CM(4, 8)
            MPM_CM(4, 10)
            MPM_CM(2, 12)
            MPM_CM(2, 14)
            MPM_CM(2, 16)
            default:
                throw Error(MPM_ERR_RUNTIME, "slab size out of range");
        }
#undef MPM_CM
    } else {
        throw Error(MPM_ERR_RUNTIME, "no contraction of this slab in FP64");
    }
#undef MPM_CM1
#undef MPM_NB1
    MPM_HIP(hipGetLastError());
}

}  // namespace mpm

#endif  // MPM_REGION_MFMA_H
