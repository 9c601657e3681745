// Quadrupole operator (monodisperse): unknowns [3N dipole | 5Q quadrupole] components, a grid of
// 8 components (the field's 3, then the 5 quadrupole-gradient components) and the joint
// k-space coupling of monodisperse_ewald_electric_field.cu:1301-1487, 1631-1999.
//
// Spread and contraction are the region kernels of region_mfma.h with 16 real columns per
// right-hand side (exactly one column group of the matrix cores).  The grid is the z-plane slab
// where the dipole operator would take one (as far as quad_zcouple_kernel's registers reach, and
// where it needs no more memory), else the full grid, whose small problems contract per particle
// in the finish step.  Single stages work on full grids always.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "region_mfma.h"

namespace mpm {

static const double kPi = 3.14159265358979323846;

// Signed frequency index of grid index i on an axis of n points.
__device__ inline double freq(int i, int n) { return i <= (n - 1) / 2 ? i : i - n; }

// The four scalars of the coupling at wave vector k = (kx, ky, kz) with reciprocal vector G:
// sc (field of a dipole), scQ, scGP = -2 scQ, scGQ (:1301-1404), and 1 / |k|; zero at k = 0.
__device__ inline void quad_scalars(const KParams& q, double kx, double ky, double kz, double gx2eta, double o[4]) {
    o[0] = o[1] = o[2] = o[3] = 0.0;
    const double k2 = kx * kx + ky * ky + kz * kz, k = sqrt(k2);
    if (k < 1e-12) return;
    double sk, ck;
    sincos(k, &sk, &ck);
    const double t = sk / k - ck;
    const double ex = exp(-(k2 - gx2eta) / (4.0 * q.xi * q.xi));
    const double j1 = t / k, j2 = (3.0 / k2 - 1.0) * sk / k - 3.0 * ck / k2;
    const double e2 = ex / k2 * q.invV;
    o[0] = 9.0 * t * t * ex / (k2 * k2) * q.invV;
    o[1] = -22.5 * j1 * j2 * e2;
    o[2] = 112.5 * j2 * j2 * e2;
    o[3] = 1.0 / k;
}

// Full grid, coefficients of a voxel: khat (3), sc, scQ, scGP, scGQ, Qfactor (5), Qdot (first 4
// of 5; the last, 2 h1 h2, is formed from khat).
__device__ inline void quad_voxel(const KParams& q, size_t v, double o[16]) {
    const int ix = (int)(v / ((size_t)q.ny * q.nz)), iy = (int)((v / q.nz) % q.ny), iz = (int)(v % q.nz);
    const double Gx = freq(ix, q.nx) * 2.0 * kPi / q.Lx, Gy = freq(iy, q.ny) * 2.0 * kPi / q.Ly,
                 Gz = freq(iz, q.nz) * 2.0 * kPi / q.Lz;
    const double kx = Gx - q.kbx, ky = Gy - q.kby, kz = Gz;
    double f[4];
    for (int c = 0; c < 16; ++c) o[c] = 0.0;
    quad_scalars(q, kx, ky, kz, Gx * Gx * q.etax + Gy * Gy * q.etay + Gz * Gz * q.etaz, f);
    if (f[3] == 0.0) return;
    const double k = sqrt(kx * kx + ky * ky + kz * kz);
    const double h0 = kx / k, h1 = ky / k, h2 = kz / k;
    o[0] = h0;
    o[1] = h1;
    o[2] = h2;
    o[3] = f[0];
    o[4] = f[1];
    o[5] = -2.0 * f[1];
    o[6] = f[2];
    o[7] = h0 * h0 - 1.0 / 3.0;
    o[8] = h0 * h1;
    o[9] = h0 * h2;
    o[10] = h1 * h1 - 1.0 / 3.0;
    o[11] = h1 * h2;
    o[12] = h0 * h0 - h2 * h2;
    o[13] = 2.0 * h0 * h1;
    o[14] = 2.0 * h0 * h2;
    o[15] = h1 * h1 - h2 * h2;
}

__global__ void quad_kspace_kernel(double* __restrict__ k64, float* __restrict__ k32, KParams q) {
    const size_t V = (size_t)q.nx * q.ny * q.nz;
    for (size_t v = blockIdx.x * (size_t)blockDim.x + threadIdx.x; v < V; v += (size_t)gridDim.x * blockDim.x) {
        double o[16];
        quad_voxel(q, v, o);
        for (int c = 0; c < 16; ++c) {
            k64[16 * v + c] = o[c];
            k32[16 * v + c] = (float)o[c];
        }
    }
}

// Full grid: joint k-space coupling of field and gradient grids at a voxel with coefficients k
// (scale_kernel_joint, :1435-1487): Edk = E.khat, GQ = G.Qdot; E <- (sc Edk + i scQ GQ) khat,
// G <- (i scGP Edk + scGQ GQ) Qfactor.
template <typename R>
__device__ inline void quad_couple(const R (&k)[16], typename C2<R>::T* __restrict__ g, size_t V) {
    using CT = typename C2<R>::T;
    const R h0 = k[0], h1 = k[1], h2 = k[2];
    const R qd[5] = {k[12], k[13], k[14], k[15], R(2) * h1 * h2};
    CT f[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) f[c] = g[c * V];
    const R er = f[0].x * h0 + f[1].x * h1 + f[2].x * h2, ei = f[0].y * h0 + f[1].y * h1 + f[2].y * h2;
    R gr = R(0), gi = R(0);
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        gr += f[3 + c].x * qd[c];
        gi += f[3 + c].y * qd[c];
    }
    // i a (x + i y) = -a y + i a x
    const R sr = k[3] * er - k[4] * gi, si = k[3] * ei + k[4] * gr;
    const R tr = -k[5] * ei + k[6] * gr, ti = k[5] * er + k[6] * gi;
    const R hh[3] = {h0, h1, h2};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        CT o;
        o.x = sr * hh[c];
        o.y = si * hh[c];
        g[c * V] = o;
    }
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        CT o;
        o.x = tr * k[7 + c];
        o.y = ti * k[7 + c];
        g[(3 + c) * V] = o;
    }
}

// A thread per voxel and right-hand sides blockIdx.y, blockIdx.y + gridDim.y, ...: the voxel's
// 16 coefficients are read once for all of them.
template <typename R>
__global__ __launch_bounds__(256) void quad_scale_kernel(typename C2<R>::T* __restrict__ grid,
                                                         const R* __restrict__ kq, size_t V, int B) {
    const size_t v = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (v >= V) return;
    R k[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) k[c] = kq[16 * v + c];
    for (int b = blockIdx.y; b < B; b += gridDim.y) quad_couple<R>(k, grid + (size_t)b * 8 * V + v, V);
}

// ---- single stages of an operator whose applies run on the slab ----
//
// The caller's grid is a full grid [8][nx][ny][nz] of one right-hand side.  These kernels work
// from the slab's own region lists and weights and compute the coefficients they need, so that
// a stage allocates nothing and changes nothing of the operator (applies in flight go on).  A
// debugging path: one thread per voxel, one wave per particle, no matrix cores.

// Spread: a thread per voxel sums the candidates of its region in ascending particle order.
template <typename R>
__global__ __launch_bounds__(256) void quad_stage_spread_kernel(
    const double2* __restrict__ x, size_t n3, int nx, int ny, int nz, int RX, int nry, int zsb4,
    const double* __restrict__ regw, const int* __restrict__ reg_start, const int* __restrict__ reg_items,
    const int* __restrict__ reg_quads, const int* __restrict__ zmap, typename C2<R>::T* __restrict__ out) {
    using CT = typename C2<R>::T;
    const size_t V = (size_t)nx * ny * nz;
    const size_t v = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (v >= V) return;
    const int ix = (int)(v / ((size_t)ny * nz)), iy = (int)((v / nz) % ny), iz = (int)(v % nz);
    const int NW = 4 + zsb4 + kMfmaRY, p = zmap[iz];
    R ar[8], ai[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) ar[c] = ai[c] = R(0);
    if (p >= 0) {
        const int reg = (ix / RX) * nry + iy / kMfmaRY;
        const int k1 = reg_start[reg + 1];
        for (int k = reg_start[reg]; k < k1; ++k) {
            const double* w = regw + (size_t)k * NW;
            const R ww = (R)(w[ix % RX] * w[4 + zsb4 + iy % kMfmaRY] * w[4 + p]);
            if (ww == R(0)) continue;
            const double2* xp = x + 3 * (size_t)reg_items[k];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                ar[c] += ww * (R)xp[c].x;
                ai[c] += ww * (R)xp[c].y;
            }
            const int q = reg_quads ? reg_quads[k] : -1;
            if (q < 0) continue;
            const double2* xq = x + n3 + 5 * (size_t)q;
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                ar[3 + c] += ww * (R)xq[c].x;
                ai[3 + c] += ww * (R)xq[c].y;
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        CT o;
        o.x = ar[c];
        o.y = ai[c];
        out[c * V + v] = o;
    }
}

// Coupling with coefficients computed in place of the table's, rounded as the table's.
template <typename R>
__global__ __launch_bounds__(256) void quad_stage_scale_kernel(typename C2<R>::T* __restrict__ grid, KParams q) {
    const size_t V = (size_t)q.nx * q.ny * q.nz;
    const size_t v = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (v >= V) return;
    double o[16];
    quad_voxel(q, v, o);
    R k[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) k[c] = (R)o[c];
    quad_couple<R>(k, grid + v, V);
}

// Contraction: a wave per particle over its W^3 stencil voxels, summed in FP64.
template <typename R>
__global__ __launch_bounds__(256) void quad_stage_contract_kernel(
    const typename C2<R>::T* __restrict__ grid, int N, int nx, int ny, int nz, int W, const int* __restrict__ base,
    const double* __restrict__ w64, const int* __restrict__ qmap, double h3, double2* __restrict__ y) {
    const int lane = threadIdx.x & 63;
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= N) return;  // whole wave
    const size_t V = (size_t)nx * ny * nz;
    const int half = W / 2, qi = qmap[i];
    const int b0 = base[i] - half, b1 = base[N + i] - half, b2 = base[2 * (size_t)N + i] - half;
    const double* w = w64 + (size_t)i * 3 * W;
    double acc[8][2];
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c][0] = acc[c][1] = 0.0;
    for (int o = lane; o < W * W * W; o += 64) {
        const int oz = o % W, oy = (o / W) % W, ox = o / (W * W);
        // base lies in the box; the stencil may be wider than an axis
        int vx = (b0 + ox) % nx, vy = (b1 + oy) % ny, vz = (b2 + oz) % nz;
        vx += vx < 0 ? nx : 0;
        vy += vy < 0 ? ny : 0;
        vz += vz < 0 ? nz : 0;
        const double ww = w[ox] * w[W + oy] * w[2 * W + oz] * h3;
        const typename C2<R>::T* g = grid + ((size_t)vx * ny + vy) * nz + vz;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            acc[c][0] += ww * (double)g[c * V].x;
            acc[c][1] += ww * (double)g[c * V].y;
        }
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        acc[c][0] = wave_sum(acc[c][0]);
        acc[c][1] = wave_sum(acc[c][1]);
    }
    if (lane) return;
#pragma unroll
    for (int c = 0; c < 3; ++c) y[3 * (size_t)i + c] = make_double2(acc[c][0], acc[c][1]);
    if (qi < 0) return;
#pragma unroll
    for (int c = 0; c < 5; ++c)
        y[3 * (size_t)N + 5 * (size_t)qi + c] = make_double2(acc[3 + c][0], acc[3 + c][1]);
}

// Slab: coupling scalars (sc, scQ, scGQ, 1 / |k|) of every column and wave number kz = 0 ..
// floor(nz / 2) (an even nz's last is the Nyquist plane, kz = -nz / 2); the others follow from
// kz -> -kz, which changes none of them (the Bloch wave vector has no z component).
__global__ void quad_kslab_kernel(double* __restrict__ k64, float* __restrict__ k32, KParams q, int nh) {
    const size_t ncols = (size_t)q.ny * q.nxp, n = ncols * nh;
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
        const int iz = (int)(e / ncols), col = (int)(e - (size_t)iz * ncols);
        const int iy = col / q.nxp, ix = col - iy * q.nxp;
        double o[4] = {0.0, 0.0, 0.0, 0.0};
        if (ix < q.nx) {  // else padding
            const double Gx = freq(ix, q.nx) * 2.0 * kPi / q.Lx, Gy = freq(iy, q.ny) * 2.0 * kPi / q.Ly,
                         Gz = freq(iz, q.nz) * 2.0 * kPi / q.Lz;
            quad_scalars(q, Gx - q.kbx, Gy - q.kby, Gz, Gx * Gx * q.etax + Gy * Gy * q.etay + Gz * Gz * q.etaz, o);
        }
        for (int c = 0; c < 4; ++c) {
            k64[4 * e + c] = o[c];
            k32[4 * e + c] = (float)o[c];
        }
    }
}

// Slab: for every in-plane wave vector (column) and right-hand side, the z transform of the
// 8 components from the Zs planes to all wave numbers, the coupling, and the transform back,
// without a k-space grid in memory.  Two lanes per column and right-hand side, one for the real
// and one for the imaginary parts.
//
// The coupling has rank two, so only sums over components are transformed: with
// A = kx E_x + ky E_y, Z = E_z, G0 = kx^2 Q0 + 2 kx ky Q1 + ky^2 Q3, G1 = 2 (kx Q2 + ky Q4) and
// G2 = Q0 + Q3 (per plane, five sequences instead of eight),
//   Edk = (A^ + kz Z^) / k,  GQ = (G0^ + kz G1^ - kz^2 G2^) / k^2,
// and the outputs are combinations of the five back transforms of s / k, kz s / k, t, t / k^2
// and kz t / k^2 (s, t the two coupled scalars).  Wave numbers +-kz share their coefficients
// and the sums C = sum_a f_a cos, S = sum_a f_a sin (values C -+ i S): 9 + 10 multiply-adds
// per lane, plane and pair, all of real times real, so that the two lanes of a column meet
// only in the coupling (12 exchanges per pair).  cos / sin [kz][16 planes] are uniform over the
// wave (scalar loads).  Everything between the loads and the stores is FP64 over either grid:
// FP64 issues at the rate of unpacked FP32 here, and the sums of an FP32 grid stay as exact
// as the transforms around them.
//
// Bound by multiply-adds: about 7,000 instructions per lane for 9 planes and nz = 61
// (a thread for both parts, sums in FP32, held 256 registers and spilled: 330 against
// 285 us at 210 x 114 columns, 15 right-hand sides; the full grid's z transforms and scaling,
// which this replaces there, took 4.08 ms).  Planes past Zs hold zeros and are not stored.  Blocks are numbered so that each
// XCD keeps one column block for all right-hand sides (its coefficients stay in its L2).
constexpr int kQuadCols = 128;  // columns per block

template <typename R, int ZS>
__global__ __launch_bounds__(2 * kQuadCols, ZS < 10 ? 2 : 1) void quad_zcouple_kernel(
    typename C2<R>::T* __restrict__ kbuf, int B, int Zs, KParams q, const R* __restrict__ kc,
    const double* __restrict__ zcs, int nh, int ncb) {
    const int slot = blockIdx.x >> 3;
    const int cb = 8 * (slot / B) + (blockIdx.x & 7), b = slot % B;
    const int ncols = q.ny * q.nxp;
    const int col = cb * kQuadCols + (threadIdx.x >> 1), part = threadIdx.x & 1;
    if (cb >= ncb || col >= ncols) return;  // both lanes of a column
    const int iy = col / q.nxp, ix = col - iy * q.nxp;
    if (ix >= q.nx) return;  // padding: never read
    const double kx = freq(ix, q.nx) * 2.0 * kPi / q.Lx - q.kbx, ky = freq(iy, q.ny) * 2.0 * kPi / q.Ly - q.kby;
    const double dkz = 2.0 * kPi / q.Lz;
    const double sg = part ? -1.0 : 1.0;
    R* g = reinterpret_cast<R*>(kbuf + (size_t)b * 8 * Zs * ncols + col) + part;
    const size_t pstr = 2 * (size_t)ncols, cstr = (size_t)Zs * pstr;
    double fA[ZS], fZ[ZS], f0[ZS], f1[ZS], f2[ZS];
#pragma unroll
    for (int a = 0; a < ZS; ++a) {
        // planes past Zs: the last one's values, masked (no branch around the loads)
        const R* ga = g + min(a, Zs - 1) * pstr;
        double v[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = (double)keep_if(ga[c * cstr], a < Zs);
        fA[a] = kx * v[0] + ky * v[1];
        fZ[a] = v[2];
        f0[a] = kx * (kx * v[3] + 2.0 * ky * v[4]) + ky * ky * v[6];
        f1[a] = 2.0 * (kx * v[5] + ky * v[7]);
        f2[a] = v[3] + v[6];
    }
    double o0[ZS], o1[ZS], o2[ZS], o3[ZS], o4[ZS];  // s/k, kz s/k, t, t/k^2, kz t/k^2
#pragma unroll
    for (int a = 0; a < ZS; ++a) o0[a] = o1[a] = o2[a] = o3[a] = o4[a] = 0.0;
    using R4 = typename Mfma<R>::V4;
    const R4* kp = reinterpret_cast<const R4*>(kc) + col;
    R4 next = kp[0];
    for (int iz = 0; iz < nh; ++iz) {
        const R4 kq = next;  // the next pair's coefficients are fetched while this one is summed
        next = kp[(size_t)min(iz + 1, nh - 1) * ncols];
        const double sc = kq[0], scq = kq[1], scg = kq[2], ik = kq[3], scp = -2.0 * scq;
        const double* cs = zcs + 32 * iz;  // cos [16], sin [16]
        const bool nyq = 2 * iz == q.nz, single = iz == 0 || nyq;
        const double kz = (nyq ? -iz : iz) * dkz, kz2 = kz * kz;
        double cA = 0.0, sA = 0.0, cZ = 0.0, sZ = 0.0, cH = 0.0, sH = 0.0, cG = 0.0, sG = 0.0;
#pragma unroll
        for (int a = 0; a < ZS; ++a) {
            const double c = cs[a], s = cs[16 + a], h = f0[a] - kz2 * f2[a];
            cA += fA[a] * c;
            sA += fA[a] * s;
            cZ += fZ[a] * c;
            sZ += fZ[a] * s;
            cH += h * c;
            sH += h * s;
            cG += f1[a] * c;
            sG += f1[a] * s;
        }
        // this lane's part of the values at +kz (C - i S) and -kz (C + i S)
        sA = sg * swap_lane1(sA);
        sZ = sg * swap_lane1(sZ);
        sH = sg * swap_lane1(sH);
        sG = sg * swap_lane1(sG);
        const double ik2 = ik * ik;
        const double ep = ik * ((cA + sA) + kz * (cZ + sZ)), gp = ik2 * ((cH + sH) + kz * (cG + sG));
        const double em = single ? 0.0 : ik * ((cA - sA) - kz * (cZ - sZ));
        const double gm = single ? 0.0 : ik2 * ((cH - sH) - kz * (cG - sG));
        // s = sc Edk + i scQ GQ, t = i scGP Edk + scGQ GQ with scGP = -2 scQ, as sums and
        // differences over +-kz (i x: this lane's part is -sg times the other lane's)
        const double es = ep + em, ed = ep - em, gs = gp + gm, gd = gp - gm;
        const double ies = -sg * swap_lane1(es), ied = -sg * swap_lane1(ed), igs = -sg * swap_lane1(gs),
                     igd = -sg * swap_lane1(gd);
        const double ss = sc * es + scq * igs, sd = sc * ed + scq * igd;
        const double ts = scg * gs + scp * ies, td = scg * gd + scp * ied;
        // sums go with the cosines, i times the differences with the sines (sequences with a
        // factor kz: the other way round)
        const double iss = -sg * swap_lane1(ss), isd = -sg * swap_lane1(sd), its = -sg * swap_lane1(ts),
                     itd = -sg * swap_lane1(td);
        const double kk = ik * kz, kk2 = ik2 * kz;
        const double c0 = ik * ss, s0 = ik * isd, c1 = kk * sd, s1 = kk * iss, c3 = ik2 * ts, s3 = ik2 * itd,
                     c4 = kk2 * td, s4 = kk2 * its;
#pragma unroll
        for (int a = 0; a < ZS; ++a) {
            const double c = cs[a], s = cs[16 + a];
            o0[a] += c0 * c + s0 * s;
            o1[a] += c1 * c + s1 * s;
            o2[a] += ts * c + itd * s;
            o3[a] += c3 * c + s3 * s;
            o4[a] += c4 * c + s4 * s;
        }
    }
#pragma unroll
    for (int a = 0; a < ZS; ++a) {
        if (a < Zs) {
            R* o = g + a * pstr;
            const double tr = o2[a] * (1.0 / 3.0);
            o[0] = (R)(kx * o0[a]);
            o[cstr] = (R)(ky * o0[a]);
            o[2 * cstr] = (R)o1[a];
            o[3 * cstr] = (R)(kx * kx * o3[a] - tr);
            o[4 * cstr] = (R)(kx * ky * o3[a]);
            o[5 * cstr] = (R)(kx * o4[a]);
            o[6 * cstr] = (R)(ky * ky * o3[a] - tr);
            o[7 * cstr] = (R)(ky * o4[a]);
        }
    }
}

// NL lanes per (particle, right-hand side), lanes then right-hand sides fastest, particles
// in spatial order: the particle's region contractions (partial [slot][16 B], null: none) or with
// GATHER the contraction itself over the particle's stencil voxels of the full grid, the
// real-space couplings of every neighbour's dipole and quadrupole (dipole -> field,
// quadrupole -> field, dipole -> gradient, quadrupole -> gradient, :1631-1869 with the
// cross-term signs of tests/quadrupole_field.py:214-215), the self terms (sc + self_perp for
// the field, 2.5 sc + self_grad / 2 for the gradient) and the optional left Jacobi scaling.
// Each lane takes every NL-th slot or voxel and neighbour; a butterfly sum over the lanes (fixed
// order) leaves component c of the result in lane c, which stores it.  FP64 sums.  Pair data [16]:
// u (3), perp, para - perp, cos, sin, field_quad_1..3, grad_quad_1..4.
constexpr int kQuadLanes = 8;

// Stencils of the full grid for the gather.
struct QuadStencil {
    int n[3], W, m;           // m = 65536 / W + 1: o / W = o m >> 16 for o < W^3 <= 13^3
    const int* base;          // [3][N] wrapped base voxel
    const double* w64;        // [N][3][W]
};

template <int NL, bool GATHER, typename R>
__global__ __launch_bounds__(256) void quad_finish_kernel(SlotTable tab, int B, int parts, int N,
                                                          const double* __restrict__ partial,
                                                          const int* __restrict__ ps_start,
                                                          const int* __restrict__ ps_items,
                                                          const int* __restrict__ qmap, double h3,
                                                          const int* __restrict__ nb_start,
                                                          const int* __restrict__ nb_j,
                                                          const double* __restrict__ pairq,
                                                          const double2* __restrict__ selfc, double self_perp,
                                                          double self_grad, int jacobi,
                                                          const int* __restrict__ order,
                                                          const typename C2<R>::T* __restrict__ grid,
                                                          QuadStencil st) {
    __shared__ const double2* s_x[kMaxSlots];
    __shared__ double2* s_y[kMaxSlots];
    __shared__ int s_row[kMaxSlots];
#pragma unroll
    for (int k = 0; k < kMaxSlots; ++k)  // uniform indices: no per-lane walk of the argument
        if (threadIdx.x == k) {
            s_x[k] = tab.x[k];
            s_y[k] = tab.y[k];
            s_row[k] = tab.row[k];
        }
    __syncthreads();
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int item = t / NL, sub = t % NL;  // NL divides the wave: the lanes of an item share it
    const int ii = item / B, b = item - ii * B;
    if (ii >= N) return;  // whole items only
    const int i = order[ii];
    const int qi = qmap[i];
    const double2* x = s_x[b];
    double acc[8][2];
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c][0] = acc[c][1] = 0.0;
    if constexpr (GATHER) {
        if (parts & MPM_PART_RECIP) {
            const size_t plane = (size_t)st.n[1] * st.n[2], V = st.n[0] * plane;
            const typename C2<R>::T* g = grid + (size_t)b * 8 * V;
            const double* w = st.w64 + (size_t)i * 3 * st.W;
            int s[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                s[d] = (st.base[(size_t)d * N + i] - st.W / 2) % st.n[d];
                s[d] += s[d] < 0 ? st.n[d] : 0;
            }
            const int SS = st.W * st.W * st.W;
            for (int o = sub; o < SS; o += NL) {
                const int oxy = o * st.m >> 16, ox = oxy * st.m >> 16;
                const int oy = oxy - ox * st.W, oz = o - oxy * st.W;
                int v[3] = {s[0] + ox, s[1] + oy, s[2] + oz};
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    while (v[d] >= st.n[d]) v[d] -= st.n[d];  // more than once where W exceeds the axis
                const double ww = w[ox] * w[st.W + oy] * w[2 * st.W + oz];
                const typename C2<R>::T* gv = g + v[0] * plane + (size_t)v[1] * st.n[2] + v[2];
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    if (c < 3 || qi >= 0) {
                        acc[c][0] += ww * (double)gv[c * V].x;
                        acc[c][1] += ww * (double)gv[c * V].y;
                    }
            }
        }
    } else if (partial) {
        const int s1 = ps_start[i + 1];
        for (int sl = ps_start[i] + sub; sl < s1; sl += NL) {
            const double* pp = partial + ((size_t)ps_items[sl] * B + b) * 16;
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                acc[c][0] += pp[2 * c];
                acc[c][1] += pp[2 * c + 1];
            }
        }
    }
    if (GATHER || partial) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            acc[c][0] *= h3;
            acc[c][1] *= h3;
        }
    }
    if (parts & MPM_PART_REAL) {
        const int k1 = nb_start[i + 1];
        for (int k = nb_start[i] + sub; k < k1; k += NL) {
            const int jn = nb_j[k];
            const int qs = qmap[jn];
            const double* pc = pairq + 16 * (size_t)k;
            const double u[3] = {pc[0], pc[1], pc[2]};
            const double cp = pc[3], cd = pc[4], ec = pc[5], es = pc[6];
            const double t0 = pc[7], t1 = pc[8], t2 = pc[9], g1 = pc[10], g2 = pc[11], g3 = pc[12], g4 = pc[13];
            const double rr[5] = {u[0] * u[0], u[0] * u[1], u[0] * u[2], u[1] * u[1], u[1] * u[2]};
            const double I5[5] = {1.0, 0.0, 0.0, 1.0, 0.0};
            double2 pp[3], qq[5];
#pragma unroll
            for (int c = 0; c < 3; ++c) pp[c] = x[3 * (size_t)jn + c];
            const size_t qb = 3 * (size_t)N + 5 * (size_t)max(qs, 0);
#pragma unroll
            for (int c = 0; c < 5; ++c) qq[c] = qs >= 0 ? x[qb + c] : make_double2(0.0, 0.0);
            double f[8][2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const double p0 = h ? pp[0].y : pp[0].x, p1 = h ? pp[1].y : pp[1].x, p2 = h ? pp[2].y : pp[2].x;
                const double qv[5] = {h ? qq[0].y : qq[0].x, h ? qq[1].y : qq[1].x, h ? qq[2].y : qq[2].x,
                                      h ? qq[3].y : qq[3].x, h ? qq[4].y : qq[4].x};
                const double rp = p0 * u[0] + p1 * u[1] + p2 * u[2];
                const double Qr[3] = {qv[0] * u[0] + qv[1] * u[1] + qv[2] * u[2],
                                      qv[1] * u[0] + qv[3] * u[1] + qv[4] * u[2],
                                      qv[2] * u[0] + qv[4] * u[1] - (qv[0] + qv[3]) * u[2]};
                const double Qrr = Qr[0] * u[0] + Qr[1] * u[1] + Qr[2] * u[2];
                const double pv[3] = {p0, p1, p2};
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    f[c][h] = cp * pv[c] + cd * rp * u[c] + 0.5 * (Qrr * t0 * u[c] + 2.0 * t1 * Qr[c]);
                const double PrrP[5] = {2.0 * p0 * u[0], p0 * u[1] + p1 * u[0], p0 * u[2] + p2 * u[0],
                                        2.0 * p1 * u[1], p1 * u[2] + p2 * u[1]};
                const double QrrQ[5] = {2.0 * Qr[0] * u[0], Qr[0] * u[1] + Qr[1] * u[0], Qr[0] * u[2] + Qr[2] * u[0],
                                        2.0 * Qr[1] * u[1], Qr[1] * u[2] + Qr[2] * u[1]};
#pragma unroll
                for (int c = 0; c < 5; ++c)
                    f[3 + c][h] = 0.5 * (Qrr * ((g1 + g3) * I5[c] + g4 * rr[c]) + qv[c] * g2 + 2.0 * g3 * QrrQ[c]) -
                                  (rp * (t0 * rr[c] + (t1 + t2) * I5[c]) + PrrP[c] * t1);
            }
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                acc[c][0] += f[c][0] * ec - f[c][1] * es;
                acc[c][1] += f[c][0] * es + f[c][1] * ec;
            }
        }
    }
#pragma unroll
    for (int m = 1; m < NL; m <<= 1)
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            acc[c][0] += __shfl_xor(acc[c][0], m, NL);
            acc[c][1] += __shfl_xor(acc[c][1], m, NL);
        }
    const int c = sub;
    if (c >= (qi >= 0 ? 8 : 3)) return;
    double yr = 0.0, yi = 0.0;
#pragma unroll
    for (int cc = 0; cc < 8; ++cc)
        if (cc == c) {
            yr = acc[cc][0];
            yi = acc[cc][1];
        }
    const size_t e = c < 3 ? 3 * (size_t)i + c : 3 * (size_t)N + 5 * (size_t)qi + (c - 3);
    const double2 sc = selfc[(size_t)s_row[b] * N + i];
    if (parts & MPM_PART_REAL) {
        const double2 xv = x[e];
        const double fr = c < 3 ? sc.x + self_perp : 2.5 * sc.x + 0.5 * self_grad;
        const double fi = c < 3 ? sc.y : 2.5 * sc.y;
        yr += fr * xv.x - fi * xv.y;
        yi += fr * xv.y + fi * xv.x;
    }
    double2 inv = make_double2(1.0, 0.0);
    if (jacobi) {
        const double den = sc.x * sc.x + sc.y * sc.y;
        if (den > 1e-30) inv = make_double2(sc.x / den, -sc.y / den);
    }
    s_y[b][e] = make_double2(yr * inv.x - yi * inv.y, yr * inv.y + yi * inv.x);
}

// k-space tables of the current layout, positions aside.
void EwaldOp::build_quad_tables() {
    const int threads = 256;
    if (!slab) {
        d_kq64.resize(16 * V);
        d_kq32.resize(16 * V);
        const int blocks = (int)std::min<size_t>((V + threads - 1) / threads, 65535);
        hipLaunchKernelGGL(quad_kspace_kernel, dim3(blocks), dim3(threads), 0, nullptr, d_kq64.p, d_kq32.p, kparams());
        MPM_HIP(hipGetLastError());
        return;
    }
    const int nh = S.n[2] / 2 + 1;
    const size_t n = (size_t)nh * kspace_cols();
    d_kqs64.resize(4 * n);
    d_kqs32.resize(4 * n);
    const int blocks = (int)std::min<size_t>((n + threads - 1) / threads, 65535);
    hipLaunchKernelGGL(quad_kslab_kernel, dim3(blocks), dim3(threads), 0, nullptr, d_kqs64.p, d_kqs32.p, kparams(), nh);
    MPM_HIP(hipGetLastError());
}

// cos and sin of 2 pi kz z_a / nz, [kz][16 cos, 16 sin], of the slab's planes z_a: these move
// with the particles, also where their number stays.
void EwaldOp::build_quad_phases() {
    if (zcs_planes == zlist && zcs_nz == S.n[2]) return;
    const int nz = S.n[2], nh = nz / 2 + 1;
    std::vector<double> zc((size_t)32 * nh, 0.0);
    for (int k = 0; k < nh; ++k)
        for (int a = 0; a < Zs; ++a) {
            const int m = (int)(((long long)k * zlist[a]) % nz);
            zc[32 * (size_t)k + a] = std::cos(2.0 * kPi * m / nz);
            zc[32 * (size_t)k + 16 + a] = 2 * m == nz || m == 0 ? 0.0 : std::sin(2.0 * kPi * m / nz);
        }
    zcs_planes.clear();
    d_zcs64.upload(zc.data(), zc.size());
    zcs_planes = zlist;
    zcs_nz = nz;
}

// The contraction as part of the finish step, a wave per particle and right-hand side over the
// stencil voxels of the full grid: up to three waves per SIMD one launch and more lanes decide
// (FP32, an apply with the gather / on the regions: 900 particles with 7-point stencils, 1
// right-hand side 61 / 87 us, 2 70 / 92, 4 108 / 121, 8 152 / 160; 1500 with 9-point stencils, 1 86 /
// 102, 2 113 / 122, 4 184 / 157; 3000 with 5-point stencils, 1 77 / 87, 2 99 / 93).  The slab, whose
// regions hold all planes, is faster on the regions at every size.
bool EwaldOp::quad_gather(int B) const { return !slab && N * B <= 3072; }

template <typename R>
void EwaldOp::launch_quads(const SlotTable& t, int B, int parts, hipStream_t s, int jacobi) {
    using CT = typename C2<R>::T;
    const bool fp32 = std::is_same<R, float>::value;
    CT* grid = reinterpret_cast<CT*>(cur_grid);
    CT* kgrid = reinterpret_cast<CT*>(cur_kgrid);
    const int Ni = (int)N;
    const RegionSet rs = region_set(slab);
    const RegionGeom rg = region_geom(slab);
    // the region kernels address the grid with 32-bit element offsets
    MPM_REQUIRE(!(parts & MPM_PART_RECIP) || 2ull * (unsigned long long)B * grid_elems_per_rhs() < (1ull << 32),
                MPM_ERR_UNSUPPORTED, "reciprocal grid too large for one transform call");
    if ((parts & MPM_PART_RECIP) && (phases & 1)) {
        ProfScope ps("spread", s, B);
        region_spread<R, 8>(ps, s, rs, rg, t, B, d_regw64.p, 3 * (size_t)N, grid);
    }
    if ((parts & MPM_PART_RECIP) && (phases & 2)) {
        {
            ProfScope ps("fft", s, B);
            line_fft<R>(grid, slab ? kgrid : grid, B, true, s);
        }
        if (slab) {
            ProfScope ps("zfused", s, B);
            const int nh = S.n[2] / 2 + 1, ncb = (kspace_cols() + kQuadCols - 1) / kQuadCols;
            const dim3 gz((unsigned)(8 * ((ncb + 7) / 8) * B));
            const R* kc = fp32 ? reinterpret_cast<const R*>(d_kqs32.p) : reinterpret_cast<const R*>(d_kqs64.p);
#define MPM_QZ(ZSV)                                                                                               \
    case ZSV:                                                                                                     \
        ps.kernel("quad_zcouple_kernel", {type_name<R>(), #ZSV});                                                 \
        hipLaunchKernelGGL((quad_zcouple_kernel<R, ZSV>), gz, dim3(2 * kQuadCols), 0, s, kgrid, B, Zs, kparams(), kc, \
                           d_zcs64.p, nh, ncb);                                                                   \
        break;
            switch (Zs == 9 ? 9 : rs.zsb) {
                MPM_QZ(4)
                MPM_QZ(6)
                MPM_QZ(8)
                MPM_QZ(9)  // a flat layer with 9-point stencils
                MPM_QZ(10)
                default:
                    throw Error(MPM_ERR_RUNTIME, "slab size out of range");
            }
#undef MPM_QZ
            MPM_HIP(hipGetLastError());
        } else {
            ProfScope ps("scale", s, B);
            ps.kernel("quad_scale_kernel", {type_name<R>()});
            const R* kq = fp32 ? reinterpret_cast<const R*>(d_kq32.p) : reinterpret_cast<const R*>(d_kq64.p);
            const unsigned nb = (unsigned)((V + 255) / 256);
            // right-hand sides of a voxel in one thread once the voxels alone fill the GPU
            const unsigned gy = (unsigned)std::min<size_t>(B, std::max<size_t>(1, 4096 / nb));
            hipLaunchKernelGGL((quad_scale_kernel<R>), dim3(nb, gy), dim3(256), 0, s, grid, kq, V, B);
            MPM_HIP(hipGetLastError());
        }
        {
            ProfScope ps("fft", s, B);
            line_fft<R>(grid, slab ? kgrid : grid, B, false, s);
        }
    }
    if (!(phases & 4)) return;
    const bool gather = quad_gather(B);
    const double* part = nullptr;
    if (!gather && (parts & MPM_PART_RECIP)) {  // summed in FP64 over either grid
        ProfScope ps("contract", s, B);
        const bool aligned = (reinterpret_cast<uintptr_t>(grid) % 32) == 0;
        const bool vec = aligned && (slab ? (nyp % 2 == 0 && S.n[1] % 2 == 0) : S.n[2] % 2 == 0);
        region_contract<double, 8, R>(ps, s, rs, rg, vec, B, d_regw64.p, grid, d_partial64.p);
        part = d_partial64.p;
    }
    ProfScope ps("gather", s, B);
    const double h3 = S.h[0] * S.h[1] * S.h[2];
    const QuadStencil st{{S.n[0], S.n[1], S.n[2]}, S.width, 65536 / S.width + 1, d_base.p, d_w64.p};
    auto finish = [&](auto kernel, int lanes) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(((size_t)Ni * B * lanes + 255) / 256)), dim3(256), 0, s, t, B, parts,
                           Ni, part, d_ps_start.p, d_ps_items.p, d_qmap.p, h3, d_nb_start.p, d_nb_j.p, d_pairc.p,
                           d_selfc.p, self_perp, quad_self_grad, jacobi, d_order.p, grid, st);
    };
    ps.kernel("quad_finish_kernel", {gather ? 64 : kQuadLanes, tbool(gather), type_name<R>()});
    if (gather) finish(quad_finish_kernel<64, true, R>, 64);
    else finish(quad_finish_kernel<kQuadLanes, false, R>, kQuadLanes);
    MPM_HIP(hipGetLastError());
}
template void EwaldOp::launch_quads<float>(const SlotTable&, int, int, hipStream_t, int);
template void EwaldOp::launch_quads<double>(const SlotTable&, int, int, hipStream_t, int);

// The W^3 points of every particle, their wrapped voxels and Gaussian weights
// C exp(-2 xi^2 sum gd^2/eta) (the dipole weights, :687-816) as the reference keeps them; the
// kernels work from separable weights, so these exist for callers that ask for their address:
// built when first asked for, and from then on by every set_positions.
void EwaldOp::ensure_quad_stencils() {
    quad_stencils_wanted = true;
    if (quad_stencils_valid || N == 0 || last_xyz.empty()) return;
    const int W = S.width, half = S.half, Nn = (int)N;
    const int SS = W * W * W;
    const double prod_eta = S.eta[0] * S.eta[1] * S.eta[2];
    const double Cs = std::pow(2.0 * xi * xi / kPi, 1.5) * std::sqrt(1.0 / prod_eta);
    std::vector<double> sw((size_t)Nn * SS);
    std::vector<int> pidx((size_t)Nn * SS);
    for (int i = 0; i < Nn; ++i) {
        int g[3];
        double dd[3];
        for (int d = 0; d < 3; ++d) {
            const double p = last_xyz[3 * (size_t)i + d];
            g[d] = (int)std::round(p / S.h[d]);
            dd[d] = g[d] * S.h[d] - p;
        }
        size_t item = (size_t)i * SS;
        for (int ox = -half; ox <= half; ++ox)
            for (int oy = -half; oy <= half; ++oy)
                for (int oz = -half; oz <= half; ++oz, ++item) {
                    const int off[3] = {ox, oy, oz};
                    double a = 0.0;
                    int w[3];
                    for (int d = 0; d < 3; ++d) {
                        w[d] = ((g[d] + off[d]) % S.n[d] + S.n[d]) % S.n[d];
                        const double gd = dd[d] + off[d] * S.h[d];
                        a += gd * gd / S.eta[d];
                    }
                    pidx[item] = (w[0] * S.n[1] + w[1]) * S.n[2] + w[2];
                    sw[item] = Cs * std::exp(-2.0 * xi * xi * a);
                }
    }
    std::vector<float> sw32(sw.begin(), sw.end());
    d_sw64.upload(sw.data(), sw.size());
    d_sw32.upload(sw32.data(), sw32.size());
    d_pidx.upload(pidx.data(), pidx.size());
    quad_stencils_valid = true;
}

// The full-grid coefficient table, for callers that ask for its address (kept current from
// then on, as the stencils).
void EwaldOp::ensure_quad_scale_coef() {
    quad_coef_wanted = true;
    if (!slab || N == 0 || quad_coef_valid) return;
    d_kq64.resize(16 * V);
    d_kq32.resize(16 * V);
    const int blocks = (int)std::min<size_t>((V + 255) / 256, 65535);
    hipLaunchKernelGGL(quad_kspace_kernel, dim3(blocks), dim3(256), 0, nullptr, d_kq64.p, d_kq32.p, kparams());
    MPM_HIP(hipGetLastError());
    MPM_HIP(hipDeviceSynchronize());
    quad_coef_valid = true;
}

void EwaldOp::refresh_quad_addresses() {
    if (quad_stencils_wanted) ensure_quad_stencils();
    if (quad_coef_wanted) ensure_quad_scale_coef();
}

// Stage `which` (1 spread, 2 transforms and coupling, 3 contraction into y) of one right-hand
// side on a full grid, for an operator whose applies run on the slab.
template <typename R>
void EwaldOp::stage_quads_full(int which, const double2* x, void* grid, double2* y, hipStream_t s) {
    using CT = typename C2<R>::T;
    CT* g = reinterpret_cast<CT*>(grid);
    const dim3 gv((unsigned)((V + 255) / 256)), blk(256);
    if (which == 1) {
        ProfScope ps("spread", s, 1);
        ps.kernel("quad_stage_spread_kernel", {type_name<R>()});
        hipLaunchKernelGGL((quad_stage_spread_kernel<R>), gv, blk, 0, s, x, 3 * (size_t)N, S.n[0], S.n[1], S.n[2],
                           reg_rx, reg_nry, (region_set(true).zsb + 3) & ~3, d_regw64.p, d_reg_start.p, d_reg_items.p,
                           qidx_h.empty() ? nullptr : d_reg_quads.p, d_zmap.p, g);
    } else if (which == 2) {
        {
            ProfScope ps("fft", s, 1);
            stage_fft<R>(grid, true, s);
        }
        {
            ProfScope ps("scale", s, 1);
            ps.kernel("quad_stage_scale_kernel", {type_name<R>()});
            hipLaunchKernelGGL((quad_stage_scale_kernel<R>), gv, blk, 0, s, g, kparams());
            MPM_HIP(hipGetLastError());
        }
        ProfScope ps("fft", s, 1);
        stage_fft<R>(grid, false, s);
    } else {
        ProfScope ps("contract", s, 1);
        ps.kernel("quad_stage_contract_kernel", {type_name<R>()});
        hipLaunchKernelGGL((quad_stage_contract_kernel<R>), dim3((unsigned)((N + 3) / 4)), blk, 0, s, g, (int)N, S.n[0],
                           S.n[1], S.n[2], S.width, d_base.p, d_w64.p, d_qmap.p, S.h[0] * S.h[1] * S.h[2], y);
    }
    MPM_HIP(hipGetLastError());
}
template void EwaldOp::stage_quads_full<float>(int, const double2*, void*, double2*, hipStream_t);
template void EwaldOp::stage_quads_full<double>(int, const double2*, void*, double2*, hipStream_t);

}  // namespace mpm
