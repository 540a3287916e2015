// pair_device.h -- device building blocks of the direct pair kernels: the pair
// terms of every variant, table interpolation, wraps and far-tile tests, and
// the scalars a launch carries.  Included by the translation units that hold
// pair kernels (everything here has internal linkage).
#pragma once

#include "internal.h"

#include <algorithm>
#include <cmath>

namespace steps {

namespace {

struct KScalars {
    int64_t N;
    int64_t id_min;
    int64_t nrows;
    int64_t jchunk;
    double L, halfL;
    // T3 table: grid nodes per axis, first x/y node of the device layout
    int ng, t3_lo;
    // S1R2 table
    int nrho, nz;
    double rho_max;
    // S1R2 image sum
    int images;
    double image_cut;
    // Newton-correction constant, passed in so that it lives in a register
    // for the whole loop instead of being rematerialised per pair
    double c15;
    // -5/3, the constant of mr3_scaled
    double cm53;
    // reciprocals of the table grid spacings: T3 Ng/L, S1R2 1/drho and Nz/Lz
    double inv_gs, inv_drho, inv_dzg;
    double last_r;  // S1R2: index of the last rho node, Nrho - 1 (Nrho >= 2)
    // FP32 copies for the mixed-precision S1R2 pair
    float Lf, halfLf, rho_maxf, inv_drhof, inv_dzgf, last_rf;
    float inv_gsf;  // FP32 copy of inv_gs for the mixed-precision T3 pair
    float wrap_epsf;  // 1e-6 L: the band around |d| = L/2 where an FP32 displacement may wrap otherwise
};

// ---------------------------------------------------------------------------
// FP64 building blocks
// ---------------------------------------------------------------------------

// Copy a wave-uniform constant into a VGPR once, so that an FMA taking it and
// another SGPR constant (VOP3 reads at most one SGPR on gfx9) does not
// re-materialise it with a v_mov in every pair.
__device__ __forceinline__ double in_vgpr(double x) {
    double r;
    asm("v_mov_b64 %0, %1" : "=v"(r) : "s"(x));
    return r;
}

// r2^(-3/2): v_rsq_f64 seed y (relative error |d| <= 5.2e-8 on gfx950,
// probed), e = 1 - r2*y^2 ~= -2d, y^3 * (1 - e)^(-3/2) ~= y^3 * (1 + 1.5 e).
// The dropped terms, 1.875 e^2 + ..., bound the relative error by 2.1e-14
// (one-sided: the result is never too large); one correction term instead of
// two saves an FMA per pair (3.5% of the R3 pair kernel, measured).
// r2 == 0 gives NaN: the caller's softening branch owns it.
__device__ __forceinline__ double inv_r3(double r2, double c15) {
    const double y = __builtin_amdgcn_rsq(r2);
    const double t = y * y;
    const double e = fma(-r2, t, 1.0);
    return (t * y) * fma(e, c15, 1.0);
}

// m r2^(-3/2) for a source whose record carries mp = -1.5 m (the FP64 R3 and
// nearest-image kernels' source copies, tiles_kernel): with y = rsq(r2) and
// t = y^2, mp y^3 (r2 t - 5/3) = m y^3 (2.5 - 1.5 r2 t) = m y^3 (1 + 1.5 e),
// e = 1 - r2 t, which is inv_r3's first-order correction times m, in 5 VALU
// (y m', t (y m'), r2 t - 5/3, the product, and t) instead of inv_r3's 5 plus
// the mass multiply.  r2 t - 5/3 lies near -2/3, so its rounding adds 1 ulp.
__device__ __forceinline__ double mr3_scaled(double r2, double mp, double cm53) {
    const double y = __builtin_amdgcn_rsq(r2);
    const double t = y * y;
    const double b = t * (y * mp);
    return b * fma(r2, t, cm53);
}

// The mass of a source whose record carries -1.5 m (within 2 ulp of m); only
// the rare pairs inside the softening length need it.
__device__ __forceinline__ double unscaled_mass(double mp) { return mp * (-2.0 / 3.0); }

// forces_cuda.cu:466-519, written out as the reference does (beta powers and
// divisions); only reached for r < beta, so its cost does not matter.
__device__ __forceinline__ double softening_exact(double r, double beta) {
    const double half_beta = beta * 0.5;
    const double r2 = r * r;
    const double r3 = r2 * r;
    const double inv_r3v = 1.0 / r3;
    if (r >= beta) return inv_r3v;
    const double b2 = beta * beta, b3 = b2 * beta, b4 = b2 * b2, b5 = b4 * beta, b6 = b3 * b3;
    if (r > half_beta) {
        const double c0 = -32.0 / (3.0 * b6), c1 = 38.4 / b5, c2 = -48.0 / b4;
        const double c3 = 64.0 / (3.0 * b3), c4 = -1.0 / 15.0;
        return c0 * r3 + c1 * r2 + c2 * r + c3 + c4 * inv_r3v;
    }
    const double c0 = 32.0 / b6, c1 = -38.4 / b5, c2 = (32.0 / 3.0) / b3;
    return c0 * r3 + c1 * r2 + c2;
}

__device__ __forceinline__ int imodp(int i, int n) {
    int r = i % n;  // forces_cuda.cu:87-92
    return (r < 0) ? (r + n) : r;
}

// imodp(i, n) without an integer division for i in [-n, 2n), which covers
// every index a nearest-image displacement produces; other values (positions
// outside the box) take the general remainder in a branch waves rarely enter.
__device__ __forceinline__ int wrap_index(int i, int n) {
    int r = (i < 0) ? i + n : ((i >= n) ? i - n : i);
    if ((unsigned)r >= (unsigned)n) r = imodp(i, n);
    return r;
}

// One period step for an index known to lie in [-n, 2n).
__device__ __forceinline__ int wrap_once(int i, int n) {
    return (i < 0) ? i + n : ((i >= n) ? i - n : i);
}

// x^(-1/2) for x > 0: v_rsq_f64 seed and a first-order Newton correction,
// y * (1 - e)^(-1/2) ~= y * (1 + e/2) with e = 1 - x*y^2; the dropped
// 3e^2/8 bounds the relative error by 4e-15.
__device__ __forceinline__ double rsqrt_f64(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x, y * y, 1.0);
    return fma(y * e, 0.5, y);
}

// Eight-byte aligned pair of doubles: a 16-byte load at any 8-byte boundary.
typedef double double2u __attribute__((ext_vector_type(2), aligned(8)));

// Catmull-Rom weights and first node of one axis (forces_cuda.cu:93-111):
// u in grid units from the first cell centre, nodes i0-1 .. i0+2.
__device__ __forceinline__ int t3_axis(double d, const KScalars &k, double w[4]) {
    const double u = (d + k.L * 0.5) * k.inv_gs - 0.5;
    const double uf = floor(u);
    const double t = u - uf;
    const double t2 = t * t, t3 = t * t2;
    w[0] = -0.5 * t3 + t2 - 0.5 * t;
    w[1] = 1.5 * t3 - 2.5 * t2 + 1.0;
    w[2] = -1.5 * t3 + 2.0 * t2 + 0.5 * t;
    w[3] = 0.5 * t3 - 0.5 * t2;
    return wrap_index((int)uf, k.ng);
}

// forces_cuda.cu:93-167: tricubic Catmull-Rom interpolation of the T3 table
// (cell-centred grid, periodic index wrap), read from the device layout of
// t3_device_layout: x and y nodes lo..Ng-1, a node i < lo read at its mirror
// Ng-1-i with its own component negated (the sign rides on that axis'
// weight, so x-negated and y-negated values never need a select), and each
// stencil's four z nodes as twelve contiguous doubles (six 16-byte loads).
// The contraction runs z, then y, then x: Sum_i wx_i Sum_j wy_j Sum_k wz_k T.
// The reference divides by the grid spacing; multiplying by its reciprocal
// moves u by at most an ulp, and the interpolant is continuous in u.
struct T3Stencil {
    double wx[4], wy[4], wz[4], wxs[4], wys[4];
    unsigned mx[4], my[4];  // layout x / y node of each stencil plane
    int iz0;                // first z node + 1 = layout z index of the run
};

__device__ __forceinline__ void t3_stencil(const KScalars &k, double dx, double dy, double dz, T3Stencil &s) {
    const int Ng = k.ng, lo = k.t3_lo;
    const int ix0 = t3_axis(dx, k, s.wx);
    const int iy0 = t3_axis(dy, k, s.wy);
    s.iz0 = t3_axis(dz, k, s.wz);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int jx = wrap_once(ix0 - 1 + q, Ng);  // Ng >= 3
        const int jy = wrap_once(iy0 - 1 + q, Ng);
        s.mx[q] = (unsigned)((jx >= lo) ? jx - lo : Ng - 1 - lo - jx);
        s.my[q] = (unsigned)((jy >= lo) ? jy - lo : Ng - 1 - lo - jy);
        s.wxs[q] = (jx >= lo) ? s.wx[q] : -s.wx[q];
        s.wys[q] = (jy >= lo) ? s.wy[q] : -s.wy[q];
    }
}

// The staged contraction over the 16 (x, y) rows; load(i, j, v) fills v with
// the stencil's twelve z-run values of table row (mx[i], my[j]), node-major
// (v[3q + c] = component c of z node q).
template <class Load>
__device__ __forceinline__ void t3_contract(const T3Stencil &s, Load load, double &Dx, double &Dy, double &Dz) {
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        double u0 = 0.0, u1 = 0.0, u2 = 0.0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            double v[12];
            load(i, j, v);
            double t0 = s.wz[0] * v[0], t1 = s.wz[0] * v[1], t2 = s.wz[0] * v[2];
#pragma unroll
            for (int q = 1; q < 4; ++q) {
                t0 = fma(s.wz[q], v[3 * q], t0);
                t1 = fma(s.wz[q], v[3 * q + 1], t1);
                t2 = fma(s.wz[q], v[3 * q + 2], t2);
            }
            u0 = fma(s.wy[j], t0, u0);
            u1 = fma(s.wys[j], t1, u1);
            u2 = fma(s.wy[j], t2, u2);
        }
        s0 = fma(s.wxs[i], u0, s0);
        s1 = fma(s.wx[i], u1, s1);
        s2 = fma(s.wx[i], u2, s2);
    }
    Dx = s0;
    Dy = s1;
    Dz = s2;
}

// The same contraction reading the LDS window: (x, y) of the four z nodes as
// aligned 16-byte pairs, and the z components of six nodes from the even
// start a = iz0 & ~1 as three aligned 16-byte pairs (an 8-byte-aligned pair
// read costs ~2.8x an aligned one in LDS, probed).  wz5 carries the four
// weights at the nodes' places and 0 at the extra one, so each FMA chain is
// the four-node chain (a zero-weight term adds a signed zero at most).
template <class Load>
__device__ __forceinline__ void t3_contract_win(const T3Stencil &s, const double wz5[5], Load load, double &Dx,
                                                double &Dy, double &Dz) {
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        double u0 = 0.0, u1 = 0.0, u2 = 0.0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            double vxy[8], vz[6];
            load(i, j, vxy, vz);
            double t0 = s.wz[0] * vxy[0], t1 = s.wz[0] * vxy[1], t2 = wz5[0] * vz[0];
#pragma unroll
            for (int q = 1; q < 4; ++q) {
                t0 = fma(s.wz[q], vxy[2 * q], t0);
                t1 = fma(s.wz[q], vxy[2 * q + 1], t1);
            }
#pragma unroll
            for (int q = 1; q < 5; ++q) t2 = fma(wz5[q], vz[q], t2);
            u0 = fma(s.wy[j], t0, u0);
            u1 = fma(s.wys[j], t1, u1);
            u2 = fma(s.wy[j], t2, u2);
        }
        s0 = fma(s.wxs[i], u0, s0);
        s1 = fma(s.wx[i], u1, s1);
        s2 = fma(s.wx[i], u2, s2);
    }
    Dx = s0;
    Dy = s1;
    Dz = s2;
}

// Twelve contiguous doubles (a z run of the device layout) as six 16-byte loads.
__device__ __forceinline__ void t3_load_aos(const double *p, double *v) {
    const double2u *r = (const double2u *)p;
#pragma unroll
    for (int h = 0; h < 6; ++h) {
        const double2u a = r[h];
        v[2 * h] = a.x;
        v[2 * h + 1] = a.y;
    }
}

__device__ __forceinline__ void t3_interp(const double *__restrict__ T, const KScalars &k, double dx,
                                          double dy, double dz, double &Dx, double &Dy, double &Dz) {
    T3Stencil s;
    t3_stencil(k, dx, dy, dz, s);
    const unsigned NY = (unsigned)(k.ng - k.t3_lo), NZ = (unsigned)(k.ng + 3);
    // z node iz0-1+q sits at layout index iz0+q (one ghost below)
    t3_contract(
        s, [&](int i, int j, double *v) { t3_load_aos(T + ((s.mx[i] * NY + s.my[j]) * NZ + (unsigned)s.iz0) * 3u, v); },
        Dx, Dy, Dz);
}

// S1R2 table in the device layout of s1r2_device_layout: one row per rho
// node -1 .. Nrho (the ghost rows repeat the edge nodes, which is the
// reference's clamp of the rho index), each row the z nodes -1 .. Nz + 1
// (periodic ghosts), each node (D_rho, D_z) as 16 bytes.  Node (ir, iz) sits
// at ((ir + 1) * (Nz + 3) + iz + 1) * 16 bytes; s1r2_row(T, k, ir) + iz + 1
// points at it.
// Row offsets use the full-rate 24-bit multiply (v_mul_u32_u24; the 32-bit
// v_mul_lo_u32 issues at a quarter of the rate): make_plan keeps Nrho + 2 and
// Nz + 3 below 2^24, and the 2^28-node cap keeps the products in 32 bits.
__device__ __forceinline__ const double2 *s1r2_row(const double *__restrict__ T, const KScalars &k, int ir) {
    return (const double2 *)((const char *)T + __umul24((unsigned)(ir + 1), (unsigned)(k.nz + 3)) * 16u);
}

// A z index in [lo_ok, hi_ok] needs no wrap (the ghost rows cover it); any
// other value (a position outside the box) takes the general periodic
// remainder, so every read stays inside the table.
__device__ __forceinline__ int s1r2_zfix(int iz, int lo_ok, int hi_ok, int Nz) {
    if (iz < lo_ok || iz > hi_ok) iz = imodp(iz, Nz);
    return iz;
}

// forces_cuda.cu:188-455: NGP / CIC / TSC interpolation of (D_rho, D_z) at
// (rho, z), rho clamped to [0, rho_max], z periodic.  Returns q = D_rho / rho
// (0 on the axis) and D_z: the caller forms D_x = q dx, D_y = q dy.
// Divisions by the grid spacings become multiplications by their reciprocals
// and rho, 1/rho come from one reciprocal square root (each within an ulp or
// two of the reference's sqrt and divides; the interpolants are continuous).
// The interpolation split into its index math and a gather over rho rows:
// row(ir) returns the z run of rho node ir (device layout: z nodes -1 .. Nz+1),
// from the global table or from an LDS window of rows; s1r2_rows gives the
// rho nodes [lo, hi] a pair's stencil reads.
template <int ORDER>
__device__ __forceinline__ void s1r2_rows(const KScalars &k, double rho, int &lo, int &hi) {
    if (ORDER == 0) {
        lo = hi = (int)floor(fmin(rho, k.rho_max) * k.inv_drho + 0.5);
    } else if (ORDER == 2) {
        lo = (int)floor(fmin(rho * k.inv_drho, k.last_r));
        hi = lo + 1;
    } else {
        const int jr = (int)floor(fmin(rho * k.inv_drho, k.last_r) + 0.5);
        lo = jr - 1;
        hi = jr + 1;
    }
}

template <int ORDER, class Row>
__device__ __forceinline__ void s1r2_gather(Row row, const KScalars &k, double rho, double uz, double &Dr,
                                            double &Dzv) {
    const int Nz = k.nz;
    if (ORDER == 0) {
        const int ir = (int)floor(fmin(rho, k.rho_max) * k.inv_drho + 0.5);  // in [0, Nrho-1]
        const int iz = s1r2_zfix((int)floor(uz + 0.5), 0, Nz, Nz);
        const double2 t = row(ir)[iz + 1];
        Dr = t.x;
        Dzv = t.y;
    } else if (ORDER == 2) {
        // rho beyond rho_max clamps to the last node (forces_cuda.cu:225-239);
        // at ur = Nrho-1 the upper node is the ghost copy of the last one
        const double ur = fmin(rho * k.inv_drho, k.last_r);
        const double urf = floor(ur);
        const double fr = ur - urf;
        const int ir0 = (int)urf;
        const double uzf = floor(uz);
        const double fz = uz - uzf;
        const int iz0 = s1r2_zfix((int)uzf, -1, Nz - 1, Nz);
        const double2 *r0 = row(ir0) + (iz0 + 1);  // z nodes iz0, iz0 + 1
        const double2 *r1 = row(ir0 + 1) + (iz0 + 1);
        const double2 t00 = r0[0], t01 = r0[1], t10 = r1[0], t11 = r1[1];
        // bilinear as two lerps in rho and one in z (same interpolant as the
        // reference's four weights, fewer operations)
        const double a0 = fma(fr, t10.x - t00.x, t00.x), b0 = fma(fr, t11.x - t01.x, t01.x);
        const double a1 = fma(fr, t10.y - t00.y, t00.y), b1 = fma(fr, t11.y - t01.y, t01.y);
        Dr = fma(fz, b0 - a0, a0);
        Dzv = fma(fz, b1 - a1, a1);
    } else {
        const double ur = fmin(rho * k.inv_drho, k.last_r);
        const double urf = floor(ur + 0.5), uzf = floor(uz + 0.5);
        const int jr = (int)urf;  // in [0, Nrho-1]; nodes jr-1 .. jr+1 (ghosts at the ends)
        const int jz = s1r2_zfix((int)uzf, 0, Nz, Nz);
        const double sr = ur - urf, sz = uz - uzf;
        const double wr[3] = {0.5 * (0.5 - sr) * (0.5 - sr), 0.75 - sr * sr,
                              0.5 * (0.5 + sr) * (0.5 + sr)};
        const double wz[3] = {0.5 * (0.5 - sz) * (0.5 - sz), 0.75 - sz * sz,
                              0.5 * (0.5 + sz) * (0.5 + sz)};
        Dr = 0.0;
        Dzv = 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double2 *rr = row(jr - 1 + c) + jz;  // rho node jr-1+c, z nodes jz-1 .. jz+1
            const double w0 = wr[c] * wz[0], w1 = wr[c] * wz[1], w2 = wr[c] * wz[2];
            const double2 a = rr[0], b = rr[1], d = rr[2];
            Dr += w0 * a.x + w1 * b.x + w2 * d.x;
            Dzv += w0 * a.y + w1 * b.y + w2 * d.y;
        }
    }
}

// rho = |(dx, dy)|, its reciprocal, and the z grid coordinate of dz.
__device__ __forceinline__ void s1r2_coords(const KScalars &k, double dx, double dy, double dz, double &rho,
                                            double &inv_rho, double &uz) {
    const double rxy2 = fma(dx, dx, dy * dy);
    inv_rho = (rxy2 > 0.0) ? rsqrt_f64(rxy2) : 0.0;
    rho = rxy2 * inv_rho;
    uz = fma(dz + k.halfL, k.inv_dzg, -0.5);
}

template <int ORDER>
__device__ __forceinline__ void s1r2_interp(const double *__restrict__ T, const KScalars &k, double dx, double dy,
                                            double dz, double &q, double &Dz) {
    double rho, inv_rho, uz, Dr, Dzv;
    s1r2_coords(k, dx, dy, dz, rho, inv_rho, uz);
    s1r2_gather<ORDER>([&](int ir) { return s1r2_row(T, k, ir); }, k, rho, uz, Dr, Dzv);
    q = Dr * inv_rho;
    Dz = Dzv;
}

// An LDS copy of the S1R2 table rows for rho nodes w0 .. w0 + nw - 1 (each
// the full z run of the device layout), valid when ok.
struct S1R2Win {
    const double2 *win;
    int w0, nw;
    bool ok;
};

// s1r2_interp reading the rho rows from the window when they all lie in it,
// else from the global table (the same values either way).
template <int ORDER>
__device__ __forceinline__ void s1r2_interp_win(const double *__restrict__ T, const KScalars &k, double dx, double dy,
                                                double dz, double &q, double &Dz, const S1R2Win sw) {
    double rho, inv_rho, uz, Dr, Dzv;
    s1r2_coords(k, dx, dy, dz, rho, inv_rho, uz);
    bool in = false;
    if (sw.ok) {
        int lo, hi;
        s1r2_rows<ORDER>(k, rho, lo, hi);
        in = lo >= sw.w0 && hi < sw.w0 + sw.nw;
    }
    if (in) {
        const unsigned nz3 = (unsigned)(k.nz + 3);
        s1r2_gather<ORDER>([&](int ir) { return sw.win + __umul24((unsigned)(ir - sw.w0), nz3); }, k, rho, uz, Dr,
                           Dzv);
    } else {
        s1r2_gather<ORDER>([&](int ir) { return s1r2_row(T, k, ir); }, k, rho, uz, Dr, Dzv);
    }
    q = Dr * inv_rho;
    Dz = Dzv;
}

// Softened coefficient for a pair, with the tile bound B = (h_i + h_max,tile)^2:
// only pairs with r2 < B can be inside h_i + h_j, so the exact test (and the
// softening_exact evaluation) runs in a branch that almost no wave takes.
__device__ __forceinline__ double pair_w_tile(double r2, double B, double hi,
                                              const double *__restrict__ soft, int64_t j,
                                              const KScalars &k) {
    double w = inv_r3(r2, k.c15);
    if (r2 < B) {
        const double beta = hi + soft[j];
        if (r2 < beta * beta) w = softening_exact(sqrt(r2), beta);
    }
    return w;
}

// pair_w_tile times the source mass, for a source carrying mp = -1.5 m.
__device__ __forceinline__ double pair_s_tile(double r2, double B, double hi, double mp,
                                              const double *__restrict__ soft, int64_t j, const KScalars &k) {
    double s = mr3_scaled(r2, mp, k.cm53);
    if (r2 < B) {
        const double beta = hi + soft[j];
        if (r2 < beta * beta) s = unscaled_mass(mp) * softening_exact(sqrt(r2), beta);
    }
    return s;
}

// One pair (i = lane row, j = uniform source) for variant V, FP64.  WIN: an
// S1R2 lookup pair reads its rho rows from the window when they all lie in
// it, else from the global table (the same values either way).  MS: the
// source record carries -1.5 m instead of m (R3 and nearest-image variants;
// the FP64 kernel's source copies, mr3_scaled).
// One nearest-image wrap, d - L sign(d) when |d| > L/2 (forces_cuda.cu:
// 622-627, 833-836; positions in [0, L) need no second one), as a multiply
// by 0 or 1 in the FMA rather than two 64-bit selects: fma(-1, c, d) is the
// subtraction d - c, fma(-0, c, d) is d.
__device__ __forceinline__ double wrap_half(double d, const KScalars &k) {
    return fma(fabs(d) > k.halfL ? -1.0 : 0.0, copysign(k.L, d), d);
}

template <int V, bool WIN = false, bool MS = false>
__device__ __forceinline__ void pair_f64(const KScalars &k, const double *__restrict__ table,
                                         const double *__restrict__ soft, const int64_t j,
                                         const double4 pj, const double xi, const double yi,
                                         const double zi, const double hi, const double B,
                                         double &fx, double &fy, double &fz, const S1R2Win sw = S1R2Win{}) {
    double dx = pj.x - xi, dy = pj.y - yi, dz = pj.z - zi;
    if (V == PV_R3) {
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        const double s = MS ? pair_s_tile(r2, B, hi, pj.w, soft, j, k) : pj.w * pair_w_tile(r2, B, hi, soft, j, k);
        fx = fma(s, dx, fx);
        fy = fma(s, dy, fy);
        fz = fma(s, dz, fz);
    } else if (V == PV_T3_NEAREST || V == PV_T3_EWALD) {
        // forces_cuda.cu:622-627: d - L*d/|d| when |d| > L/2 (d/|d| is exactly +-1)
        dx = wrap_half(dx, k);
        dy = wrap_half(dy, k);
        dz = wrap_half(dz, k);
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        if (V == PV_T3_NEAREST) {
            const double s = MS ? pair_s_tile(r2, B, hi, pj.w, soft, j, k) : pj.w * pair_w_tile(r2, B, hi, soft, j, k);
            fx = fma(s, dx, fx);
            fy = fma(s, dy, fy);
            fz = fma(s, dz, fz);
        } else {
            const double w = pair_w_tile(r2, B, hi, soft, j, k);
            double Dx, Dy, Dz;
            t3_interp(table, k, dx, dy, dz, Dx, Dy, Dz);
            fx = fma(pj.w, fma(w, dx, -Dx), fx);
            fy = fma(pj.w, fma(w, dy, -Dy), fy);
            fz = fma(pj.w, fma(w, dz, -Dz), fz);
        }
    } else if (V == PV_S1R2_IMAGES) {
        // forces_cuda.cu:723-737: raw dz, images m in [-(P+1), P+1], cut |dz+mL| < (P+0.6)L
        const double rxy2 = fma(dx, dx, dy * dy);
        double sx = 0.0, sz = 0.0;
        for (int m = -k.images; m <= k.images; ++m) {
            const double dze = dz + (double)m * k.L;
            if (fabs(dze) < k.image_cut) {
                const double r2 = fma(dze, dze, rxy2);
                const double s = pj.w * pair_w_tile(r2, B, hi, soft, j, k);
                sx += s;
                sz = fma(s, dze, sz);
            }
        }
        fx = fma(sx, dx, fx);
        fy = fma(sx, dy, fy);
        fz += sz;
    } else {
        // forces_cuda.cu:833-836: nearest z-image only
        dz = wrap_half(dz, k);
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        if (V == PV_S1R2_NEAREST) {
            const double s = MS ? pair_s_tile(r2, B, hi, pj.w, soft, j, k) : pj.w * pair_w_tile(r2, B, hi, soft, j, k);
            fx = fma(s, dx, fx);
            fy = fma(s, dy, fy);
            fz = fma(s, dz, fz);
        } else {
            const double w = pair_w_tile(r2, B, hi, soft, j, k);
            // m (w d - D) with D_x = q dx, D_y = q dy: x and y share m (w - q)
            constexpr int ORD = (V == PV_S1R2_NGP) ? 0 : ((V == PV_S1R2_CIC) ? 2 : 4);
            double q, Dz;
            s1r2_interp_win<ORD>(table, k, dx, dy, dz, q, Dz, WIN ? sw : S1R2Win{});
            const double sxy = pj.w * (w - q);
            fx = fma(sxy, dx, fx);
            fy = fma(sxy, dy, fy);
            fz = fma(pj.w, fma(w, dz, -Dz), fz);
        }
    }
}

// ---------------------------------------------------------------------------
// FP64 pair kernel: sources in tiles of kTile (64); per tile each lane forms
// B = (h_i + h_max,tile)^2 once, then UNR sources at a time come in through
// scalar loads and are applied to the NI rows of the lane.
// ---------------------------------------------------------------------------
// R3 pair of a tile that no row of the wave can reach within its softening
// bound: the plain r^-3 law, no per-pair test (pj.w = -1.5 m).
__device__ __forceinline__ void pair_r3_far(const KScalars &k, const double4 pj, const double xi, const double yi,
                                            const double zi, double &fx, double &fy, double &fz) {
    const double dx = pj.x - xi, dy = pj.y - yi, dz = pj.z - zi;
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    const double s = mr3_scaled(r2, pj.w, k.cm53);
    fx = fma(s, dx, fx);
    fy = fma(s, dy, fy);
    fz = fma(s, dz, fz);
}

// The nearest-image test (|d| > L/2 -> d -/+ L, forces_cuda.cu:622-627 and
// :833-836) for every source of a tile at once: the displacements from x to
// the tile (centre c, half extent e on this axis) lie in [c - e - x, c + e - x].
// All inside (-L/2, L/2): shift 0; all above L/2: every one wraps to d - L,
// shift -L; all below -L/2: shift +L (margins of rel * L/2 cover the rounding
// of the displacements: 1e-12 for FP64 ones, 1e-5 for FP32 ones).  False when
// the tile straddles a wrap.  d + shift is the reference's d -/+ L to the bit.
__device__ __forceinline__ bool tile_shift(double x, double c, double e, const KScalars &k, double &s,
                                           double rel = 1e-12) {
    const double m = k.halfL * rel;
    s = 0.0;
    if (fabs(x - c) + e < k.halfL - m) return true;
    if (c - e - x > k.halfL + m) {
        s = -k.L;
        return true;
    }
    if (c + e - x < -k.halfL - m) {
        s = k.L;
        return true;
    }
    return false;
}

// x moved by a period towards c when it lies more than half a period away
// (positions inside the box need at most one step).
__device__ __forceinline__ double near_image(double x, double c, const KScalars &k) {
    const double d = x - c;
    return (d > k.halfL) ? x - k.L : ((d < -k.halfL) ? x + k.L : x);
}

// The R3 pair of a far tile with per-axis nearest-image shifts.
__device__ __forceinline__ void pair_far_shift(const KScalars &k, const double4 pj, const double xi, const double yi,
                                               const double zi, const double sx, const double sy, const double sz,
                                               double &fx, double &fy, double &fz) {
    const double dx = (pj.x - xi) + sx, dy = (pj.y - yi) + sy, dz = (pj.z - zi) + sz;
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    const double s = mr3_scaled(r2, pj.w, k.cm53);  // pj.w = -1.5 m
    fx = fma(s, dx, fx);
    fy = fma(s, dy, fy);
    fz = fma(s, dz, fz);
}

// Squared distance from a point to an axis-aligned box (centre c, half
// extents e); every source of the tile is at least this far from the point.
__device__ __forceinline__ double box_dist2(double x, double y, double z, const double4 &c, const double4 &e) {
    const double gx = fmax(fabs(x - c.x) - e.x, 0.0);
    const double gy = fmax(fabs(y - c.y) - e.y, 0.0);
    const double gz = fmax(fabs(z - c.z) - e.z, 0.0);
    return fma(gx, gx, fma(gy, gy, gz * gz));
}

__device__ __forceinline__ void mixed_pair(const float4 pj, const float xr, const float yr,
                                           const float zr, const float B, bool &near, float &ax,
                                           float &ay, float &az) {
    const float dx = pj.x - xr, dy = pj.y - yr, dz = pj.z - zr;
    const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
    const float y = __builtin_amdgcn_rsqf(r2);
    const float s = (y * y) * (y * pj.w);
    if (r2 < B) {
        near = true;
    } else {
        ax = fmaf(s, dx, ax);
        ay = fmaf(s, dy, ay);
        az = fmaf(s, dz, az);
    }
}

constexpr int s1r2_order(int V) { return V == PV_S1R2_CIC ? 2 : 4; }

// FP32 copy of the device layout (s1r2_row): same rows, 8-byte nodes.
__device__ __forceinline__ const float2 *s1r2_row32(const float2 *__restrict__ T, const KScalars &k, int ir) {
    return (const float2 *)((const char *)T + __umul24((unsigned)(ir + 1), (unsigned)(k.nz + 3)) * 8u);
}

// s1r2_interp in FP32 (CIC, TSC): returns q = D_rho / rho and D_z.
// An LDS copy of the FP32 S1R2 table rows for rho nodes w0 .. w0 + nw - 1.
struct S1R2Win32 {
    const float2 *win;
    int w0, nw;
    bool ok;
};

// WIN: the rows come from the window when the stencil's rho nodes all lie in
// it, else from the global table (the same values either way).
template <int ORDER, bool WIN = false>
__device__ __forceinline__ void s1r2_interp_f32(const float2 *__restrict__ T, const KScalars &k, float dx,
                                                float dy, float dz, float &q, float &Dz,
                                                const S1R2Win32 sw = S1R2Win32{}) {
    const int Nz = k.nz;
    const float rxy2 = fmaf(dx, dx, dy * dy);
    const float inv_rho = (rxy2 > 0.0f) ? __builtin_amdgcn_rsqf(rxy2) : 0.0f;
    const float rho = rxy2 * inv_rho;
    const float uz = fmaf(dz + k.halfLf, k.inv_dzgf, -0.5f);
    const float lastr = k.last_rf;
    float Dr, Dzv;
    static_assert(ORDER == 2 || ORDER == 4, "FP32 interpolation is CIC or TSC");
    auto gather = [&](auto rowf) {
    if (ORDER == 2) {
        const float ur = fminf(rho * k.inv_drhof, lastr);
        const float urf = floorf(ur);
        const float fr = ur - urf;
        const int ir0 = (int)urf;
        const float uzf = floorf(uz);
        const float fz = uz - uzf;
        const int iz0 = s1r2_zfix((int)uzf, -1, Nz - 1, Nz);
        const float2 *r0 = rowf(ir0) + (iz0 + 1);
        const float2 *r1 = rowf(ir0 + 1) + (iz0 + 1);
        const float2 t00 = r0[0], t01 = r0[1], t10 = r1[0], t11 = r1[1];
        const float a0 = fmaf(fr, t10.x - t00.x, t00.x), b0 = fmaf(fr, t11.x - t01.x, t01.x);
        const float a1 = fmaf(fr, t10.y - t00.y, t00.y), b1 = fmaf(fr, t11.y - t01.y, t01.y);
        Dr = fmaf(fz, b0 - a0, a0);
        Dzv = fmaf(fz, b1 - a1, a1);
    } else {
        const float ur = fminf(rho * k.inv_drhof, lastr);
        const float urf = floorf(ur + 0.5f), uzf = floorf(uz + 0.5f);
        const int jr = (int)urf;
        const int jz = s1r2_zfix((int)uzf, 0, Nz, Nz);
        const float sr = ur - urf, sz = uz - uzf;
        const float wr[3] = {0.5f * (0.5f - sr) * (0.5f - sr), 0.75f - sr * sr, 0.5f * (0.5f + sr) * (0.5f + sr)};
        const float wz[3] = {0.5f * (0.5f - sz) * (0.5f - sz), 0.75f - sz * sz, 0.5f * (0.5f + sz) * (0.5f + sz)};
        Dr = 0.0f;
        Dzv = 0.0f;
#pragma unroll
        for (int row = 0; row < 3; ++row)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float2 t = rowf(jr - 1 + c)[jz + row];
                const float w = wr[c] * wz[row];
                Dr = fmaf(w, t.x, Dr);
                Dzv = fmaf(w, t.y, Dzv);
            }
    }
    };
    bool in = false;
    if (WIN && sw.ok) {
        const float ur = fminf(rho * k.inv_drhof, lastr);
        const int lo = (ORDER == 2) ? (int)floorf(ur) : (int)floorf(ur + 0.5f) - 1;
        in = lo >= sw.w0 && lo + (ORDER == 2 ? 1 : 2) < sw.w0 + sw.nw;
    }
    if (in) {
        const unsigned nz3 = (unsigned)(k.nz + 3);
        gather([&](int ir) { return sw.win + __umul24((unsigned)(ir - sw.w0), nz3); });
    } else {
        gather([&](int ir) { return s1r2_row32(T, k, ir); });
    }
    q = Dr * inv_rho;
    Dz = Dzv;
}

// FP32 displacement with the nearest z-image (forces_cuda.cu:833-836) and r^2;
// T3 nearest image: the nearest image on every axis (forces_cuda.cu:622-627).
// bnd: a wrapped axis lies within 1e-6 L of L/2, where the FP32 displacement
// (off by a few ulp of L) may take the other image than the FP64 one: such a
// pair is left to the FP64 redo with the close pairs, so every pair takes the
// reference's image.  (On the S1R2 N = 524288 cylinder about 4% of the rows
// had one pair in that band, whose flipped image set the p99 error.)
template <int V>
__device__ __forceinline__ float mixed_r2_z(const KScalars &k, const float4 pj, float xr, float yr, float zr,
                                            float &dx, float &dy, float &dz, bool &bnd) {
    dx = pj.x - xr;
    dy = pj.y - yr;
    dz = pj.z - zr;
    bnd = fabsf(fabsf(dz) - k.halfLf) < k.wrap_epsf;
    if (V == PV_T3_NEAREST)
        bnd = bnd || fabsf(fabsf(dx) - k.halfLf) < k.wrap_epsf || fabsf(fabsf(dy) - k.halfLf) < k.wrap_epsf;
    if (V == PV_T3_NEAREST) {
        if (dx > k.halfLf) dx -= k.Lf;
        else if (dx < -k.halfLf) dx += k.Lf;
        if (dy > k.halfLf) dy -= k.Lf;
        else if (dy < -k.halfLf) dy += k.Lf;
    }
    if (dz > k.halfLf) dz -= k.Lf;
    else if (dz < -k.halfLf) dz += k.Lf;
    return fmaf(dx, dx, fmaf(dy, dy, dz * dz));
}

template <int V, bool WIN = false>
__device__ __forceinline__ void mixed_pair_z(const KScalars &k, const float2 *__restrict__ T, const float4 pj,
                                             float xr, float yr, float zr, float B, bool &near, float &ax,
                                             float &ay, float &az, const S1R2Win32 sw = S1R2Win32{}) {
    float dx, dy, dz;
    bool bnd;
    const float r2 = mixed_r2_z<V>(k, pj, xr, yr, zr, dx, dy, dz, bnd);
    const bool nr = r2 < B || bnd;  // left to the FP64 redo (r2 may be 0 here)
    near = near || nr;
    const float y = __builtin_amdgcn_rsqf(r2);
    const float y3 = nr ? 0.0f : (y * y) * y;
    const float m = nr ? 0.0f : pj.w;
    if (V == PV_S1R2_NEAREST || V == PV_T3_NEAREST) {
        const float s = y3 * m;
        ax = fmaf(s, dx, ax);
        ay = fmaf(s, dy, ay);
        az = fmaf(s, dz, az);
    } else {
        float q, Dz;
        s1r2_interp_f32<s1r2_order(V), WIN>(T, k, dx, dy, dz, q, Dz, sw);
        const float sxy = m * (y3 - q);
        ax = fmaf(sxy, dx, ax);
        ay = fmaf(sxy, dy, ay);
        az = fmaf(m, fmaf(y3, dz, -Dz), az);
    }
}

// FP32 pairs of a far tile (no pair within the softening bound, no straddled
// wrap) with the nearest image (z only for S1R2, every axis for T3):
// mixed_pair_z's arithmetic without the per-pair wrap and bound tests, the
// wrap applied as a per-lane shift.  With FLUSH the FP32 sums are added to
// the FP64 accumulators f* after every UNR sources: on the T3 nearest-image
// lattice at 64^3 this took the p99 error against FP64 from 1.09e-5 to
// 9.7e-6 for 1% of the speed (on the S1R2 cylinder it changed nothing there
// and cost 4%, so S1R2 keeps one FP32 sum per tile).
template <bool SHIFT, bool XY, bool FLUSH, int NI, int UNR>
__device__ __forceinline__ void mixed_far_tile_z(const float4 *__restrict__ tr, const int cnt, const float *xr,
                                                 const float *yr, const float *zr, const float *sx,
                                                 const float *sy, const float *sz, float *ax, float *ay,
                                                 float *az, double *fx, double *fy, double *fz) {
    auto pair = [&](const float4 pj, const int q) {
        const float dx = (SHIFT && XY) ? (pj.x - xr[q]) + sx[q] : pj.x - xr[q];
        const float dy = (SHIFT && XY) ? (pj.y - yr[q]) + sy[q] : pj.y - yr[q];
        const float dz = SHIFT ? (pj.z - zr[q]) + sz[q] : pj.z - zr[q];
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        const float y = __builtin_amdgcn_rsqf(r2);
        const float s = ((y * y) * y) * pj.w;
        ax[q] = fmaf(s, dx, ax[q]);
        ay[q] = fmaf(s, dy, ay[q]);
        az[q] = fmaf(s, dz, az[q]);
    };
    int j = 0;
    for (; j + UNR <= cnt; j += UNR) {
        float4 pj[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) pj[u] = tr[j + u];
#pragma unroll
        for (int u = 0; u < UNR; ++u)
#pragma unroll
            for (int q = 0; q < NI; ++q) pair(pj[u], q);
        if (FLUSH) {
#pragma unroll
            for (int q = 0; q < NI; ++q) {
                fx[q] += (double)ax[q];
                fy[q] += (double)ay[q];
                fz[q] += (double)az[q];
                ax[q] = ay[q] = az[q] = 0.0f;
            }
        }
    }
    for (; j < cnt; ++j) {
        const float4 pj = tr[j];
#pragma unroll
        for (int q = 0; q < NI; ++q) pair(pj, q);
    }
}

// A window row holds the (x, y) components of its NZ z nodes as 16-byte pairs
// (2 NZ doubles), then their z components (NZ doubles and two zeros, so that
// six nodes from an even start stay inside); rows start on 16-byte
// boundaries.  A stencil row is then seven aligned 16-byte reads
// (t3_contract_win).  Earlier forms: four aligned reads for (x, y) and two
// 8-byte-aligned pair reads for z, 30.2 G pairs/s.  Measured at 64^3 (row-major
// pencils): node-major rows (24 bytes a node, six unaligned pair reads) 21.3
// G pairs/s, with bank-conflict stalls on 57% of LDS cycles; three component
// runs, 20.9; this layout, 26.7.  Rows padded to 256 bytes (so that a change
// of row keeps the bank pattern) fit fewer windows: 27.9 against 30.2 with
// serpentine pencils, and on the current kernel 30.3 against 34.4 (rows at
// odd multiples of 128 bytes: 32.4).
__host__ __device__ constexpr unsigned t3_win_stride(unsigned nz3) { return (nz3 + 1u) & ~1u; }

// Layout nodes one axis of the window needs: sources in cell columns
// [smin, smax], rows in columns [bmin, bmax].  d / h lies in (s - b - 1,
// s - b + 1) (mod Ng), so the stencils' unfolded nodes lie in
// [smin - bmax + (Ng-1)/2 - 2, smax - bmin + Ng/2 + 2] (mod Ng); their images
// in the folded layout are a contiguous range [f0, f0 + nf).  False when the
// range is too wide to be one.
__device__ __forceinline__ bool t3_win_axis(int smin, int smax, int bmin, int bmax, int Ng, int lo, int &f0,
                                            int &nf) {
    const int nlo = (smin - bmax) + (Ng - 1) / 2 - 2;
    const int nhi = (smax - bmin) + Ng / 2 + 2;
    if (nhi - nlo >= Ng / 2) return false;
    int mn = Ng, mxv = -1;
    for (int n = nlo; n <= nhi; ++n) {
        const int jj = imodp(n, Ng);
        const int m = (jj >= lo) ? jj - lo : Ng - 1 - lo - jj;
        mn = min(mn, m);
        mxv = max(mxv, m);
    }
    f0 = mn;
    nf = mxv - mn + 1;
    return true;
}

// Cell column y of a pencil key (order_kernels.hip reverses y in odd x columns).
__device__ __forceinline__ int pencil_y(uint32_t key, int Ng) {
    const int by = (int)((key >> 10) & 1023u);
    return ((key >> 20) & 1u) ? Ng - 1 - by : by;
}

struct T3Stencil32 {
    float wx[4], wy[4], wz[4], wxs[4], wys[4];
    unsigned mx[4], my[4];
    int iz0;
};

// t3_axis in FP32 (forces_cuda.cu:93-111).
__device__ __forceinline__ int t3_axis_f32(float d, const KScalars &k, float w[4]) {
    const float u = (d + k.halfLf) * k.inv_gsf - 0.5f;
    const float uf = floorf(u);
    const float t = u - uf;
    const float t2 = t * t, t3 = t * t2;
    w[0] = -0.5f * t3 + t2 - 0.5f * t;
    w[1] = 1.5f * t3 - 2.5f * t2 + 1.0f;
    w[2] = -1.5f * t3 + 2.0f * t2 + 0.5f * t;
    w[3] = 0.5f * t3 - 0.5f * t2;
    return wrap_index((int)uf, k.ng);
}

__device__ __forceinline__ void t3_stencil_f32(const KScalars &k, float dx, float dy, float dz, T3Stencil32 &s) {
    const int Ng = k.ng, lo = k.t3_lo;
    const int ix0 = t3_axis_f32(dx, k, s.wx);
    const int iy0 = t3_axis_f32(dy, k, s.wy);
    s.iz0 = t3_axis_f32(dz, k, s.wz);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int jx = wrap_once(ix0 - 1 + q, Ng);
        const int jy = wrap_once(iy0 - 1 + q, Ng);
        s.mx[q] = (unsigned)((jx >= lo) ? jx - lo : Ng - 1 - lo - jx);
        s.my[q] = (unsigned)((jy >= lo) ? jy - lo : Ng - 1 - lo - jy);
        s.wxs[q] = (jx >= lo) ? s.wx[q] : -s.wx[q];
        s.wys[q] = (jy >= lo) ? s.wy[q] : -s.wy[q];
    }
}

// t3_contract in FP32 over 16-byte nodes: load(i, j, n) fills n[q] with z
// node iz0 - 1 + q of table row (mx[i], my[j]).
template <class Load>
__device__ __forceinline__ void t3_contract_f32(const T3Stencil32 &s, Load load, float &Dx, float &Dy, float &Dz) {
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float u0 = 0.0f, u1 = 0.0f, u2 = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float4 n[4];
            load(i, j, n);
            float t0 = s.wz[0] * n[0].x, t1 = s.wz[0] * n[0].y, t2 = s.wz[0] * n[0].z;
#pragma unroll
            for (int q = 1; q < 4; ++q) {
                t0 = fmaf(s.wz[q], n[q].x, t0);
                t1 = fmaf(s.wz[q], n[q].y, t1);
                t2 = fmaf(s.wz[q], n[q].z, t2);
            }
            u0 = fmaf(s.wy[j], t0, u0);
            u1 = fmaf(s.wys[j], t1, u1);
            u2 = fmaf(s.wy[j], t2, u2);
        }
        s0 = fmaf(s.wxs[i], u0, s0);
        s1 = fmaf(s.wx[i], u1, s1);
        s2 = fmaf(s.wx[i], u2, s2);
    }
    Dx = s0;
    Dy = s1;
    Dz = s2;
}

// Nearest-image displacement in FP64, rounded to FP32; returns the FP32 r^2.
// The main loop and the FP64 redo both call it, so they take the same
// near-pair decisions.
__device__ __forceinline__ float t3_mixed_disp(const KScalars &k, const double4 &pj, double xi, double yi, double zi,
                                               float &dx, float &dy, float &dz) {
    double ex = pj.x - xi, ey = pj.y - yi, ez = pj.z - zi;
    if (fabs(ex) > k.halfL) ex -= copysign(k.L, ex);
    if (fabs(ey) > k.halfL) ey -= copysign(k.L, ey);
    if (fabs(ez) > k.halfL) ez -= copysign(k.L, ez);
    dx = (float)ex;
    dy = (float)ey;
    dz = (float)ez;
    return fmaf(dx, dx, fmaf(dy, dy, dz * dz));
}

__device__ __forceinline__ double radial_correction(double r, double R, const double *T,
                                                    int size) {
    // forces_cuda.cu:41-70 (linear interpolation; nodes assumed at R/size*i)
    const double step = R / (double)size;
    const int i = (int)floor(r / R * (size - 1));
    double c = T[size - 1];
    if (i < size - 1) {
        const double X1 = step * i, Y1 = T[i], X2 = step * (i + 1), Y2 = T[i + 1];
        const double A = (Y2 - Y1) / (X2 - X1);
        const double B = Y1 - A * X1;
        c = A * r + B;
    }
    return c;
}

// The external term of a row at x (modes of EvalPlan::ext_mode).
__device__ __forceinline__ void add_external(double f[3], const double4 &x, const double *radial, int ext_mode,
                                             double ext_coeff, double Rsim, int radial_size) {
    if (ext_mode == 3) {
        // forces_cuda.cu:698-701: mass_in_unit_sphere * x * correction(r_xy), x and y only
        const double corr = radial_correction(sqrt(x.x * x.x + x.y * x.y), Rsim, radial, radial_size);
        f[0] += ext_coeff * x.x * corr;
        f[1] += ext_coeff * x.y * corr;
    } else if (ext_mode != 0) {
        // forces_cuda.cu:545-556 (mode 1, xyz) and :848-857 (mode 2, xy)
        f[0] += ext_coeff * x.x;
        f[1] += ext_coeff * x.y;
        if (ext_mode == 1) f[2] += ext_coeff * x.z;
    }
}

// The launch scalars of an evaluation.
inline KScalars make_scalars(const EvalPlan &p) {
    KScalars k{};
    k.N = p.N;
    k.id_min = p.id_min;
    k.nrows = p.nrows;
    k.jchunk = p.jchunk;
    k.L = p.L;
    k.halfL = 0.5 * p.L;
    k.ng = p.t3_ng;
    k.t3_lo = p.t3_lo;
    k.nrho = p.s1r2_nrho;
    k.nz = p.s1r2_nz;
    k.rho_max = kRadialExtent * p.Rsim;
    k.images = p.images;
    k.image_cut = (((double)p.images) - 0.4) * p.L;
    k.c15 = 1.5;
    k.cm53 = -5.0 / 3.0;
    k.inv_gs = (p.t3_ng > 0 && p.L > 0) ? 1.0 / (p.L / (double)p.t3_ng) : 0.0;
    const double drho = k.rho_max / (double)std::max(1, p.s1r2_nrho - 1);
    k.inv_drho = (drho > 0.0) ? 1.0 / drho : 0.0;
    k.inv_dzg = (p.s1r2_nz > 0 && p.L > 0) ? 1.0 / (p.L / (double)p.s1r2_nz) : 0.0;
    k.last_r = (double)std::max(1, p.s1r2_nrho - 1);
    k.Lf = (float)p.L;
    k.halfLf = (float)(0.5 * p.L);
    k.wrap_epsf = (float)(1e-6 * p.L);
    k.rho_maxf = (float)k.rho_max;
    k.inv_drhof = (float)k.inv_drho;
    k.inv_dzgf = (float)k.inv_dzg;
    k.last_rf = (float)k.last_r;
    k.inv_gsf = (float)k.inv_gs;
    return k;
}

}  // namespace

}  // namespace steps
