// sym_kernels.hip -- direct pair forces with every unordered pair evaluated
// once (Newton's third law), for evaluations of (nearly) all rows.
//
// The one-sided kernels (pair_kernels.hip) evaluate each pair twice, once per
// row, and run at the VALU issue limit: the only way to less time is less
// arithmetic per interaction.  Displacement, r^2, the reciprocal square root
// and the softening are the same for both sides of a pair, and only the two
// mass products and six accumulations belong to one side, so one evaluation
// for both costs 18 FP64 VALU + one v_rsq_f64 per two interactions instead of
// 14 + 1 per one.  What makes it pay on a wave64 machine is how the second
// side is summed:
//   * a lane holds NI target rows in VGPRs with their FP64 sums; a tile of 64
//     sources is staged in LDS and at step s lane l takes source
//     (l + s) mod 64, so the 64 lanes always hold 64 different sources and
//     each source's partial sum rides along in VGPRs: after every step it
//     moves one lane down (v_mov_b32 with DPP wave_rol:1, six dwords for NI
//     pairs), and after 64 steps it is back in its own lane, complete for
//     the wave's 64*NI rows.  No atomics and no cross-lane reduction;
//   * the four waves of a workgroup take the same tile with their own rows;
//     their four source sums are added through LDS in wave order.
// Blocks of kSymBlock rows are paired cyclically: block b takes the source
// blocks b, b+1 .. b+H (mod S), H = S/2, with the last offset taken by half
// of the blocks when S is even, so every unordered block pair is evaluated
// exactly once and all workgroups do the same work.  A (block, offset) pair's
// source sums go to a slot of their own, [offset][3][N], the row sums of a
// task (a run of tiles) to another, and the reduction adds the slots in a
// fixed order, so two evaluations are bitwise equal.  When the slots of all
// offsets do not fit the scratch, the offsets are done in groups of launches,
// each followed by a reduction onto running sums; the additions and their
// order do not depend on the grouping.
//
// Measured against the one-sided kernels (resident or one-shot calls, copies
// included): R3 N = 16384 KDK runs 1.32 -> 0.98 ms, N = 100003 6.7 -> 4.4 ms,
// N = 10^6 487 -> 373 ms (1.34 T pair evaluations/s, 2.67 T interactions/s;
// the loop alone reaches 1.41); T3 nearest image at 64^3 50.2 -> 29.1 ms.
// Errors against 64-bit sums are smaller (shorter addition chains).  Bound by
// FP64 VALU issue: ~100 of the ~107 cycles a pair evaluation takes per SIMD
// are its 18 FP64 instructions and the quarter-rate v_rsq_f64.
#include "pair_device.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace steps {

namespace {

constexpr int kSymWaves = kBlock / 64;

struct SymArgs {
    const double4 *rec;   // sources and rows: (x, y, z, -1.5 m)
    const double *soft;
    const double4 *tiles;  // per 64 records: bounding-box centre, largest softening length
    const double4 *ext;    // half extents
    const float4 *jrel;    // mixed: FP32 offsets from the tile's centre, and the mass
    const double *table;   // T3 Ewald or S1R2 table, device layout
    const float4 *tab32;   // ... its FP32 copy, 16-byte nodes (mixed precision)
    const float2 *tab32s;  // S1R2: the FP32 copy of the table (mixed precision)
    const uint32_t *keys;  // pencil keys of the records (T3 Ewald)
    double *part;
    KScalars k;
    int blocks, half;      // S and H
    int tb, tpt;           // tiles per block, tiles per task
    int cell_tasks, cell_offs;
    int cell0;             // first cell of this launch
};

// Slot layout of one cell: cell_tasks row-sum slots, then cell_offs
// source-sum slots, each [3][N].
__host__ __device__ inline size_t sym_slot(int64_t n, int cell, int cell_tasks, int cell_offs, int slot) {
    return ((size_t)cell * (size_t)(cell_tasks + cell_offs) + (size_t)slot) * 3u * (size_t)n;
}

// A kernel runs one evaluation per launch (blocks x tasks of the launch's
// cells), or several evaluations packed into one launch (flat grid, each
// workgroup finds its evaluation among at most kMaxPack).  Packed, small
// evaluations share the chip: a server wave of 16 T3 nearest 21^3 1.40 ms (2.36 one
// after another), of 16 S1R2 CIC N = 1536 0.52 (0.85), of 16 T3 Ewald N = 216 1.30
// (3.5).
struct SymSeg {
    SymArgs a;
    int blk_begin;
};
struct SymPack {
    const SymSeg *segs;
    int nseg;
};

__device__ __forceinline__ const SymArgs &sym_this(const SymArgs &in, int &b, unsigned &by) {
    b = blockIdx.x;
    by = blockIdx.y;
    return in;
}
__device__ __forceinline__ SymArgs sym_this(const SymPack &in, int &b, unsigned &by) {
    int s = 0;
    for (int q = 1; q < in.nseg; ++q)
        if (in.segs[q].blk_begin <= (int)blockIdx.x) s = q;
    const SymArgs a = in.segs[s].a;
    const unsigned local = blockIdx.x - (unsigned)in.segs[s].blk_begin;
    b = (int)(local % (unsigned)a.blocks);
    by = local / (unsigned)a.blocks;
    return a;
}

__device__ __forceinline__ double from_next_lane(double v) {
    // lane l receives lane (l + 1) mod 64's value
    union { double d; int i[2]; } u;
    u.d = v;
    u.i[0] = __builtin_amdgcn_update_dpp(u.i[0], u.i[0], 0x134, 0xf, 0xf, false);
    u.i[1] = __builtin_amdgcn_update_dpp(u.i[1], u.i[1], 0x134, 0xf, 0xf, false);
    return u.d;
}

__device__ __forceinline__ float from_next_lane(float v) {
    union { float f; int i; } u;
    u.f = v;
    u.i = __builtin_amdgcn_update_dpp(u.i, u.i, 0x134, 0xf, 0xf, false);
    return u.f;
}

// Walks the tiles of a task: relative tile r counts from the block's own
// first tile (offset r / tb, tile r mod tb of that source block).
struct SymWalk {
    int r, end;
    int tile, off;
    __device__ __forceinline__ bool settle(const SymArgs &a, int b, int ntiles) {
        for (; r < end; ++r) {
            off = r / a.tb;
            if (off > a.half) return false;
            // the last offset of an even number of blocks: half of the blocks
            if (off > 0 && 2 * off == a.blocks && b >= off) {
                r = (off + 1) * a.tb - 1;
                continue;
            }
            int jb = b + off;
            if (jb >= a.blocks) jb -= a.blocks;
            tile = jb * a.tb + (r - off * a.tb);
            if (tile < ntiles) return true;
            r = (off + 1) * a.tb - 1;  // the rest of the (last) source block is empty
        }
        return false;
    }
};

// One pair for both sides: u = -(2/3) r^-3 (mr3_scaled's correction without
// the mass), the row's sum gets m_j r^-3 d, the source's m_i r^-3 d (its sign
// is applied in the reduction).  NEAR: a pair within the bound B is left to
// sym_close_pair (r2 may be 0 here) and reported.  NEAR = 2, a block with
// itself: a pair at r2 <= rskip is not worth reporting (rskip is 0 where the
// row is softened: the self pair's force is 0 then; else negative).
// UNIT: both masses are 1 (the sums are scaled once, at their end).
template <int NEAR, bool UNIT>
__device__ __forceinline__ void sym_pair(const double dx, const double dy, const double dz, const double mi,
                                         const double mj, const double cm53, const double B, const double rskip,
                                         bool &close, double &fx,
                                         double &fy, double &fz, double &gx, double &gy, double &gz) {
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    const double y = __builtin_amdgcn_rsq(r2);
    const double t = y * y;
    double u = (t * y) * fma(r2, t, cm53);
    if (NEAR) {
        const bool c = r2 < B;
        close = close || (NEAR == 2 ? (c && r2 > rskip) : c);
        u = c ? 0.0 : u;
    }
    const double sj = UNIT ? u : u * mj, si = UNIT ? u : u * mi;
    fx = fma(sj, dx, fx);
    fy = fma(sj, dy, fy);
    fz = fma(sj, dz, fz);
    gx = fma(si, dx, gx);
    gy = fma(si, dy, gy);
    gz = fma(si, dz, gz);
}

// A pair within the tile's softening bound, exact test and spline.
__device__ __forceinline__ void sym_close_pair(const double r2, const double dx, const double dy, const double dz,
                                               const double mi, const double mj, const double *__restrict__ soft,
                                               const int64_t i, const int64_t j, const double cm53, double &fx,
                                               double &fy, double &fz, double &gx, double &gy, double &gz) {
    const double beta = soft[i] + soft[j];
    const double y = __builtin_amdgcn_rsq(r2);
    const double t = y * y;
    double u = (t * y) * fma(r2, t, cm53);
    if (r2 < beta * beta) u = softening_exact(sqrt(r2), beta) * (-2.0 / 3.0);
    const double sj = u * mj, si = u * mi;
    fx = fma(sj, dx, fx);
    fy = fma(sj, dy, fy);
    fz = fma(sj, dz, fz);
    gx = fma(si, dx, gx);
    gy = fma(si, dy, gy);
    gz = fma(si, dz, gz);
}

template <int K> struct IntC { static constexpr int value = K; };

// EQ: every particle has the same mass, which then multiplies the finished sums
// instead of each pair (16 FP64 VALU for 18; T3 nearest 64^3 31.1 -> 29.1 ms); in
// between masses are 1, or 0 for rows and sources past the end, whose tiles
// keep the products.
template <int V, int NI, bool EQ, class In>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void sym_kernel(const In in) {
    int b;
    unsigned by;
    const SymArgs &a = sym_this(in, b, by);
    __shared__ __align__(2048) double2 jbuf[2][2][kTile];  // (x, y) and (z, -1.5 m) of the tile's sources
    __shared__ double gsum[2][kSymWaves][3][kTile];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t N = a.k.N;
    const int ntiles = (int)((N + kTile - 1) / kTile);
    const int cell_l = by / a.cell_tasks, task = by % a.cell_tasks;
    const int cell = a.cell0 + cell_l;
    SymWalk w;
    w.r = cell * a.cell_offs * a.tb + task * a.tpt;
    w.end = w.r + a.tpt;

    const int64_t row0 = ((int64_t)b * kSymWaves + wave) * (64 * NI) + lane;
    double x[NI], y[NI], z[NI], m[NI], fx[NI], fy[NI], fz[NI];
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int64_t r = row0 + q * 64;
        const double4 p = a.rec[min(r, N - 1)];
        x[q] = p.x;
        y[q] = p.y;
        z[q] = p.z;
        m[q] = r < N ? (EQ ? 1.0 : p.w) : 0.0;  // rows past the end: the last particle again, without mass
        fx[q] = fy[q] = fz[q] = 0.0;
    }
    const double cm53 = a.k.cm53;
    const double mass = EQ ? a.rec[0].w : 1.0;
    const bool whole = EQ && (int64_t)(b + 1) * (kSymWaves * 64 * NI) <= N;  // no row past the end

    auto stage = [&](int buf, int tile) {  // wave 0: one source per lane
        const int64_t j = (int64_t)tile * kTile + lane;
        const double4 p = a.rec[min(j, N - 1)];
        jbuf[buf][0][lane] = make_double2(p.x, p.y);
        jbuf[buf][1][lane] = make_double2(p.z, j < N ? (EQ ? 1.0 : p.w) : 0.0);
    };
    // source (lane + s) mod 64 of a tile at byte offset o = 16 ((lane + s) mod 64)
    auto source = [&](int buf, unsigned o, double2 &pa, double2 &pb) {
        const char *p = (const char *)&jbuf[buf][0][0] + o;
        pa = *(const double2 *)p;
        pb = *(const double2 *)(p + sizeof(double2) * kTile);
    };
    constexpr unsigned kWrap = sizeof(double2) * kTile - 1;
    bool have = w.settle(a, b, ntiles);
    if (have && wave == 0) stage(0, w.tile);
    __syncthreads();

    for (int it = 0; have; ++it) {
        const int buf = it & 1;
        const int tile = w.tile, off = w.off;
        // the next tile's records, stored to the other buffer after this tile
        SymWalk nw = w;
        ++nw.r;
        const bool more = nw.settle(a, b, ntiles);
        if (more && wave == 0) stage(buf ^ 1, nw.tile);

        const double4 tc = a.tiles[tile], te = a.ext[tile];
        // far: no source of the tile within any row's softening bound (widened
        // by 1e-9 for rounding); wrap: an axis on which some lane sees the
        // tile on both sides of a period wrap.  Other axes take the row's
        // image on the tile's side (tile_shift).
        bool far = true, wx = false, wy = false, wz = false;
        double B = 0.0;  // the largest of the lane's softening bounds
        double rskip = 0.0;
        if (V != PV_R3) {
#pragma unroll
            for (int q = 0; q < NI; ++q) {
                const double4 p = a.rec[min(row0 + q * 64, N - 1)];
                double sh;
                if (V == PV_T3_NEAREST) {
                    wx = !tile_shift(p.x, tc.x, te.x, a.k, sh) || wx;
                    wy = !tile_shift(p.y, tc.y, te.y, a.k, sh) || wy;
                }
                wz = !tile_shift(p.z, tc.z, te.z, a.k, sh) || wz;
            }
            wx = __any(wx);
            wy = __any(wy);
            wz = __any(wz);
        }
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            const int64_t r = min(row0 + q * 64, N - 1);
            if (V != PV_R3) {
                const double4 p = a.rec[r];
                double sx = 0.0, sy = 0.0, sz = 0.0;
                if (!wz) tile_shift(p.z, tc.z, te.z, a.k, sz);
                if (V == PV_T3_NEAREST) {
                    if (!wx) tile_shift(p.x, tc.x, te.x, a.k, sx);
                    if (!wy) tile_shift(p.y, tc.y, te.y, a.k, sy);
                }
                x[q] = p.x - sx;
                y[q] = p.y - sy;
                z[q] = p.z - sz;
            }
            const double h = a.soft[r], bb = h + tc.w;
            if (!(h > 0.0)) rskip = -1.0;
            const double Bq = bb * bb;
            B = fmax(B, Bq);
            // distance to the box over the axes that are on one side
            const double ax = wx ? 0.0 : fmax(fabs(x[q] - tc.x) - te.x, 0.0);
            const double ay = wy ? 0.0 : fmax(fabs(y[q] - tc.y) - te.y, 0.0);
            const double az = wz ? 0.0 : fmax(fabs(z[q] - tc.z) - te.z, 0.0);
            far = far && fma(ax, ax, fma(ay, ay, az * az)) > Bq * (1.0 + 1e-9);
        }
        far = __all(far);

        double gx = 0.0, gy = 0.0, gz = 0.0;
        bool close = false;
        // the 64 steps; WM: axes wrapped per pair (bit 0 x, 1 y, 2 z)
        auto steps = [&](auto near, auto wm, auto unit) {
            constexpr int NEAR = decltype(near)::value;
            constexpr int WM = decltype(wm)::value;
            constexpr bool UNIT = decltype(unit)::value;
            unsigned o = (unsigned)lane * 16u;
            double2 na, nb;
            source(buf, o, na, nb);
#pragma unroll 2
            for (int s = 0; s < kTile; ++s) {
                const double2 pa = na, pb = nb;
                o = (o + 16u) & kWrap;
                source(buf, o, na, nb);  // the next step's (the last one re-reads the first)
#pragma unroll
                for (int q = 0; q < NI; ++q) {
                    double dx = pa.x - x[q], dy = pa.y - y[q], dz = pb.x - z[q];
                    if (WM & 1) dx = wrap_half(dx, a.k);
                    if (WM & 2) dy = wrap_half(dy, a.k);
                    if (WM & 4) dz = wrap_half(dz, a.k);
                    sym_pair<NEAR, UNIT>(dx, dy, dz, m[q], pb.y, cm53, B, rskip, close, fx[q], fy[q], fz[q], gx, gy, gz);
                }
                gx = from_next_lane(gx);
                gy = from_next_lane(gy);
                gz = from_next_lane(gz);
            }
        };
        auto variants = [&](auto near, auto unit) {
            const int wm = (wx ? 1 : 0) | (wy ? 2 : 0) | (wz ? 4 : 0);
            if (wm == 0) steps(near, IntC<0>{}, unit);
            else if (V == PV_S1R2_NEAREST) steps(near, IntC<4>{}, unit);
            else if (V == PV_T3_NEAREST) {
                if (wm == 1) steps(near, IntC<1>{}, unit);
                else if (wm == 2) steps(near, IntC<2>{}, unit);
                else if (wm == 4) steps(near, IntC<4>{}, unit);
                else steps(near, IntC<7>{}, unit);
            }
        };
        // near tiles keep the products: a tenth of them or less
        if (far) {
            if (whole && (int64_t)(tile + 1) * kTile <= N) variants(IntC<0>{}, std::bool_constant<EQ>{});
            else variants(IntC<0>{}, std::false_type{});
        } else if (V == PV_R3 && off == 0) variants(IntC<2>{}, std::false_type{});
        else variants(IntC<1>{}, std::false_type{});
        if (__any(close)) {
            // rare: the pairs within the bound, with the exact softening
            // (every lane goes round, so that the source sums do).  Not those
            // of rows and sources past the end, copies of the last particle
            // that would all take it (T3 nearest N = 8500: one workgroup held
            // the kernel for twice its time, 0.18 ms a call, now 0.12); a
            // periodic row is formed again for the next tile
            if (V != PV_R3 && (int64_t)(b + 1) * (kSymWaves * 64 * NI) > N) {
#pragma unroll
                for (int q = 0; q < NI; ++q)
                    if (row0 + q * 64 >= N) x[q] = NAN;
            }
#pragma unroll 1
            for (int s = 0; s < kTile; ++s) {
                const int id = (lane + s) & 63;
                double2 pa, pb;
                source(buf, (unsigned)id * 16u, pa, pb);
                const int64_t jt = (int64_t)tile * kTile + id, j = min(jt, N - 1);
                const double Bj = jt < N ? B : 0.0;
#pragma unroll
                for (int q = 0; q < NI; ++q) {
                    double dx = pa.x - x[q], dy = pa.y - y[q], dz = pb.x - z[q];
                    if (V == PV_T3_NEAREST && wx) dx = wrap_half(dx, a.k);
                    if (V == PV_T3_NEAREST && wy) dy = wrap_half(dy, a.k);
                    if (V != PV_R3 && wz) dz = wrap_half(dz, a.k);
                    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
                    if (r2 < Bj) sym_close_pair(r2, dx, dy, dz, m[q], pb.y, a.soft, min(row0 + q * 64, N - 1), j, cm53,
                                               fx[q], fy[q], fz[q], gx, gy, gz);
                }
                gx = from_next_lane(gx);
                gy = from_next_lane(gy);
                gz = from_next_lane(gz);
            }
        }
        if (off > 0) {
            gsum[buf][wave][0][lane] = gx;
            gsum[buf][wave][1][lane] = gy;
            gsum[buf][wave][2][lane] = gz;
        }
        // one barrier a tile: closes the source sums and the next tile's
        // records; both buffers are reused two tiles on, past the next barrier
        __syncthreads();
        if (off > 0 && tid < 3 * kTile) {
            const int c = tid >> 6;
            const int64_t j = (int64_t)tile * kTile + lane;
            double g = gsum[buf][0][c][lane];
#pragma unroll
            for (int v = 1; v < kSymWaves; ++v) g += gsum[buf][v][c][lane];
            if (j < N)
                a.part[sym_slot(N, cell_l, a.cell_tasks, a.cell_offs, a.cell_tasks + off - cell * a.cell_offs) +
                       (size_t)c * N + j] = EQ ? g * mass : g;
        }
        w = nw;
        have = more;
    }

    double *out = a.part + sym_slot(N, cell_l, a.cell_tasks, a.cell_offs, task);
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int64_t r = row0 + q * 64;
        if (r < N) {
            out[r] = EQ ? fx[q] * mass : fx[q];
            out[N + r] = EQ ? fy[q] * mass : fy[q];
            out[2 * N + r] = EQ ? fz[q] * mass : fz[q];
        }
    }
}

// ---------------------------------------------------------------------------
// Mixed precision, R3 and T3 nearest image: the scheme of sym_kernel with FP32
// pairs.  A tile's sources are FP32 offsets from the tile's centre (jrel), a
// row's offset is formed in FP64 (its image nearest the tile on periodic
// axes) and rounded once per tile.  FP32 sums: a source's run over eight steps
// of NI rows (32 pairs), a row's over 32 sources, or eight in the nearest-image
// modes, whose forces are small residuals; both are then added in FP64, the
// source's in LDS.  (Over 64 pairs each: 4% faster in R3, 3% in T3, but a
// median row's error 4.8e-7 instead of 3.3e-7 at N = 100000, where the
// one-sided kernel has 4.6e-7, and 4.7e-7 instead of 3.1e-7 on a lattice.)  Pairs within the bound, or
// within 1e-6 L of half a period on an axis that is wrapped per pair (where
// FP32 could take the other image), are done again in FP64.
//
// Measured against the one-sided kernels (ms): R3 N = 16384 0.235 -> 0.192,
// 100003 4.0 -> 2.8, 1.5 10^6 580 -> 492; T3 nearest, one mass, 40^3 2.40 ->
// 2.17 and 64^3 28.4 -> 27.7 against this kernel with the products, 38.3
// one-sided; below N = 14336 the one-sided kernel is
// as fast (R3 N = 9000: 0.189 against 0.217).  Bound by VALU issue at ~65
// cycles a pair evaluation and SIMD for 17.5 instructions: fewer or more waves
// (2, 3, 5, 6 per SIMD) and 8 rows per lane all measured 0-15% slower.  Six of
// them are FMAs on three VGPR operands, where the one-sided kernel has three
// and takes its sources from SGPRs, so the gain stays below FP64's.
// ---------------------------------------------------------------------------
// The power of two at or below |m|, in the FP32 range (1 for no mass).
__device__ __forceinline__ double unit_mass(double m) {
    return m == 0.0 ? 1.0 : ldexp(1.0, max(-126, min(127, ilogb(m))));
}

// EQ: sym_kernel's, the masses one value (R3: unit_mass) or 0 and one product
// at the end.
template <int V, int NI, bool EQ, class In>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void sym_mixed_kernel(const In in) {
    int b;
    unsigned by;
    const SymArgs &a = sym_this(in, b, by);
    constexpr int kFlush = 32 / NI, kRowFlush = V == PV_R3 ? 4 * kFlush : kFlush;  // steps of an FP32 sum
    __shared__ __align__(1024) float4 jbuf[2][kTile];
    __shared__ double gsum[2][kSymWaves][3][kTile];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t N = a.k.N;
    const int ntiles = (int)((N + kTile - 1) / kTile);
    const int cell_l = by / a.cell_tasks, task = by % a.cell_tasks;
    const int cell = a.cell0 + cell_l;
    SymWalk w;
    w.r = cell * a.cell_offs * a.tb + task * a.tpt;
    w.end = w.r + a.tpt;

    KScalars k = a.k;
    const int64_t row0 = ((int64_t)b * kSymWaves + wave) * (64 * NI) + lane;
    const double um = EQ && V == PV_R3 ? unit_mass(a.rec[0].w) : 1.0;  // what a particle of EQ has in the pairs
    double fx[NI], fy[NI], fz[NI];
    float m[NI];
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int64_t r = row0 + q * 64;
        m[q] = r < N ? (EQ ? (float)um : (float)a.rec[min(r, N - 1)].w) : 0.0f;
        fx[q] = fy[q] = fz[q] = 0.0;
    }
    auto stage = [&](int buf, int tile) {  // wave 0: one source per lane
        const int64_t j = (int64_t)tile * kTile + lane;
        float4 p = a.jrel[min(j, N - 1)];
        if (EQ) p.w = (float)um;
        if (j >= N) p.w = 0.0f;
        jbuf[buf][lane] = p;
    };
    const double mass = EQ ? a.rec[0].w / um : 1.0;
    const bool whole = EQ && (int64_t)(b + 1) * (kSymWaves * 64 * NI) <= N;  // no row past the end
    bool have = w.settle(a, b, ntiles);
    if (have && wave == 0) stage(0, w.tile);
    __syncthreads();

    for (int it = 0; have; ++it) {
        const int buf = it & 1;
        const int tile = w.tile, off = w.off;
        SymWalk nw = w;
        ++nw.r;
        const bool more = nw.settle(a, b, ntiles);
        if (more && wave == 0) stage(buf ^ 1, nw.tile);

        const double4 tc = a.tiles[tile], te = a.ext[tile];
        bool far = true, wx = false, wy = false, wz = false;  // as in sym_kernel
        // R3: r^-3 of every pair is well inside the FP32 range (r from 1e-12, or
        // the bound, to 3.5e12), so the masses may come after it
        bool mid = true;
        const float reach = 2e12f - (float)fmax(fmax(te.x, te.y), te.z);
        float B = 0.0f;
        if (V != PV_R3) {
#pragma unroll
            for (int q = 0; q < NI; ++q) {
                const double4 p = a.rec[min(row0 + q * 64, N - 1)];
                double sh;
                if (V == PV_T3_NEAREST) {
                    wx = !tile_shift(p.x, tc.x, te.x, k, sh, 1e-5) || wx;
                    wy = !tile_shift(p.y, tc.y, te.y, k, sh, 1e-5) || wy;
                }
                wz = !tile_shift(p.z, tc.z, te.z, k, sh, 1e-5) || wz;
            }
            wx = __any(wx);
            wy = __any(wy);
            wz = __any(wz);
        }
        // the row's coordinate on one axis: its image on the tile's side, or
        // (wrapped per pair) the one nearest the tile's centre
        auto place = [&](double x, double c, double e, bool wrapped) {
            if (wrapped) return near_image(x, c, k);
            double sh = 0.0;
            tile_shift(x, c, e, k, sh, 1e-5);
            return x - sh;
        };
        float x[NI], y[NI], z[NI], ax[NI], ay[NI], az[NI];
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            const int64_t r = min(row0 + q * 64, N - 1);
            double4 p = a.rec[r];
            if (V == PV_T3_NEAREST) {
                p.x = place(p.x, tc.x, te.x, wx);
                p.y = place(p.y, tc.y, te.y, wy);
            }
            if (V != PV_R3) p.z = place(p.z, tc.z, te.z, wz);
            x[q] = (float)(p.x - tc.x);
            y[q] = (float)(p.y - tc.y);
            z[q] = (float)(p.z - tc.z);
            ax[q] = ay[q] = az[q] = 0.0f;
            // widened by 1e-5: FP32 rounding of r2 cannot hide a pair within the bound
            const float bq = (float)((a.soft[r] + tc.w) * (1.0 + 1e-5));
            B = fmaxf(B, bq * bq);
            const double gx = wx ? 0.0 : fmax(fabs(p.x - tc.x) - te.x, 0.0);
            const double gy = wy ? 0.0 : fmax(fabs(p.y - tc.y) - te.y, 0.0);
            const double gz = wz ? 0.0 : fmax(fabs(p.z - tc.z) - te.z, 0.0);
            const double d2 = fma(gx, gx, fma(gy, gy, gz * gz));
            far = far && d2 > (double)(bq * bq) * (1.0 + 1e-3);
            if (V == PV_R3) mid = mid && fmax(d2, (double)(bq * bq)) > 1e-24 && fmaxf(fmaxf(fabsf(x[q]), fabsf(y[q])), fabsf(z[q])) < reach;
        }
        far = __all(far);
        if (V == PV_R3) mid = __all(mid);
        if (off > 0) gsum[buf][wave][0][lane] = gsum[buf][wave][1][lane] = gsum[buf][wave][2][lane] = 0.0;

        bool close = false;
        float gx = 0.0f, gy = 0.0f, gz = 0.0f;
        // one axis' nearest image in FP32; bnd: within 1e-6 L of half a period
        auto wrap = [&](float d, bool &bnd) {
            const float h = fabsf(d) - k.halfLf;
            bnd = bnd || fabsf(h) < k.wrap_epsf;
            return h > 0.0f ? d - copysignf(k.Lf, d) : d;
        };
        auto end_rows = [&](const double scale) {
#pragma unroll
            for (int q = 0; q < NI; ++q) {
                fx[q] = fma((double)ax[q], scale, fx[q]);
                fy[q] = fma((double)ay[q], scale, fy[q]);
                fz[q] = fma((double)az[q], scale, fz[q]);
                ax[q] = ay[q] = az[q] = 0.0f;
            }
        };
        auto steps = [&](auto near, auto wm, auto unit, auto plain) {
            constexpr int NEAR = decltype(near)::value;
            constexpr int WM = decltype(wm)::value;
            constexpr bool UNIT = decltype(unit)::value;
            constexpr bool PLAIN = decltype(plain)::value;  // r^-3 by itself, then the masses
            const double scale = UNIT && PLAIN ? um : 1.0;
            unsigned o = (unsigned)lane * 16u;
            const char *base = (const char *)&jbuf[buf][0];
            float4 nj = *(const float4 *)(base + o);
            for (int s0 = 0; s0 < kTile; s0 += kFlush) {
#pragma unroll 2
                for (int s = 0; s < kFlush; ++s) {
                    const float4 pj = nj;
                    o = (o + 16u) & 1023u;
                    nj = *(const float4 *)(base + o);  // the next step's (the last one re-reads the first)
#pragma unroll
                    for (int q = 0; q < NI; ++q) {
                        float dx = pj.x - x[q], dy = pj.y - y[q], dz = pj.z - z[q];
                        bool c = false;
                        if (WM & 1) dx = wrap(dx, c);
                        if (WM & 2) dy = wrap(dy, c);
                        if (WM & 4) dz = wrap(dz, c);
                        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                        float yr = __builtin_amdgcn_rsqf(r2);
                        if (NEAR || WM) {
                            if (NEAR) c = c || r2 < B;
                            close = close || c;
                            yr = c ? 0.0f : yr;
                        }
                        const float t = yr * yr;
                        float sj, si;
                        if constexpr (!PLAIN) {
                            // the mass before r^-3, which alone leaves the FP32 range at 4e12 length
                            // units (one product more a pair: 3.5% at N = 10^6, so only where it has to be)
                            sj = t * (yr * (UNIT ? (float)um : pj.w));
                            si = UNIT ? sj : t * (yr * m[q]);
                        } else {
                            const float y3 = t * yr;
                            sj = UNIT ? y3 : y3 * pj.w;
                            si = UNIT ? y3 : y3 * m[q];
                        }
                        ax[q] = fmaf(sj, dx, ax[q]);
                        ay[q] = fmaf(sj, dy, ay[q]);
                        az[q] = fmaf(sj, dz, az[q]);
                        gx = fmaf(si, dx, gx);
                        gy = fmaf(si, dy, gy);
                        gz = fmaf(si, dz, gz);
                    }
                    gx = from_next_lane(gx);
                    gy = from_next_lane(gy);
                    gz = from_next_lane(gz);
                }
                if (off > 0) {
                    // lane l holds source (l + s0 + kFlush) mod 64's sums; the
                    // wave's LDS operations are in order
                    const int id = (lane + s0 + kFlush) & 63;
                    __builtin_amdgcn_wave_barrier();
                    gsum[buf][wave][0][id] = fma((double)gx, scale, gsum[buf][wave][0][id]);
                    gsum[buf][wave][1][id] = fma((double)gy, scale, gsum[buf][wave][1][id]);
                    gsum[buf][wave][2][id] = fma((double)gz, scale, gsum[buf][wave][2][id]);
                    __builtin_amdgcn_wave_barrier();
                }
                gx = gy = gz = 0.0f;
                if ((s0 + kFlush) % kRowFlush == 0) end_rows(scale);
            }
        };
        auto variants = [&](auto near, auto unit) {
            const int wm = (wx ? 1 : 0) | (wy ? 2 : 0) | (wz ? 4 : 0);
            if (V == PV_R3) {
                if (mid) steps(near, IntC<0>{}, unit, std::true_type{});
                else steps(near, IntC<0>{}, unit, std::false_type{});
            } else if (wm == 0) steps(near, IntC<0>{}, unit, std::true_type{});
            else if (wm == 1) steps(near, IntC<1>{}, unit, std::true_type{});
            else if (wm == 2) steps(near, IntC<2>{}, unit, std::true_type{});
            else if (wm == 4) steps(near, IntC<4>{}, unit, std::true_type{});
            else steps(near, IntC<7>{}, unit, std::true_type{});
        };
        if (far) {
            if (whole && (int64_t)(tile + 1) * kTile <= N) variants(IntC<0>{}, std::bool_constant<EQ>{});
            else variants(IntC<0>{}, std::false_type{});
        } else variants(IntC<1>{}, std::false_type{});
        if (__any(close)) {
            // rare: those pairs in FP64 from the FP64 records
            double cx = 0.0, cy = 0.0, cz = 0.0;
#pragma unroll 1
            for (int s = 0; s < kTile; ++s) {
                const int id = (lane + s) & 63;
                const float4 pj = jbuf[buf][id];
                const int64_t j = min((int64_t)tile * kTile + id, N - 1);
#pragma unroll
                for (int q = 0; q < NI; ++q) {
                    float dx = pj.x - x[q], dy = pj.y - y[q], dz = pj.z - z[q];
                    bool c = false;
                    if (V == PV_T3_NEAREST && wx) dx = wrap(dx, c);
                    if (V == PV_T3_NEAREST && wy) dy = wrap(dy, c);
                    if (V != PV_R3 && wz) dz = wrap(dz, c);
                    c = c || (!far && fmaf(dx, dx, fmaf(dy, dy, dz * dz)) < B);
                    if (c) {
                        const int64_t i = min(row0 + q * 64, N - 1);
                        const double4 pi = a.rec[i], pd = a.rec[j];
                        double ex = pd.x - pi.x, ey = pd.y - pi.y, ez = pd.z - pi.z;
                        if (V == PV_T3_NEAREST) {
                            ex = wrap_half(ex, k);
                            ey = wrap_half(ey, k);
                        }
                        if (V != PV_R3) ez = wrap_half(ez, k);
                        const double r2 = fma(ex, ex, fma(ey, ey, ez * ez));
                        const double beta = a.soft[i] + a.soft[j];
                        double u = inv_r3(r2, 1.5);
                        if (r2 < beta * beta) u = softening_exact(sqrt(r2), beta);
                        const double sj = (pj.w == 0.0f ? 0.0 : (EQ ? um : pd.w)) * u,
                                     si = (m[q] == 0.0f ? 0.0 : (EQ ? um : pi.w)) * u;
                        fx[q] = fma(sj, ex, fx[q]);
                        fy[q] = fma(sj, ey, fy[q]);
                        fz[q] = fma(sj, ez, fz[q]);
                        cx = fma(si, ex, cx);
                        cy = fma(si, ey, cy);
                        cz = fma(si, ez, cz);
                    }
                }
                cx = from_next_lane(cx);
                cy = from_next_lane(cy);
                cz = from_next_lane(cz);
            }
            if (off > 0) {
                __builtin_amdgcn_wave_barrier();
                gsum[buf][wave][0][lane] += cx;
                gsum[buf][wave][1][lane] += cy;
                gsum[buf][wave][2][lane] += cz;
            }
        }
        __syncthreads();  // as in sym_kernel
        if (off > 0 && tid < 3 * kTile) {
            const int64_t j = (int64_t)tile * kTile + lane;
            double g = gsum[buf][0][wave][lane];
#pragma unroll
            for (int v = 1; v < kSymWaves; ++v) g += gsum[buf][v][wave][lane];
            if (j < N)
                a.part[sym_slot(N, cell_l, a.cell_tasks, a.cell_offs, a.cell_tasks + off - cell * a.cell_offs) +
                       (size_t)wave * N + j] = EQ ? g * mass : g;
        }
        w = nw;
        have = more;
    }

    double *out = a.part + sym_slot(N, cell_l, a.cell_tasks, a.cell_offs, task);
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int64_t r = row0 + q * 64;
        if (r < N) {
            out[r] = EQ ? fx[q] * mass : fx[q];
            out[N + r] = EQ ? fy[q] * mass : fy[q];
            out[2 * N + r] = EQ ? fz[q] * mass : fz[q];
        }
    }
}

// ---------------------------------------------------------------------------
// T3 Ewald: the same scheme, one row per lane.  The tricubic correction reads
// 192 table values per pair, and those reads are what the pair costs; here
// they serve both sides.  Records are in z pencils.  Before each source tile
// the workgroup copies the table window that its rows' and the tile's cell
// columns can reach into LDS, unfolded in x and y, so that a stencil is 16
// rows at fixed strides from one address: no mirror or wrap per row (638 ->
// 468 VALU per pair against the folded window of body_t3_win).  ZF: a table
// mirrored in z as well is looked up at |dz| and its z component takes the sign
// of dz, so a window row holds the nodes of z >= 0 only and the window 1.3
// times the rows, 1.9 in FP32 (FP64 24^3 9.7 -> 7.0 ms, 32^3 34 -> 21.4, 40^3 80
// -> 61, 56^3 443 -> 349; mixed 24^3 5.0 -> 3.6, 40^3 42 -> 35.5).  A window that does not fit
// is taken in up to three bands of y rows, each its own pass over the steps in
// which the lanes whose stencils lie in the band take part (32^3 46 -> 34 ms;
// more bands gain nothing); a wider one leaves the tile on the global table,
// and so does a lane whose stencil leaves the window.  The eight waves of a workgroup are W / G sets of 64
// rows times G groups of 64 / G steps: fewer rows make a smaller window, so
// sparse boxes (few particles per column) take G = 4 or 8.  After the tile
// the window's memory takes the waves' source sums.
//
// Bound by LDS: 96 reads of 16 bytes per pair (ZF; 112 else), 4.3 cycles each,
// and as much again in bank conflicts (876 LDS cycles of 978 per wave step at
// 60^3 with 112).  In
// the lanes of one read the source and row indices both advance, so their
// stencils sit a few z nodes apart on 2 x 2 neighbouring rows; the (x, y)
// nodes are therefore stored by z mod 4 (lanes a few nodes apart then share
// words) and rows 4 (ZF: 12), planes 8 words apart mod 16.  Measured at 60^3: folded
// body_t3_win rows 737 ms, this layout 615; planes at 4 or 2 mod 16 695 / 652,
// rows of 104 or 108 words 630 / 633, z components as single 8-byte reads 710.
// Measured against the one-sided kernels (ms): 16^3 3.0 -> 1.3, 24^3 22.7 -> 7.0,
// 32^3 91 -> 21.4, 40^3 310 -> 61, 48^3 739 -> 155, 56^3 1440 -> 349.
//
// MX, mixed precision: the displacement is formed and wrapped in FP64 and
// rounded once, the rest of a pair is FP32, with 16-byte nodes (64 reads a
// pair); FP32 sums run over eight steps and are added in FP64,
// pairs within the softening bound are done again in FP64 (body_t3_mixed's
// scheme).  VALU (420 per pair) and LDS (490 cycles) are about even there:
// 24^3 14.6 -> 3.6 ms, 40^3 190 -> 35.5, 48^3 490 -> 93, 56^3 1092 -> 221.
// ---------------------------------------------------------------------------
constexpr int kSymT3Win = 9800;   // 16-byte words: 153 KB, one workgroup per CU
constexpr int kT3Waves = 8;
constexpr int kMxRun = 8;         // mixed: steps of an FP32 sum
constexpr int kT3Bands = 3;       // most bands of a window (see sym_t3_kernel)
constexpr int kT3MaxWinNg = 63;   // the window row is laid out for tables up to this grid

// A window row, in words: the (x, y) nodes in four runs by z mod 4, then the z
// components, two nodes a word; FP32 nodes take one word each and have no z
// part.  All z nodes (66), or those of z >= 0 (35), whose z components then
// stand twice, in pairs from even and (zodd) from odd nodes: a stencil's four
// are two words at either start, where one run takes three (FP64 36^3 40 ->
// 35 ms, 56^3 405 -> 349).
template <bool ZF> struct T3Row;
template <> struct T3Row<false> {
    static constexpr int words = 100, words32 = 68, zpairs = 66, zodd = 0;
    static __device__ __forceinline__ constexpr unsigned run(unsigned r) {
        return r == 0u ? 0u : (r == 1u ? 17u : (r == 2u ? 34u : 50u));
    }
};
template <> struct T3Row<true> {
    static constexpr int words = 76, words32 = 36, zpairs = 36, zodd = 54;
    static __device__ __forceinline__ constexpr unsigned run(unsigned r) { return 9u * r; }
};

// Words from one x plane of window rows to the next: 8 (mod 16), which with
// rows 4 (mod 16) apart spreads the 2 x 2 neighbouring rows that the lanes
// of a read mostly sit on over different banks.
__device__ __forceinline__ int t3_plane(int ny, int row) { return ny * row + ((8 - ny * row) & 15); }

// Unfolded nodes one axis of the window holds: n0 .. n0 + n - 1 (mod Ng), n0
// in [0, Ng), for sources in cell columns [smin, smax] and rows in [bmin,
// bmax] (see t3_win_axis).  n = 5 or 6 more than the columns the two span, up
// to 2 Ng + 4 where each spans the box; nodes then repeat, which the copy and
// t3_win_rel allow for (a window that wide fits on small grids only).
__device__ __forceinline__ void t3_win_nodes(int smin, int smax, int bmin, int bmax, int Ng, int &n0, int &n) {
    const int nlo = (smin - bmax) + (Ng - 1) / 2 - 2, nhi = (smax - bmin) + Ng / 2 + 2;
    n = nhi - nlo + 1;
    n0 = imodp(nlo, Ng);
}

// Stencil start of one axis relative to the window's first node: node
// floor(u) - 1 is window node rel; false when the four nodes leave the window
// (or the displacement the box).
__device__ __forceinline__ bool t3_win_rel(int i, int n0, int n, int Ng, unsigned &rel) {
    const int d = i - 1 - n0;
    rel = min((unsigned)d, (unsigned)(d + Ng));
    return (int)rel <= n - 4 && (int)rel >= 0;
}

// Catmull-Rom weights of one axis (t3_axis, t3_axis_f32 without the index wrap).
__device__ __forceinline__ int t3_weights(double d, const KScalars &k, double w[4]) {
    const double u = (d + k.L * 0.5) * k.inv_gs - 0.5;
    const double uf = floor(u);
    const double t = u - uf;
    const double t2 = t * t, t3 = t * t2;
    w[0] = -0.5 * t3 + t2 - 0.5 * t;
    w[1] = 1.5 * t3 - 2.5 * t2 + 1.0;
    w[2] = -1.5 * t3 + 2.0 * t2 + 0.5 * t;
    w[3] = 0.5 * t3 - 0.5 * t2;
    return (int)uf;
}
__device__ __forceinline__ int t3_weights(float d, const KScalars &k, float w[4]) {
    // from the centre node, not the edge: u is at most half as large, and small
    // where d is, so t keeps more of its bits
    const float u = fmaf(d, k.inv_gsf, (k.ng & 1) ? 0.0f : 0.5f);
    const float uf = floorf(u);
    const float t = u - uf;
    const float t2 = t * t, t3 = t * t2;
    w[0] = -0.5f * t3 + t2 - 0.5f * t;
    w[1] = 1.5f * t3 - 2.5f * t2 + 1.0f;
    w[2] = -1.5f * t3 + 2.0f * t2 + 0.5f * t;
    w[3] = 0.5f * t3 - 0.5f * t2;
    return (int)uf + (k.ng - 1) / 2;
}

// The z axis of a window that holds z >= 0: d >= 0, indices from node `first`
// (the one at or below z = 0, which rounding must not pass).
template <class T> __device__ __forceinline__ int t3_weights_from(T d, const KScalars &k, int first, T w[4]) {
    T u;
    if constexpr (sizeof(T) == 8) u = (d + k.L * 0.5) * k.inv_gs - 0.5 - (double)first;
    else u = fmaf(d, k.inv_gsf, (k.ng & 1) ? 0.0f : 0.5f);
    const T uf = fmax(floor(u), (T)0);
    const T t = u - uf;
    const T t2 = t * t, t3 = t * t2;
    w[0] = (T)-0.5 * t3 + t2 - (T)0.5 * t;
    w[1] = (T)1.5 * t3 - (T)2.5 * t2 + (T)1.0;
    w[2] = (T)-1.5 * t3 + (T)2.0 * t2 + (T)0.5 * t;
    w[3] = (T)0.5 * t3 - (T)0.5 * t2;
    return (int)uf;
}

template <int G, bool MX, bool ZF, class In>
__global__ __launch_bounds__(64 * kT3Waves) void sym_t3_kernel(const In in) {
    int b;
    unsigned by;
    const SymArgs &a = sym_this(in, b, by);
    constexpr int W = kT3Waves, RW = W / G;  // waves; waves of different rows
    constexpr int kSteps = kTile / G;
    constexpr int kRow = MX ? T3Row<ZF>::words32 : T3Row<ZF>::words, kZPairs = T3Row<ZF>::zpairs,
                  kZOdd = T3Row<ZF>::zodd;
    using real = std::conditional_t<MX, float, double>;
    __shared__ __align__(16) double win[2 * kSymT3Win];
    __shared__ __align__(16) double2 jbuf[2][kTile];
    __shared__ int brange[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t N = a.k.N;
    const int ntiles = (int)((N + kTile - 1) / kTile);
    const int cell_l = by / a.cell_tasks, task = by % a.cell_tasks;
    const int cell = a.cell0 + cell_l;
    SymWalk w;
    w.r = cell * a.cell_offs * a.tb + task * a.tpt;
    w.end = w.r + a.tpt;

    KScalars k = a.k;
    k.c15 = in_vgpr(a.k.c15);
    const int64_t row = (int64_t)b * (64 * RW) + (wave % RW) * 64 + lane;
    const int s0 = wave / RW * kSteps;  // the wave's first step
    const int64_t rowc = min(row, N - 1);
    const double4 p = a.rec[rowc];
    const double xi = p.x, yi = p.y, zi = p.z, mi = row < N ? p.w : 0.0, hi = a.soft[rowc];
    double fx = 0.0, fy = 0.0, fz = 0.0;
    const int Ng = k.ng, lo = k.t3_lo;
    const unsigned NY = (unsigned)(Ng - lo), NZ = (unsigned)(Ng + 3), NZ3 = 3u * NZ;
    // the window's z nodes: entries zf .. of a table row (ZF: from one below z = 0)
    const int zf = ZF ? (Ng - 1) / 2 : 0;
    const unsigned wz = NZ - (unsigned)zf, wz3 = 3u * wz;

    int bxmin = 0, bxmax = 0, bymin = 0, bymax = 0;  // the rows' cell columns
    {
        if (tid == 0) {
            brange[0] = brange[2] = INT32_MAX;
            brange[1] = brange[3] = -1;
        }
        __syncthreads();
        const uint32_t kr = a.keys[rowc];
        const int rbx = (int)(kr >> 20), rby = pencil_y(kr, Ng);
        atomicMin(&brange[0], rbx);
        atomicMax(&brange[1], rbx);
        atomicMin(&brange[2], rby);
        atomicMax(&brange[3], rby);
        __syncthreads();
        bxmin = brange[0];
        bxmax = brange[1];
        bymin = brange[2];
        bymax = brange[3];
    }
    auto stage = [&](int tile) {  // wave 0: one source per lane
        const int64_t j = (int64_t)tile * kTile + lane;
        const double4 q = a.rec[min(j, N - 1)];
        jbuf[0][lane] = make_double2(q.x, q.y);
        jbuf[1][lane] = make_double2(q.z, j < N ? q.w : 0.0);
    };
    bool have = w.settle(a, b, ntiles);
    if (have && wave == 0) stage(w.tile);

    while (have) {
        const int tile = w.tile, off = w.off;
        __syncthreads();  // records in place; the window's memory is free
        // The window's nodes, in bands of bys + 3 y rows that fit LDS: band b
        // serves the stencils that start at y rows [b bys, (b + 1) bys).
        int wx0 = 0, nx = 0, wy0 = 0, ny = 0, bys = 0, bands = 0;
        {
            const uint32_t kj = a.keys[min((int64_t)tile * kTile + lane, N - 1)];
            int sx0 = (int)(kj >> 20), sx1 = sx0, sy0 = pencil_y(kj, Ng), sy1 = sy0;
#pragma unroll
            for (int m = 32; m > 0; m >>= 1) {
                sx0 = min(sx0, __shfl_xor(sx0, m, 64));
                sx1 = max(sx1, __shfl_xor(sx1, m, 64));
                sy0 = min(sy0, __shfl_xor(sy0, m, 64));
                sy1 = max(sy1, __shfl_xor(sy1, m, 64));
            }
            t3_win_nodes(sx0, sx1, bxmin, bxmax, Ng, wx0, nx);
            t3_win_nodes(sy0, sy1, bymin, bymax, Ng, wy0, ny);
            wx0 = __builtin_amdgcn_readfirstlane(wx0);
            wy0 = __builtin_amdgcn_readfirstlane(wy0);
            nx = __builtin_amdgcn_readfirstlane(nx);
            ny = __builtin_amdgcn_readfirstlane(ny);
            bys = min(ny, (kSymT3Win / nx - 12) / kRow) - 3;  // 12: the most t3_plane adds
            bands = bys > 0 ? (ny - 3 + bys - 1) / bys : INT32_MAX;
            if (bands > kT3Bands) bands = 0;  // the global table
        }
        const double bb = hi + a.tiles[tile].w;
        const double B = bb * bb;
        // mixed: the FP32 bound, widened so that rounding cannot hide a pair
        const float Bf = (float)(bb * (1.0 + 1e-5)) * (float)(bb * (1.0 + 1e-5));
        double hx = 0.0, hy = 0.0, hz = 0.0;
        bool near = false;
        for (int band = 0; band == 0 || band < bands; ++band) {
            if (band > 0) __syncthreads();  // every wave is done with the previous band
            const int y0 = band * bys, nyb = min(bys + 3, ny - y0);
            const int plane = t3_plane(nyb, kRow);
            if (bands > 0) {
                // a wave copies whole rows (lanes along the z run), unfolding
                // them: a node below lo is its mirror with that component negated
                for (int rw = wave; rw < nx * nyb; rw += W) {
                    const int ax = rw / nyb, ay = rw - ax * nyb;
                    int jx = wx0 + ax, jy = wy0 + y0 + ay;
                    while (jx >= Ng) jx -= Ng;
                    while (jy >= Ng) jy -= Ng;
                    const bool fx_ = jx < lo, fy_ = jy < lo;
                    const unsigned mx = (unsigned)(fx_ ? Ng - 1 - lo - jx : jx - lo);
                    const unsigned my = (unsigned)(fy_ ? Ng - 1 - lo - jy : jy - lo);
                    if constexpr (MX) {
                        const float4 *src = a.tab32 + (mx * NY + my) * NZ + zf;
                        float4 *dst = (float4 *)win + ax * plane + ay * kRow;
                        for (unsigned z = lane; z < wz; z += 64) {
                            float4 v = src[z];
                            if (fx_) v.x = -v.x;
                            if (fy_) v.y = -v.y;
                            dst[T3Row<ZF>::run(z & 3u) + (z >> 2)] = v;
                        }
                    } else {
                        const double *src = a.table + (mx * NY + my) * NZ3 + 3 * zf;
                        double *dst = win + 2 * (ax * plane + ay * kRow);
                        for (unsigned o = lane; o < wz3; o += 64) {
                            const unsigned z = o / 3u, c = o - 3u * z;
                            double v = src[o];
                            if (c == 0u && fx_) v = -v;
                            if (c == 1u && fy_) v = -v;
                            dst[c < 2u ? 2u * (T3Row<ZF>::run(z & 3u) + (z >> 2)) + c : 2u * kZPairs + z] = v;
                            if (ZF && c == 2u && z > 0u) dst[2u * kZOdd + z - 1u] = v;
                        }
                        if constexpr (!ZF) {
                            // z values past the run meet zero weights
                            const unsigned pad = 2u * kZPairs + wz + lane;
                            if (pad < 2u * kRow) dst[pad] = 0.0;
                        }
                    }
                }
            }
            __syncthreads();  // the window is complete
            real gx = 0, gy = 0, gz = 0, ax = 0, ay = 0, az = 0;
            // mixed: the FP32 sums of a run of steps onto FP64 ones; a run moves
            // the sources kMxRun lanes down, and their sums with them
            constexpr bool kRuns = MX && kSteps > kMxRun;
            double bx = 0.0, by = 0.0, bz = 0.0;
            auto end_run = [&] {
                fx += (double)ax;
                fy += (double)ay;
                fz += (double)az;
                const int from = (lane + kMxRun) & 63;
                bx = __shfl(bx, from, 64) + (double)gx;
                by = __shfl(by, from, 64) + (double)gy;
                bz = __shfl(bz, from, 64) + (double)gz;
                ax = ay = az = gx = gy = gz = 0;
            };
#pragma unroll 1
            for (int s = 0; s < kSteps; ++s) {
                if (kRuns && s > 0 && s % kMxRun == 0) end_run();
                const int id = (lane + s0 + s) & 63;
                const double2 pa = jbuf[0][id], pb = jbuf[1][id];
                // the displacement is formed and wrapped in FP64 (mixed: then rounded once)
                const real dx = (real)wrap_half(pa.x - xi, k), dy = (real)wrap_half(pa.y - yi, k),
                           dz = (real)wrap_half(pb.x - zi, k);
                // the band that holds this pair's stencil: its share of the pair is
                // the correction, and band 0 also has the direct force (and, from
                // the global table, the corrections of stencils no band holds)
                real wxs[4], wys[4], wzs[4];
                unsigned rx = 0, ry = 0, iz = 0;
                bool in = false, out = band == 0;
                if (bands > 0) {
                    const int ix = t3_weights(dx, k, wxs), iy = t3_weights(dy, k, wys);
                    unsigned nz = (unsigned)Ng;
                    if constexpr (ZF) {
                        // |dz|: the z component changes sign with dz, the others are even in it
                        iz = (unsigned)t3_weights_from(dz < 0 ? -dz : dz, k, zf, wzs);
                        nz -= (unsigned)zf;
                    } else {
                        const int izi = t3_weights(dz, k, wzs);
                        iz = min((unsigned)izi, (unsigned)(izi + Ng));  // layout z index of the stencil's first node
                    }
                    const bool inx = t3_win_rel(ix, wx0, nx, Ng, rx), iny = t3_win_rel(iy, wy0, ny, Ng, ry);
                    const bool held = inx && iny && iz < nz;
                    ry -= (unsigned)y0;
                    in = held && ry < (unsigned)bys;
                    out = band == 0 && !held;
                }
                real wp = 0, mj, mr;
                if constexpr (MX) {
                    const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                    const bool nr = r2 < Bf;  // left to the FP64 redo (r2 may be 0 here)
                    near = near || nr;
                    const float y = __builtin_amdgcn_rsqf(r2);
                    wp = (nr || band > 0) ? 0.0f : (y * y) * y;
                    mj = nr ? 0.0f : (float)pb.y;
                    mr = nr ? 0.0f : (float)mi;
                } else {
                    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
                    if (band == 0) wp = pair_w_tile(r2, B, hi, a.soft, min((int64_t)tile * kTile + id, N - 1), k);
                    mj = pb.y;
                    mr = mi;
                }
                real Dx = 0, Dy = 0, Dz = 0;
                if (in) {
                    // (x, y) nodes by z mod 4: read k takes the stencil's node with
                    // z = k (mod 4), so lanes a few nodes apart read the same word
                    // or neighbouring ones
                    const unsigned r = iz & 3u, blk = iz >> 2;
                    const bool r1 = (r & 1u) != 0u, r2b = (r & 2u) != 0u;
                    const real p0 = r1 ? wzs[3] : wzs[0], p1 = r1 ? wzs[0] : wzs[1], p2 = r1 ? wzs[1] : wzs[2],
                               p3 = r1 ? wzs[2] : wzs[3];
                    const real wk[4] = {r2b ? p2 : p0, r2b ? p3 : p1, r2b ? p0 : p2, r2b ? p1 : p3};
                    const unsigned base = rx * (unsigned)plane + ry * (unsigned)kRow;
                    unsigned at[4];
#pragma unroll
                    for (unsigned q = 0; q < 4; ++q) at[q] = base + T3Row<ZF>::run(q) + blk + (q < r ? 1u : 0u);
                    real s0 = 0, s1 = 0, s2 = 0;
                    if constexpr (MX) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float4 *pk[4];
#pragma unroll
                            for (int q = 0; q < 4; ++q) pk[q] = (const float4 *)win + at[q] + i * plane;
                            float u0 = 0.0f, u1 = 0.0f, u2 = 0.0f;
#pragma unroll
                            for (int jj = 0; jj < 4; ++jj) {
                                const float4 a0 = pk[0][jj * kRow], a1 = pk[1][jj * kRow], a2 = pk[2][jj * kRow],
                                             a3 = pk[3][jj * kRow];
                                // the unused fourth component keeps the reads 16 bytes wide:
                                // a 12-byte LDS read takes twice the cycles (8 against 4.3)
                                asm volatile("" ::"v"(a0.w), "v"(a1.w), "v"(a2.w), "v"(a3.w));
                                const float t0 = fmaf(wk[3], a3.x, fmaf(wk[2], a2.x, fmaf(wk[1], a1.x, wk[0] * a0.x)));
                                const float t1 = fmaf(wk[3], a3.y, fmaf(wk[2], a2.y, fmaf(wk[1], a1.y, wk[0] * a0.y)));
                                const float t2 = fmaf(wk[3], a3.z, fmaf(wk[2], a2.z, fmaf(wk[1], a1.z, wk[0] * a0.z)));
                                u0 = fmaf(wys[jj], t0, u0);
                                u1 = fmaf(wys[jj], t1, u1);
                                u2 = fmaf(wys[jj], t2, u2);
                            }
                            s0 = fmaf(wxs[i], u0, s0);
                            s1 = fmaf(wxs[i], u1, s1);
                            s2 = fmaf(wxs[i], u2, s2);
                        }
                    } else {
                        // z components: six nodes from the even start as three words, the extra two with weight 0
                        const double wz5[5] = {r1 ? 0.0 : wzs[0], r1 ? wzs[0] : wzs[1], r1 ? wzs[1] : wzs[2],
                                               r1 ? wzs[2] : wzs[3], r1 ? wzs[3] : 0.0};
                        const double2 *w2 = (const double2 *)win;
                        const unsigned zat = base + (unsigned)(ZF && r1 ? kZOdd : kZPairs) + (iz >> 1);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const double2 *pk[4], *pz = w2 + zat + i * plane;
#pragma unroll
                            for (int q = 0; q < 4; ++q) pk[q] = w2 + at[q] + i * plane;
                            double u0 = 0.0, u1 = 0.0, u2 = 0.0;
#pragma unroll
                            for (int jj = 0; jj < 4; ++jj) {
                                const double2 a0 = pk[0][jj * kRow], a1 = pk[1][jj * kRow], a2 = pk[2][jj * kRow],
                                              a3 = pk[3][jj * kRow];
                                const double2 z0 = pz[jj * kRow], z1 = pz[jj * kRow + 1];
                                const double t0 = fma(wk[3], a3.x, fma(wk[2], a2.x, fma(wk[1], a1.x, wk[0] * a0.x)));
                                const double t1 = fma(wk[3], a3.y, fma(wk[2], a2.y, fma(wk[1], a1.y, wk[0] * a0.y)));
                                double t2;
                                if constexpr (ZF)
                                    t2 = fma(wzs[3], z1.y, fma(wzs[2], z1.x, fma(wzs[1], z0.y, wzs[0] * z0.x)));
                                else
                                    t2 = fma(wz5[4], pz[jj * kRow + 2].x,
                                             fma(wz5[3], z1.y, fma(wz5[2], z1.x, fma(wz5[1], z0.y, wz5[0] * z0.x))));
                                u0 = fma(wys[jj], t0, u0);
                                u1 = fma(wys[jj], t1, u1);
                                u2 = fma(wys[jj], t2, u2);
                            }
                            s0 = fma(wxs[i], u0, s0);
                            s1 = fma(wxs[i], u1, s1);
                            s2 = fma(wxs[i], u2, s2);
                        }
                    }
                    Dx = s0;
                    Dy = s1;
                    Dz = ZF && dz < 0 ? -s2 : s2;
                } else if (out) {
                    if constexpr (MX) {
                        T3Stencil32 st;
                        t3_stencil_f32(k, dx, dy, dz, st);
                        t3_contract_f32(
                            st,
                            [&](int i, int jj, float4 *n) {
                                const float4 *g = a.tab32 + (st.mx[i] * NY + st.my[jj]) * NZ + (unsigned)st.iz0;
#pragma unroll
                                for (int q = 0; q < 4; ++q) n[q] = g[q];
                            },
                            Dx, Dy, Dz);
                    } else {
                        t3_interp(a.table, k, dx, dy, dz, Dx, Dy, Dz);
                    }
                }
                auto mad = [](real m, real v, real acc) {
                    if constexpr (MX) return fmaf(m, v, acc);
                    else return fma(m, v, acc);
                };
                const real px = mad(wp, dx, -Dx), py = mad(wp, dy, -Dy), pz = mad(wp, dz, -Dz);
                ax = mad(mj, px, ax);
                ay = mad(mj, py, ay);
                az = mad(mj, pz, az);
                gx = from_next_lane(mad(mr, px, gx));
                gy = from_next_lane(mad(mr, py, gy));
                gz = from_next_lane(mad(mr, pz, gz));
            }
            if (kRuns) end_run();
            fx += (double)ax;
            fy += (double)ay;
            fz += (double)az;
            hx += kRuns ? bx : (double)gx;
            hy += kRuns ? by : (double)gy;
            hz += kRuns ? bz : (double)gz;
        }
        if (MX && __any(near)) {
            // rare: the pairs within the bound, in FP64 with the FP64 table
            double cx = 0.0, cy = 0.0, cz = 0.0;
#pragma unroll 1
            for (int s = 0; s < kSteps; ++s) {
                const int id = (lane + s0 + s) & 63;
                const double2 pa = jbuf[0][id], pb = jbuf[1][id];
                const double ex = wrap_half(pa.x - xi, k), ey = wrap_half(pa.y - yi, k), ez = wrap_half(pb.x - zi, k);
                const float dx = (float)ex, dy = (float)ey, dz = (float)ez;
                if (fmaf(dx, dx, fmaf(dy, dy, dz * dz)) < Bf) {
                    const double r2 = fma(ex, ex, fma(ey, ey, ez * ez));
                    const double wp = pair_w_tile(r2, B, hi, a.soft, min((int64_t)tile * kTile + id, N - 1), k);
                    double Dx, Dy, Dz;
                    t3_interp(a.table, k, ex, ey, ez, Dx, Dy, Dz);
                    const double px = fma(wp, ex, -Dx), py = fma(wp, ey, -Dy), pz = fma(wp, ez, -Dz);
                    fx = fma(pb.y, px, fx);
                    fy = fma(pb.y, py, fy);
                    fz = fma(pb.y, pz, fz);
                    cx = fma(mi, px, cx);
                    cy = fma(mi, py, cy);
                    cz = fma(mi, pz, cz);
                }
                cx = from_next_lane(cx);
                cy = from_next_lane(cy);
                cz = from_next_lane(cz);
            }
            hx += cx;
            hy += cy;
            hz += cz;
        }
        SymWalk nw = w;
        ++nw.r;
        have = nw.settle(a, b, ntiles);
        __syncthreads();  // every wave is done with the window and the records
        if (off > 0) {
            const int id = (lane + s0 + kSteps) & 63;  // the source whose sums this lane holds now
            win[(3 * wave + 0) * kTile + id] = hx;
            win[(3 * wave + 1) * kTile + id] = hy;
            win[(3 * wave + 2) * kTile + id] = hz;
        }
        if (have && wave == 0) stage(nw.tile);
        __syncthreads();
        for (int c = wave; off > 0 && c < 3; c += W) {
            const int64_t j = (int64_t)tile * kTile + lane;
            double g = win[c * kTile + lane];
#pragma unroll
            for (int v = 1; v < W; ++v) g += win[(3 * v + c) * kTile + lane];
            if (j < N)
                a.part[sym_slot(N, cell_l, a.cell_tasks, a.cell_offs, a.cell_tasks + off - cell * a.cell_offs) +
                       (size_t)c * N + j] = g;
        }
        w = nw;
    }
    if (G > 1) {
        // the row sums of the step groups, added in their order
        __syncthreads();
        win[(3 * wave + 0) * kTile + lane] = fx;
        win[(3 * wave + 1) * kTile + lane] = fy;
        win[(3 * wave + 2) * kTile + lane] = fz;
        __syncthreads();
        if (wave >= RW) return;
#pragma unroll
        for (int g = 1; g < G; ++g) {
            fx += win[(3 * (wave + g * RW) + 0) * kTile + lane];
            fy += win[(3 * (wave + g * RW) + 1) * kTile + lane];
            fz += win[(3 * (wave + g * RW) + 2) * kTile + lane];
        }
    }
    if (row < N) {
        double *out = a.part + sym_slot(N, cell_l, a.cell_tasks, a.cell_offs, task);
        out[row] = fx;
        out[N + row] = fy;
        out[2 * N + row] = fz;
    }
}

// ---------------------------------------------------------------------------
// S1R2 with the tabulated correction (CIC, TSC): the same scheme, one row per
// lane, records in input order, and the rho rows of each source tile staged in
// LDS as in body_f64 (all waves on the same tile).  D_rho is even and D_z odd
// in dz (s1r2_table_odd), so one interpolation serves both sides.  MX: the
// displacement is formed and wrapped in FP64 and rounded once (FP32 offsets
// from the tile's centre, as in sym_mixed_kernel, would carry its extent into
// the error and could take another image at half a period) -- the
// rest of a pair is FP32 (FP32 copy of the table), FP32 sums run over eight
// steps and are added in FP64 (over a tile's 64, three times the error of a
// row), and pairs within the softening bound are done again in FP64.  A tile
// whose window holds every row and whose |dz| all end within half a period
// takes the short lookup s1r2_window (CIC 93.5 -> 86 ms at N = 262144, mixed
// CIC 11.6 -> 10.9 and TSC 17.7 -> 16.6 at N = 102400).  Against the one-sided
// kernels (resident calls on the cylinder, ms): N = 262144 FP64 CIC 182 -> 86;
// N = 38220 mixed TSC 8.1 -> 2.9.  Particles in another order than by radius
// have wide tiles, whose stencils come from the global table: N = 102400
// shuffled, CIC 118.8 -> 61.4 (mixed 73.8 -> 39.0), TSC 172 -> 88 (213 -> 64).
// Bound by VALU issue and LDS reads together.
// ---------------------------------------------------------------------------
constexpr int kSymS1Win = 2368;  // 16-byte words (37 KB: four workgroups per CU), two FP32 nodes a word

// r^2 of a mixed S1R2 pair, by which the main loop leaves a pair to the FP64
// redo and the redo takes it: one order of roundings for both.
__device__ __forceinline__ float s1r2_r2(float dx, float dy, float dz, float &rxy2) {
    rxy2 = fmaf(dx, dx, dy * dy);
    return fmaf(dz, dz, rxy2);
}

__device__ __forceinline__ double fract_of(double v) { return __builtin_amdgcn_fract(v); }
__device__ __forceinline__ float fract_of(float v) { return __builtin_amdgcn_fractf(v); }

// s1r2_interp_win for a pair whose rho rows lie in the window (rows w0 .. w0 +
// nw - 1, which the caller's bounds on rho ensure; the clamp only keeps a read
// inside it) and whose |dz| is at most half a period: no test of the row or of
// the z wrap, one address for the whole stencil, cells and offsets from one
// coordinate each.  rxy2 = dx^2 + dy^2.
template <int ORD, class real, class node>
__device__ __forceinline__ void s1r2_window(const node *win, int w0, int nw, unsigned nz3, const KScalars &k,
                                            const real rxy2, const real dz, real &q, real &Dz) {
    constexpr bool F64 = sizeof(real) == 8;
    constexpr int kRows = ORD == 2 ? 2 : 3;  // the stencil's rho rows, the first one at or below rho (CIC), below it (TSC)
    real inv_rho, rho, fz, ur;
    int iz;
    if constexpr (F64) {
        const double r = fmax(rxy2, 1e-300);  // on the axis: q finite, times dx = dy = 0
        inv_rho = rsqrt_f64(r);
        rho = r * inv_rho;
        ur = fmin(rho * k.inv_drho, k.last_r);
        const double half = 0.5 * (double)k.nz;
        const double uz = ORD == 2 ? fma(dz, k.inv_dzg, half + 0.5) : fmax(fma(dz, k.inv_dzg, half), 0.0);
        iz = (int)uz;
        fz = fract_of(uz);
    } else {
        inv_rho = rxy2 > 0.0f ? __builtin_amdgcn_rsqf(rxy2) : 0.0f;
        rho = rxy2 * inv_rho;
        ur = fminf(rho * k.inv_drhof, k.last_rf);
        // from the centre of the z axis: cell coordinates keep more bits there
        const bool shift = (ORD == 2) != ((k.nz & 1) != 0);
        const int base = ORD == 2 ? (k.nz + 1) / 2 : k.nz / 2;
        float uz = fmaf(dz, k.inv_dzgf, shift ? 0.5f : 0.0f);
        if (ORD != 2) uz = fmaxf(uz, -(float)base);
        iz = (int)floorf(uz) + base;
        fz = fract_of(uz);
    }
    const real um = ORD == 2 ? ur : ur + (real)0.5;
    const int ir = (int)um - (ORD == 2 ? 0 : 1);
    const real fr = fract_of(um);
    const int rel = min(max(ir - w0, 0), nw - kRows);
    const node *p = win + (__umul24((unsigned)rel, nz3) + (unsigned)iz);
    auto mad = [](real a, real b, real c) {
        if constexpr (F64) return fma(a, b, c);
        else return fmaf(a, b, c);
    };
    real Dr;
    if constexpr (ORD == 2) {
        const node t00 = p[0], t01 = p[1], t10 = p[nz3], t11 = p[nz3 + 1];
        const real a0 = mad(fr, t10.x - t00.x, t00.x), b0 = mad(fr, t11.x - t01.x, t01.x);
        const real a1 = mad(fr, t10.y - t00.y, t00.y), b1 = mad(fr, t11.y - t01.y, t01.y);
        Dr = mad(fz, b0 - a0, a0);
        Dz = mad(fz, b1 - a1, a1);
    } else {
        const real sr = fr - (real)0.5, sz = fz - (real)0.5;
        const real wr[3] = {(real)0.5 * ((real)0.5 - sr) * ((real)0.5 - sr), (real)0.75 - sr * sr,
                            (real)0.5 * ((real)0.5 + sr) * ((real)0.5 + sr)};
        const real wz[3] = {(real)0.5 * ((real)0.5 - sz) * ((real)0.5 - sz), (real)0.75 - sz * sz,
                            (real)0.5 * ((real)0.5 + sz) * ((real)0.5 + sz)};
        Dr = 0;
        Dz = 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const node *r = p + c * nz3;
            const node a = r[0], b = r[1], d = r[2];
            Dr = mad(wr[c], mad(wz[2], d.x, mad(wz[1], b.x, wz[0] * a.x)), Dr);
            Dz = mad(wr[c], mad(wz[2], d.y, mad(wz[1], b.y, wz[0] * a.y)), Dz);
        }
    }
    q = Dr * inv_rho;
}

template <int V, bool MX, class In>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void sym_s1r2_kernel(const In in) {
    int b;
    unsigned by;
    const SymArgs &a = sym_this(in, b, by);
    constexpr int W = kSymWaves;
    constexpr int ORD = V == PV_S1R2_CIC ? 2 : 4;
    constexpr int kNodes = MX ? 2 * kSymS1Win : kSymS1Win;
    using real = std::conditional_t<MX, float, double>;
    using node = std::conditional_t<MX, float2, double2>;
    __shared__ __align__(16) double2 win[kSymS1Win];
    __shared__ __align__(16) double2 jbuf[2][kTile];
    __shared__ int rng[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t N = a.k.N;
    const int ntiles = (int)((N + kTile - 1) / kTile);
    const int cell_l = by / a.cell_tasks, task = by % a.cell_tasks;
    const int cell = a.cell0 + cell_l;
    SymWalk w;
    w.r = cell * a.cell_offs * a.tb + task * a.tpt;
    w.end = w.r + a.tpt;

    KScalars k = a.k;
    k.c15 = in_vgpr(a.k.c15);
    const int64_t row = (int64_t)b * kBlock + tid;
    const int64_t rowc = min(row, N - 1);
    const double4 p = a.rec[rowc];
    const double xi = p.x, yi = p.y, zi = p.z, mi = row < N ? p.w : 0.0, hi = a.soft[rowc];
    double fx = 0.0, fy = 0.0, fz = 0.0;
    const unsigned nz3 = (unsigned)(k.nz + 3);

    auto stage = [&](int tile) {  // wave 0: one source per lane
        const int64_t j = (int64_t)tile * kTile + lane;
        const double4 q = a.rec[min(j, N - 1)];
        jbuf[0][lane] = make_double2(q.x, q.y);
        jbuf[1][lane] = make_double2(q.z, j < N ? q.w : 0.0);
    };
    bool have = w.settle(a, b, ntiles);
    if (have && wave == 0) stage(w.tile);
    if (tid < 4) rng[tid] = (tid & 1) ? INT32_MIN : INT32_MAX;

    for (int it = 0; have; ++it) {
        const int tile = w.tile, off = w.off;
        const double4 tc = a.tiles[tile], te = a.ext[tile];
        __syncthreads();  // records and range slot in place; the window's memory is free
        // rho of every pair lies between the distances from the row to the
        // near and far sides of the tile's xy box; the stencils read rho nodes
        // floor(rho / drho) - 1 .. floor + 2
        {
            const double ax = fabs(xi - tc.x), ay = fabs(yi - tc.y);
            const double gx = fmax(ax - te.x, 0.0), gy = fmax(ay - te.y, 0.0);
            const double ex = ax + te.x, ey = ay + te.y;
            int lo = (int)floor(fmin(sqrt(fma(gx, gx, gy * gy)) * k.inv_drho, k.last_r)) - 1;
            int up = (int)floor(fmin(sqrt(fma(ex, ex, ey * ey)) * k.inv_drho, k.last_r)) + 2;
#pragma unroll
            for (int m = 32; m > 0; m >>= 1) {
                lo = min(lo, __shfl_xor(lo, m, 64));
                up = max(up, __shfl_xor(up, m, 64));
            }
            if (lane == 0) {
                atomicMin(&rng[2 * (it & 1)], lo);
                atomicMax(&rng[2 * (it & 1) + 1], up);
            }
        }
        __syncthreads();
        const int w0 = max(rng[2 * (it & 1)], -1), w1 = min(rng[2 * (it & 1) + 1], k.nrho);  // ghost rows -1, Nrho
        const int nw = w1 - w0 + 1;
        const bool wok = (int64_t)nw * nz3 <= kNodes;
        if (tid < 2) rng[2 * ((it + 1) & 1) + tid] = tid ? INT32_MIN : INT32_MAX;  // the next tile's slot
        if (wok) {
            const unsigned nn = (unsigned)nw * nz3;  // rows w0 .. w1 are contiguous
            node *dst = (node *)win;
            const node *src;
            if constexpr (MX) src = s1r2_row32(a.tab32s, k, w0);
            else src = s1r2_row(a.table, k, w0);
            for (unsigned o = tid; o < nn; o += kBlock) dst[o] = src[o];
        }
        __syncthreads();  // the window is complete
        const double bb = hi + tc.w;
        const double B = bb * bb;
        const float Bf = (float)(bb * (1.0 + 1e-5)) * (float)(bb * (1.0 + 1e-5));  // mixed: widened
        real gx = 0, gy = 0, gz = 0, ax = 0, ay = 0, az = 0;
        double hx = 0.0, hy = 0.0, hz = 0.0;
        // a run's sums onto the FP64 ones (sym_t3_kernel's end_run)
        auto end_run = [&] {
            fx += (double)ax;
            fy += (double)ay;
            fz += (double)az;
            const int from = (lane + kMxRun) & 63;
            hx = __shfl(hx, from, 64) + (double)gx;
            hy = __shfl(hy, from, 64) + (double)gy;
            hz = __shfl(hz, from, 64) + (double)gz;
            ax = ay = az = gx = gy = gz = 0;
        };
        bool near = false;
        auto steps = [&](auto fast) {
            unsigned o = (unsigned)lane * 16u;
#pragma unroll 1
            for (int s = 0; s < kTile; ++s, o = (o + 16u) & (16u * kTile - 1u)) {
                if (MX && s > 0 && s % kMxRun == 0) end_run();
                const char *at = (const char *)&jbuf[0][0] + o;
                const double2 pa = *(const double2 *)at, pb = *(const double2 *)(at + sizeof(jbuf[0]));
                const real dx = (real)(pa.x - xi), dy = (real)(pa.y - yi), dz = (real)wrap_half(pb.x - zi, k);
                real wp, mj, mr, qd, Dz, rxy2;
                if constexpr (MX) {
                    const float r2 = s1r2_r2(dx, dy, dz, rxy2);
                    const bool nr = r2 < Bf;  // left to the FP64 redo (r2 may be 0 here)
                    near = near || nr;
                    const float y = __builtin_amdgcn_rsqf(r2);
                    wp = nr ? 0.0f : (y * y) * y;
                    mj = nr ? 0.0f : (float)pb.y;
                    mr = nr ? 0.0f : (float)mi;
                } else {
                    rxy2 = fma(dx, dx, dy * dy);
                    const double r2 = fma(dz, dz, rxy2);
                    wp = pair_w_tile(r2, B, hi, a.soft, min((int64_t)tile * kTile + (o >> 4), N - 1), k);
                    mj = pb.y;
                    mr = mi;
                }
                if constexpr (decltype(fast)::value)
                    s1r2_window<ORD, real, node>((const node *)win, w0, nw, nz3, k, rxy2, dz, qd, Dz);
                else if constexpr (MX)
                    s1r2_interp_f32<ORD, true>(a.tab32s, k, dx, dy, dz, qd, Dz,
                                               S1R2Win32{(const float2 *)win, w0, nw, wok});
                else
                    s1r2_interp_win<ORD>(a.table, k, dx, dy, dz, qd, Dz, S1R2Win{win, w0, nw, wok});
                // m (w d - D) with D_x = q dx, D_y = q dy: x and y share m (w - q)
                auto mad = [](real m, real v, real acc) {
                    if constexpr (MX) return fmaf(m, v, acc);
                    else return fma(m, v, acc);
                };
                const real sxy = wp - qd, pz = mad(wp, dz, -Dz), sj = mj * sxy, si = mr * sxy;
                ax = mad(sj, dx, ax);
                ay = mad(sj, dy, ay);
                az = mad(mj, pz, az);
                gx = from_next_lane(mad(si, dx, gx));
                gy = from_next_lane(mad(si, dy, gy));
                gz = from_next_lane(mad(mr, pz, gz));
            }
        };
        // every |dz| within half a period after one wrap (else the general path)
        if (wok && __all(fabs(zi - tc.z) + te.z <= k.L * (1.5 - 1e-9))) steps(std::true_type{});
        else steps(std::false_type{});
        if (MX) {
            end_run();
        } else {
            fx += ax;
            fy += ay;
            fz += az;
            hx = gx;
            hy = gy;
            hz = gz;
        }
        if (MX && __any(near)) {
            // rare: the pairs within the bound, in FP64 with the FP64 table
            double cx = 0.0, cy = 0.0, cz = 0.0;
#pragma unroll 1
            for (int s = 0; s < kTile; ++s) {
                const int id = (lane + s) & 63;
                const double2 pa = jbuf[0][id], pb = jbuf[1][id];
                const double ex = pa.x - xi, ey = pa.y - yi, ez = wrap_half(pb.x - zi, k);
                const float dx = (float)ex, dy = (float)ey, dz = (float)ez;
                float rxy2;
                if (s1r2_r2(dx, dy, dz, rxy2) < Bf) {
                    const double r2 = fma(ex, ex, fma(ey, ey, ez * ez));
                    const double wp = pair_w_tile(r2, B, hi, a.soft, min((int64_t)tile * kTile + id, N - 1), k);
                    double qd, Dz;
                    s1r2_interp<ORD>(a.table, k, ex, ey, ez, qd, Dz);
                    const double sxy = wp - qd, pz = fma(wp, ez, -Dz);
                    fx = fma(pb.y * sxy, ex, fx);
                    fy = fma(pb.y * sxy, ey, fy);
                    fz = fma(pb.y, pz, fz);
                    cx = fma(mi * sxy, ex, cx);
                    cy = fma(mi * sxy, ey, cy);
                    cz = fma(mi, pz, cz);
                }
                cx = from_next_lane(cx);
                cy = from_next_lane(cy);
                cz = from_next_lane(cz);
            }
            hx += cx;
            hy += cy;
            hz += cz;
        }
        SymWalk nw_ = w;
        ++nw_.r;
        have = nw_.settle(a, b, ntiles);
        __syncthreads();  // every wave is done with the window and the records
        double *gsum = (double *)win;
        if (off > 0) {
            gsum[(3 * wave + 0) * kTile + lane] = hx;
            gsum[(3 * wave + 1) * kTile + lane] = hy;
            gsum[(3 * wave + 2) * kTile + lane] = hz;
        }
        if (have && wave == 0) stage(nw_.tile);
        __syncthreads();
        if (off > 0 && wave < 3) {
            const int64_t j = (int64_t)tile * kTile + lane;
            double g = gsum[wave * kTile + lane];
#pragma unroll
            for (int v = 1; v < W; ++v) g += gsum[(3 * v + wave) * kTile + lane];
            if (j < N)
                a.part[sym_slot(N, cell_l, a.cell_tasks, a.cell_offs, a.cell_tasks + off - cell * a.cell_offs) +
                       (size_t)wave * N + j] = g;
        }
        w = nw_;
    }
    if (row < N) {
        double *out = a.part + sym_slot(N, cell_l, a.cell_tasks, a.cell_offs, task);
        out[row] = fx;
        out[N + row] = fy;
        out[2 * N + row] = fz;
    }
}

// The slots of one launch onto the running sums: cell by cell, the row sums
// of its tasks, then its source sums (with the sign of the other side).  The
// last launch's reduction adds the external term (reduce_kernel's) and writes
// F for the rows asked for, in input order.
struct SymReduceArgs {
    const double *part;
    double *acc;           // running sums [3][N]
    const uint32_t *perm;  // sorted row -> input row, or null
    const double4 *jrec;   // input order
    const double *radial;
    double *F;
    int64_t N, id_min, nrows;
    int blocks, half, block_rows, cell_tasks, cell_offs, cell0, cells;
    int first, last;
    int ext_mode, radial_size;
    double ext_coeff, Rsim;
};

// One thread per row and component (blockIdx.y): at N = 16384 the slots are
// 144 deep and the row count alone would leave most CUs idle.
__global__ __launch_bounds__(256) void sym_reduce_kernel(const SymReduceArgs a) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.N) return;
    const int c = blockIdx.y;
    const int b = (int)(k / a.block_rows);
    const size_t slot = 3u * (size_t)a.N;
    const double *p = a.part + (size_t)c * a.N + k;
    double f = a.first ? 0.0 : a.acc[(size_t)c * a.N + k];
    for (int cl = 0; cl < a.cells; ++cl) {
#pragma unroll 8
        for (int t = 0; t < a.cell_tasks; ++t, p += slot) f += *p;
        const int off0 = (a.cell0 + cl) * a.cell_offs;
#pragma unroll 4
        for (int o = 0; o < a.cell_offs; ++o, p += slot) {
            const int off = off0 + o;
            // slots nobody wrote: the block's own offset, offsets past H, and
            // the half of the blocks that took the last offset as rows
            if (off == 0 || off > a.half || (2 * off == a.blocks && b < off)) continue;
            f -= *p;
        }
    }
    if (!a.last) {
        a.acc[(size_t)c * a.N + k] = f;
        return;
    }
    const int64_t r = a.perm ? (int64_t)a.perm[k] : k;
    if (r < a.id_min || r >= a.id_min + a.nrows) return;
    double g[3] = {f, f, f};
    add_external(g, a.jrec[r], a.radial, a.ext_mode, a.ext_coeff, a.Rsim, a.radial_size);
    a.F[3 * (r - a.id_min) + c] = c == 0 ? g[0] : (c == 1 ? g[1] : g[2]);
}

}  // namespace

namespace {

// Rows per lane: the moving sums, the LDS reads and the address arithmetic of
// a step are paid once per NI pairs.  2 rows measured 1.25 T evaluations/s in
// the bare loop, 4 1.41 T (128 VGPRs, 4 waves per SIMD); 8 rows (168 VGPRs, 3
// waves) 1.48 T there, but the tested loops spill and fewer tiles are far of
// a 512-row wave: 402 against 387 ms at N = 10^6.
constexpr int kSymNI = 4;
// Below this many particles the triangle of block pairs leaves too few equal
// tasks to fill the chip (N = 9000: 0.129 against 0.167 ms).
constexpr int64_t kSymMinN = 8192;
constexpr int64_t kSymMixedMinN = 14336;  // mixed (R3 N = 13000: 0.228 against 0.234 ms, 16384: 0.235 against 0.194)
constexpr int64_t kSymS1MinN = 1024;      // S1R2 with a table (N = 1536, CIC: 0.110 against 0.131 ms)
constexpr int64_t kSymT3MinN = 128;       // T3 Ewald (N = 216: 0.32 against 0.70 ms, 13^3: 0.57 against 2.8)
// Scratch the slots may take; the offsets go in as many launches as that
// needs (128 MiB: 4.5 against 4.3 ms at N = 100003, 33.2 against 31.0 ms for
// the 64^3 nearest image).
constexpr size_t kSymBytes = (size_t)256 << 20;

bool sym_variant(const EvalPlan &p) {
    if (p.variant == PV_T3_EWALD) return p.t3_ng <= kT3MaxWinNg;  // either precision
    if (p.variant == PV_S1R2_CIC || p.variant == PV_S1R2_TSC) return true;
    if (p.variant == PV_R3 || p.variant == PV_T3_NEAREST) return true;
    // mixed: the one-sided kernel wraps one axis only and is the faster and the
    // more exact (N = 524288: 84 against 90 ms, median error 9.1e-8 against 1.2e-7)
    return p.variant == PV_S1R2_NEAREST && p.precision == STEPS_PREC_FP64;
}

// Rows of a T3 Ewald workgroup: with c particles per cell column, R rows and a
// tile span about (R + 64) / c columns in y, and their stencils start on 4
// rows more (a partial column at either end).  A window of 5 planes holds
// 25 y rows (FP32 nodes: 54), 3 of them for the last stencils.  The most rows
// that share a window need the fewest copies; the fewest bands go first.
// Measured (ms, 64 / 128 / 256 / 512 rows): 24^3 (c = 3.5) 7.0 / 8.0 / 9.8 /
// 9.9, 28^3 (5.5) 14.2 / 13.2 / 18.1 / 24.6, 32^3 (8.3) 21.5 / 25.9 / 27.1 / 53,
// 40^3 (16) 71 / 62 / 68 / 75, 48^3 (28) 192 / 165 / 155 / 190, 56^3 (44) 448 /
// 383 / 361 / 349.  Mixed: 24^3 3.6 / 4.0 / 4.0, 28^3 7.6 / 6.6 / 8.4, 32^3 14.2 /
// 12.4 / 12.0 / 17.7, 40^3 48 / 40 / 37 / 36, 56^3 306 / 253 / 231 / 221.
int sym_t3_rows(const EvalPlan &p) {
    const double c = (double)p.N / ((double)p.t3_ng * p.t3_ng);
    const int row = p.precision == STEPS_PREC_MIXED ? T3Row<true>::words32 : T3Row<true>::words;
    const int starts = (kSymT3Win / 5 - 12) / row - 3;
    int best = 64;
    double fewest = INFINITY;
    for (int rows = 64; rows <= 64 * kT3Waves; rows *= 2) {
        const double bands = std::ceil(((rows + 64) / c + 4.0) / starts);
        if (bands <= kT3Bands && bands <= fewest) {
            best = rows;
            fewest = bands;
        }
    }
    return best;
}

int64_t sym_min_n(const EvalPlan &p) {
    if (p.variant == PV_T3_EWALD) return kSymT3MinN;
    if (is_s1r2_lookup(p.variant)) return kSymS1MinN;
    return p.precision == STEPS_PREC_MIXED ? kSymMixedMinN : kSymMinN;
}

struct SymShape {
    int tb, cell_tasks, cell_offs, half, cells;
};

SymShape sym_shape(const EvalPlan &p) {
    SymShape s;
    s.tb = p.sym_block_rows / kTile;
    s.cell_tasks = std::max(1, s.tb / p.sym_task_tiles);
    s.cell_offs = std::max(1, p.sym_task_tiles / s.tb);
    s.half = p.sym_blocks / 2;
    s.cells = (s.half + s.cell_offs) / s.cell_offs;  // offsets 0 .. half
    return s;
}

size_t sym_cell_bytes(const EvalPlan &p) {
    const SymShape s = sym_shape(p);
    return (size_t)(s.cell_tasks + s.cell_offs) * 3u * (size_t)p.N * sizeof(double);
}

size_t sym_acc_bytes(const EvalPlan &p) {
    return p.sym_launch_cells < p.sym_cells ? 3u * (size_t)p.N * sizeof(double) : 0;
}

struct SymKernel {
    void (*one)(const SymArgs);
    void (*packed)(const SymPack);
    unsigned threads;
};

// The kernel of an evaluation.
SymKernel sym_kernel_of(const EvalPlan &p) {
    const bool mx = p.precision == STEPS_PREC_MIXED;
    if (p.variant == PV_T3_EWALD) {
        const bool zf = p.t3_lo > 0 && p.t3_sym.mirror_z;
        auto of = [&](auto g) {
            constexpr int G = decltype(g)::value;
            constexpr unsigned T = 64 * kT3Waves;
            if (mx) return zf ? SymKernel{sym_t3_kernel<G, true, true, SymArgs>, sym_t3_kernel<G, true, true, SymPack>, T}
                              : SymKernel{sym_t3_kernel<G, true, false, SymArgs>, sym_t3_kernel<G, true, false, SymPack>, T};
            return zf ? SymKernel{sym_t3_kernel<G, false, true, SymArgs>, sym_t3_kernel<G, false, true, SymPack>, T}
                      : SymKernel{sym_t3_kernel<G, false, false, SymArgs>, sym_t3_kernel<G, false, false, SymPack>, T};
        };
        switch (p.sym_block_rows) {
        case 512: return of(IntC<1>{});
        case 256: return of(IntC<2>{});
        case 128: return of(IntC<4>{});
        default: return of(IntC<8>{});
        }
    }
    if (is_s1r2_lookup(p.variant)) {
        auto of = [&](auto v) {
            constexpr int V = decltype(v)::value;
            return mx ? SymKernel{sym_s1r2_kernel<V, true, SymArgs>, sym_s1r2_kernel<V, true, SymPack>, kBlock}
                      : SymKernel{sym_s1r2_kernel<V, false, SymArgs>, sym_s1r2_kernel<V, false, SymPack>, kBlock};
        };
        return p.variant == PV_S1R2_CIC ? of(IntC<PV_S1R2_CIC>{}) : of(IntC<PV_S1R2_TSC>{});
    }
    if (mx) {
        auto of = [&](auto v) {
            constexpr int V = decltype(v)::value;
            return p.equal_mass
                       ? SymKernel{sym_mixed_kernel<V, kSymNI, true, SymArgs>, sym_mixed_kernel<V, kSymNI, true, SymPack>, kBlock}
                       : SymKernel{sym_mixed_kernel<V, kSymNI, false, SymArgs>, sym_mixed_kernel<V, kSymNI, false, SymPack>, kBlock};
        };
        return p.variant == PV_R3 ? of(IntC<PV_R3>{}) : of(IntC<PV_T3_NEAREST>{});
    }
    auto of = [&](auto v) {
        constexpr int V = decltype(v)::value;
        return p.equal_mass ? SymKernel{sym_kernel<V, kSymNI, true, SymArgs>, sym_kernel<V, kSymNI, true, SymPack>, kBlock}
                            : SymKernel{sym_kernel<V, kSymNI, false, SymArgs>, sym_kernel<V, kSymNI, false, SymPack>, kBlock};
    };
    switch (p.variant) {
    case PV_R3: return of(IntC<PV_R3>{});
    case PV_T3_NEAREST: return of(IntC<PV_T3_NEAREST>{});
    default: return of(IntC<PV_S1R2_NEAREST>{});
    }
}

SymArgs sym_args(const EvalPlan &p, const SymBuffers &b) {
    const SymShape s = sym_shape(p);
    SymArgs a{};
    a.rec = b.rec;
    a.soft = b.soft;
    a.tiles = b.tiles;
    a.ext = b.ext;
    a.table = b.table;
    a.keys = b.keys;
    a.tab32 = b.tab32;
    a.jrel = b.jrel;
    a.tab32s = (const float2 *)b.tab32;
    a.part = b.part;
    a.k = make_scalars(p);
    a.blocks = p.sym_blocks;
    a.half = s.half;
    a.tb = s.tb;
    a.tpt = p.sym_task_tiles;
    a.cell_tasks = s.cell_tasks;
    a.cell_offs = s.cell_offs;
    return a;
}

hipError_t launch_sym_reduce(const EvalPlan &p, const SymBuffers &b, int cell0, int cells, double *F, hipStream_t st) {
    const SymShape s = sym_shape(p);
    SymReduceArgs r{};
    r.part = b.part;
    r.acc = b.part + sym_cell_bytes(p) / sizeof(double) * (size_t)p.sym_launch_cells;
    r.perm = b.perm;
    r.jrec = b.jrec;
    r.radial = p.radial;
    r.F = F;
    r.N = p.N;
    r.id_min = p.id_min;
    r.nrows = p.nrows;
    r.blocks = p.sym_blocks;
    r.half = s.half;
    r.block_rows = p.sym_block_rows;
    r.cell_tasks = s.cell_tasks;
    r.cell_offs = s.cell_offs;
    r.cell0 = cell0;
    r.cells = cells;
    r.first = cell0 == 0;
    r.last = F != nullptr;
    r.ext_mode = p.ext_mode;
    r.radial_size = p.radial_size;
    r.ext_coeff = p.ext_coeff;
    r.Rsim = p.Rsim;
    hipLaunchKernelGGL(sym_reduce_kernel, dim3((unsigned)((p.N + 255) / 256), 3), dim3(256), 0, st, r);
    return hipGetLastError();
}

// First cell of the last launch.
int sym_last_cell0(const EvalPlan &p) { return (p.sym_cells - 1) / p.sym_launch_cells * p.sym_launch_cells; }

}  // namespace

// The triangle pays when (nearly) every row is asked for: it evaluates
// N^2 / 2 pairs at ~1.45 times the cost of a one-sided pair, the one-sided
// kernel nrows N of them.
void sym_plan(EvalPlan &p) {
    p.sym = false;
    if (p.bh || p.N < sym_min_n(p) || p.N > INT32_MAX || 3 * p.nrows < 2 * p.N || !sym_variant(p)) return;
    p.sym = true;
    p.sym_block_rows = p.variant == PV_T3_EWALD ? sym_t3_rows(p)
                       : is_s1r2_lookup(p.variant) ? kBlock
                                                   : kBlock * kSymNI;
    p.sym_blocks = (int)((p.N + p.sym_block_rows - 1) / p.sym_block_rows);
    const int tb = p.sym_block_rows / kTile, offsets = p.sym_blocks / 2 + 1;
    // Tasks of several offsets where there are plenty (fewer row-sum slots),
    // of parts of an offset where there are few: at 4 workgroups a CU the chip
    // holds 1024, and twice that leaves a short last wave (at least 1100 / 2200
    // tasks, ms: R3 N = 16384 0.239 / 0.226, 30000 0.554 / 0.522, mixed 30000
    // 0.411 / 0.390, T3 nearest 32^3 0.750 / 0.727; 4400 gains nothing).
    int tiles = tb;
    if ((int64_t)p.sym_blocks * offsets >= 16384) tiles = 2 * tb;
    if ((int64_t)p.sym_blocks * offsets >= 4 * 16384) tiles = 4 * tb;
    while (tiles > 1 && tiles <= tb && (int64_t)p.sym_blocks * offsets * (tb / tiles) < 2200) tiles /= 2;
    p.sym_task_tiles = tiles;
    const SymShape s = sym_shape(p);
    p.sym_cells = s.cells;
    const size_t most = std::max(kSymBytes, (size_t)p.splits * 3u * (size_t)p.nrows * sizeof(double));
    p.sym_launch_cells = (int)std::min<size_t>((size_t)s.cells, std::max<size_t>(1, most / sym_cell_bytes(p)));
}

size_t sym_bytes(const EvalPlan &p) {
    return p.sym ? sym_cell_bytes(p) * (size_t)p.sym_launch_cells + sym_acc_bytes(p) : 0;
}

// Cells a launch with which its workgroups fill the chip once (one a CU for T3
// Ewald, whose window takes a CU's LDS, else four).  Evaluations (ms) with as
// many cells as 256 MiB hold / these / one at a time / the one-sided kernel:
// R3 N = 30000 0.43 / 0.51 / 0.70 / 0.63, 100003 3.9 / 4.5 / 6.1 / 6.2, 300000
// 32.8 / 35.4 / 57 / 46 (mixed 21.2 / 24.1 / 44 / 28.8); T3 Ewald 32^3 21.3 / 22.9
// / 22.9 / 91; S1R2 CIC N = 102400 15.6 / 20.9 / 31.9 / 44.9; T3 nearest 64^3 29.2 /
// 32.0 / 43.7 / 48.3 (mixed 30.2 / 40.5 / 99.6 / 37.2).
int sym_lean_cells(const EvalPlan &p) {
    const int fill = p.variant == PV_T3_EWALD ? 256 : 1024, each = p.sym_blocks * sym_shape(p).cell_tasks;
    return std::max(1, (fill + each - 1) / each);
}

bool sym_fit(EvalPlan &p, size_t bytes) {
    while (p.sym && scratch_bytes(p) > bytes) {
        if (p.sym_launch_cells == 1) return false;
        p.sym_launch_cells = p.sym_launch_cells > 8 ? p.sym_launch_cells * 7 / 8 : p.sym_launch_cells - 1;
    }
    return true;
}

bool masses_equal(const double *M, int64_t n) {
    for (int64_t i = 1; i < n; ++i)
        if (!(M[i] == M[0])) return false;
    return n > 0;
}

bool sym_selected(const EvalPlan &p) {
    return p.sym && (p.variant != PV_T3_EWALD || p.t3_sym.odd) && (!is_s1r2_lookup(p.variant) || p.s1r2_odd);
}

hipError_t launch_sym_pairs(const EvalPlan &p, const SymBuffers &b, hipStream_t st) {
    const SymKernel k = sym_kernel_of(p);
    SymArgs a = sym_args(p, b);
    for (int c0 = 0; c0 < p.sym_cells; c0 += p.sym_launch_cells) {
        const int cells = std::min(p.sym_launch_cells, p.sym_cells - c0);
        a.cell0 = c0;
        hipLaunchKernelGGL(k.one, dim3((unsigned)a.blocks, (unsigned)(cells * a.cell_tasks)), dim3(k.threads), 0, st, a);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess && c0 + cells < p.sym_cells) e = launch_sym_reduce(p, b, c0, cells, nullptr, st);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

const void *sym_pack_kind(const EvalPlan &p) {
    return p.sym_launch_cells >= p.sym_cells ? (const void *)sym_kernel_of(p).packed : nullptr;
}

size_t sym_desc_bytes() { return sizeof(SymSeg); }

int64_t sym_describe(const EvalPlan &p, const SymBuffers &b, void *host_descs, int idx, int64_t blk_begin) {
    SymSeg g;
    g.a = sym_args(p, b);
    g.blk_begin = (int)blk_begin;
    ((SymSeg *)host_descs)[idx] = g;
    return (int64_t)p.sym_blocks * p.sym_cells * g.a.cell_tasks;
}

hipError_t launch_sym_packed(const EvalPlan &p, const void *dev_descs, int nseg, int64_t blocks, hipStream_t st) {
    const SymKernel k = sym_kernel_of(p);
    hipLaunchKernelGGL(k.packed, dim3((unsigned)blocks), dim3(k.threads), 0, st, SymPack{(const SymSeg *)dev_descs, nseg});
    return hipGetLastError();
}

hipError_t launch_sym_finish(const EvalPlan &p, const SymBuffers &b, double *F, hipStream_t st) {
    const int c0 = sym_last_cell0(p);
    return launch_sym_reduce(p, b, c0, p.sym_cells - c0, F, st);
}

}  // namespace steps
