// pair_kernels.hip -- direct O(N^2) pair-force kernels for gfx950 (MI355X).
//
// Work decomposition (one force evaluation = rows id_min..id_max against all
// N sources, self pair included as in forces_cuda.cu:531 and forces.cc:538):
//   * a workgroup of 256 lanes (4 wave64) owns kBlockRows = 256*NI target rows,
//     NI rows per lane held in VGPRs together with their FP64 accumulators;
//   * blockIdx.y selects one of `splits` contiguous source ranges, so small N
//     still fills 256 CUs; every (row-block, split) writes its FP64 partial
//     sums to partials[split][3][nrows] and a second kernel adds the splits in
//     fixed order (deterministic, no atomics) and adds the external term;
//   * the source particle j is wave-uniform, so its record (x,y,z,m) is
//     fetched with scalar loads into SGPRs and reaches all 64 lanes as a VALU
//     scalar operand -- the broadcast costs no VALU or LDS instruction;
//   * sources are processed in tiles of 64; a tiny pre-pass stores each tile's
//     largest softening length, so one v_cmp against (h_i + h_max,tile)^2
//     replaces the per-pair h_i + h_j test, and the exact cubic-spline branch
//     (r < h_i + h_j, forces_cuda.cu:466-519, the reference's own formula)
//     runs only when some lane of the wave is that close;
//   * 1/r^3 uses v_rsq_f64 (2^-24 accurate on gfx950) plus one first-order
//     Newton correction; the R3 and nearest-image FP64 kernels read source
//     copies whose mass slot holds -1.5 m, which folds the mass into that
//     correction (mr3_scaled: 5 VALU instead of 6).
#include "pair_device.h"

#include <algorithm>
#include <cmath>

namespace steps {

namespace {

// Everything one evaluation's pair kernel reads: rows (caller order),
// sources (the same arrays for FP64; spatially ordered copies for the mixed
// path, which jrel and the tiles describe), tables, partial sums, scalars.
struct PairArgs {
    const double4 *irec;
    const double *isoft;
    const double4 *jrec;
    const double *soft;
    const float4 *jrel;
    const double4 *tiles;
    const double4 *tile_ext;  // half extents of the tiles' bounding boxes (sorted sources)
    const double4 *sub;       // centres of the 8-source sub-tiles (mixed S1R2 CIC / TSC)
    const double *table;
    const float2 *tab32;      // FP32 S1R2 table (mixed)
    const float4 *t3tab32;    // FP32 T3 table, (Dx, Dy, Dz, 0) per node (mixed)
    const uint32_t *keys;     // pencil keys of the sorted particles (T3 Ewald), else null
    double *part;
    KScalars k;
};

// One evaluation inside a packed launch: its arguments, its row-block count
// and the first flat workgroup index it owns.
struct PackSeg {
    PairArgs a;
    int nbx;
    int blk_begin;
};

// S1R2 CIC / TSC kernels: LDS for the rho rows of one source tile (39 KB:
// four workgroups per CU; 19 rows of a 128-cell z run), filled from the
// global table at each tile; a tile whose rows do not fit reads the global
// table.  The table loads otherwise co-limit these kernels on the vector-L1
// path (4 and 9 16-byte loads per pair).  At N = 524288 (cylinder, sources in
// input order): CIC 345 -> 394 and TSC 192 -> 251 G pairs/s, bitwise the same
// sums; windows of 52 KB (3 workgroups) and 26 KB (6) were slower (360 / 250,
// 390 / 225), and NGP, one load per pair, lost 15% and keeps the global reads.
constexpr int kS1R2WinNodes = 2496;

template <int V, int NI, int UNR>
__device__ __forceinline__ void body_f64(const PairArgs &a, const int bx, const int split) {
    const double4 *__restrict__ irec = a.irec;
    const double *__restrict__ isoft = a.isoft;
    const double4 *__restrict__ jrec = a.jrec;
    const double *__restrict__ soft = a.soft;
    const double4 *__restrict__ tiles = a.tiles;
    const double4 *__restrict__ ext = a.tile_ext;
    const double *__restrict__ table = a.table;
    double *__restrict__ part = a.part;
    KScalars k = a.k;
    k.c15 = in_vgpr(a.k.c15);
    const int tid = threadIdx.x;
    const int64_t row_base = (int64_t)bx * (kBlock * NI);
    const int64_t j0 = (int64_t)split * k.jchunk;  // multiple of kTile
    const int64_t j1 = min(k.N, j0 + k.jchunk);

    double xi[NI], yi[NI], zi[NI], hi[NI], fx[NI], fy[NI], fz[NI];
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int64_t r = min(row_base + q * kBlock + tid, k.nrows - 1);
        const double4 p = irec[k.id_min + r];
        xi[q] = p.x;
        yi[q] = p.y;
        zi[q] = p.z;
        hi[q] = isoft[k.id_min + r];
        fx[q] = fy[q] = fz[q] = 0.0;
    }

    // S1R2 lookup: per source tile, the rho rows every pair of the workgroup
    // can read, staged in LDS (see kS1R2WinNodes); range slots alternate
    // between tiles so that one barrier closes the atomics and the previous
    // tile's reads of the window
    constexpr bool SWIN = V == PV_S1R2_CIC || V == PV_S1R2_TSC;
    // sources carry -1.5 m (scaled_sources, mr3_scaled)
    constexpr bool MSC = V == PV_R3 || V == PV_T3_NEAREST || V == PV_S1R2_NEAREST;
    __shared__ __align__(16) double2 s1win[SWIN ? kS1R2WinNodes : 1];
    __shared__ int s1rng[4];
    if (SWIN) {
        if (tid < 4) s1rng[tid] = (tid & 1) ? INT32_MIN : INT32_MAX;
        __syncthreads();
    }

    // loop bounds in 32 bits, relative to the tile: the loop tests stay on the
    // SALU (a 64-bit signed compare would take two VALU instructions per trip)
    const int ntiles = (int)((j1 - j0 + kTile - 1) / kTile);
    for (int ti = 0; ti < ntiles; ++ti) {
        const int64_t t0 = j0 + (int64_t)ti * kTile;
        const double4 tc = tiles[t0 / kTile];
        const double hmax = tc.w;
        double B[NI];
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            const double b = hi[q] + hmax;
            B[q] = b * b;
        }
        const int cnt = (ti + 1 < ntiles) ? kTile : (int)(j1 - t0);  // sources in this tile
        const double4 *__restrict__ tj = jrec + t0;
        int u0 = 0;
        S1R2Win sw{s1win, 0, 0, false};
        if (SWIN) {
            // rho of every pair with this tile lies between the distances from
            // the row to the near and far sides of the tile's xy box; the
            // stencils read rho nodes floor(rho / drho) - 1 .. floor + 2
            const double4 te = ext[t0 / kTile];
            const double ax = fabs(xi[0] - tc.x), ay = fabs(yi[0] - tc.y);
            const double gx = fmax(ax - te.x, 0.0), gy = fmax(ay - te.y, 0.0);
            const double ex = ax + te.x, ey = ay + te.y;
            const int lo = (int)floor(fmin(sqrt(fma(gx, gx, gy * gy)) * k.inv_drho, k.last_r)) - 1;
            const int hi = (int)floor(fmin(sqrt(fma(ex, ex, ey * ey)) * k.inv_drho, k.last_r)) + 2;
            int *rg = s1rng + 2 * (ti & 1);
            atomicMin(&rg[0], lo);
            atomicMax(&rg[1], hi);
            __syncthreads();  // ranges complete; every wave is done with the previous window
            const int w0 = max(rg[0], -1), w1 = min(rg[1], k.nrho);  // ghost rows -1 and Nrho
            if (tid < 2) s1rng[2 * ((ti + 1) & 1) + tid] = tid ? INT32_MIN : INT32_MAX;  // next tile's slot
            const unsigned nz3 = (unsigned)(k.nz + 3);
            sw.w0 = w0;
            sw.nw = w1 - w0 + 1;
            sw.ok = (int64_t)sw.nw * nz3 <= kS1R2WinNodes;
            if (sw.ok) {
                const double2 *src = s1r2_row(table, k, w0);  // rows w0 .. w1 are contiguous
                const unsigned nn = (unsigned)sw.nw * nz3;
                for (unsigned o = tid; o < nn; o += kBlock) s1win[o] = src[o];
            }
            __syncthreads();  // the window is complete
        }
        if (V == PV_R3 || V == PV_T3_NEAREST || V == PV_S1R2_NEAREST) {
            // Spatially ordered sources: when the tile's bounding box lies
            // outside every lane's softening bound (B widened by 1e-9 for
            // rounding) and, for the periodic variants, every lane sees the
            // whole tile on one side of each wrap (tile_shift), its pairs are
            // the R3 pair, with fixed per-lane shifts where the tile wraps:
            // same arithmetic, no per-pair tests
            const double4 te = ext[t0 / kTile];
            bool far = true, shifted = false;
            double sx[NI], sy[NI], sz[NI];
#pragma unroll
            for (int q = 0; q < NI; ++q) {
                sx[q] = sy[q] = sz[q] = 0.0;
                if (V != PV_R3) {
                    far = far && tile_shift(zi[q], tc.z, te.z, k, sz[q]);
                    if (V == PV_T3_NEAREST)
                        far = far && tile_shift(xi[q], tc.x, te.x, k, sx[q]) && tile_shift(yi[q], tc.y, te.y, k, sy[q]);
                    shifted = shifted || sx[q] != 0.0 || sy[q] != 0.0 || sz[q] != 0.0;
                }
                far = far && box_dist2(xi[q] - sx[q], yi[q] - sy[q], zi[q] - sz[q], tc, te) > B[q] * (1.0 + 1e-9);
            }
            if (__all(far)) {
                if (V != PV_R3 && __any(shifted)) {
                    for (; u0 + UNR <= cnt; u0 += UNR) {
                        double4 pj[UNR];
#pragma unroll
                        for (int u = 0; u < UNR; ++u) pj[u] = tj[u0 + u];
#pragma unroll
                        for (int u = 0; u < UNR; ++u)
#pragma unroll
                            for (int q = 0; q < NI; ++q)
                                pair_far_shift(k, pj[u], xi[q], yi[q], zi[q], sx[q], sy[q], sz[q], fx[q], fy[q], fz[q]);
                    }
                    for (; u0 < cnt; ++u0) {
                        const double4 pj = tj[u0];
#pragma unroll
                        for (int q = 0; q < NI; ++q)
                            pair_far_shift(k, pj, xi[q], yi[q], zi[q], sx[q], sy[q], sz[q], fx[q], fy[q], fz[q]);
                    }
                    continue;
                }
                for (; u0 + UNR <= cnt; u0 += UNR) {
                    double4 pj[UNR];
#pragma unroll
                    for (int u = 0; u < UNR; ++u) pj[u] = tj[u0 + u];
#pragma unroll
                    for (int u = 0; u < UNR; ++u)
#pragma unroll
                        for (int q = 0; q < NI; ++q) pair_r3_far(k, pj[u], xi[q], yi[q], zi[q], fx[q], fy[q], fz[q]);
                }
                for (; u0 < cnt; ++u0) {
                    const double4 pj = tj[u0];
#pragma unroll
                    for (int q = 0; q < NI; ++q) pair_r3_far(k, pj, xi[q], yi[q], zi[q], fx[q], fy[q], fz[q]);
                }
                continue;
            }
        }
        for (; u0 + UNR <= cnt; u0 += UNR) {
            double4 pj[UNR];
#pragma unroll
            for (int u = 0; u < UNR; ++u) pj[u] = tj[u0 + u];
#pragma unroll
            for (int u = 0; u < UNR; ++u)
#pragma unroll
                for (int q = 0; q < NI; ++q)
                    pair_f64<V, SWIN, MSC>(k, table, soft, t0 + u0 + u, pj[u], xi[q], yi[q], zi[q], hi[q], B[q], fx[q],
                                      fy[q], fz[q], sw);
        }
        for (; u0 < cnt; ++u0) {
            const double4 pj = tj[u0];
#pragma unroll
            for (int q = 0; q < NI; ++q)
                pair_f64<V, SWIN, MSC>(k, table, soft, t0 + u0, pj, xi[q], yi[q], zi[q], hi[q], B[q], fx[q], fy[q], fz[q],
                                  sw);
        }
    }

#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int64_t r = row_base + q * kBlock + tid;
        if (r < k.nrows) {
            double *out = part + (size_t)split * 3u * (size_t)k.nrows;
            out[r] = fx[q];
            out[k.nrows + r] = fy[q];
            out[2 * k.nrows + r] = fz[q];
        }
    }
}

// ---------------------------------------------------------------------------
// mixed-precision pair kernel (R3): FP32 pair arithmetic on positions
// recentred on each 64-source tile (offsets from the tile's bounding-box
// centre, prepared once per evaluation), FP32 sums inside a tile, FP64 across
// tiles; pairs inside the softening radius are recomputed in FP64 from the
// FP64 records, so close-pair forces keep full precision.
// ---------------------------------------------------------------------------
// Rows come from (irec, isoft) in the caller's order; sources from the
// spatially ordered copies (jrec, soft) that jrel and the tiles describe.
template <int NI, int UNR>
__device__ __forceinline__ void body_mixed_r3(const PairArgs &a, const int bx, const int split) {
    const double4 *__restrict__ irec = a.irec;
    const double *__restrict__ isoft = a.isoft;
    const double4 *__restrict__ jrec = a.jrec;
    const double *__restrict__ soft = a.soft;
    const float4 *__restrict__ jrel = a.jrel;
    const double4 *__restrict__ tiles = a.tiles;
    double *__restrict__ part = a.part;
    KScalars k = a.k;
    k.c15 = in_vgpr(a.k.c15);
    const int tid = threadIdx.x;
    const int64_t row_base = (int64_t)bx * (kBlock * NI);
    const int64_t j0 = (int64_t)split * k.jchunk;  // multiple of kTile
    const int64_t j1 = min(k.N, j0 + k.jchunk);

    double xi[NI], yi[NI], zi[NI], hi[NI], fx[NI], fy[NI], fz[NI];
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int64_t r = min(row_base + q * kBlock + tid, k.nrows - 1);
        const double4 p = irec[k.id_min + r];
        xi[q] = p.x;
        yi[q] = p.y;
        zi[q] = p.z;
        hi[q] = isoft[k.id_min + r];
        fx[q] = fy[q] = fz[q] = 0.0;
    }

    const int ntiles = (int)((j1 - j0 + kTile - 1) / kTile);  // 32-bit loop bounds: SALU tests
    for (int ti = 0; ti < ntiles; ++ti) {
        const int64_t t0 = j0 + (int64_t)ti * kTile;
        const double4 c = tiles[t0 / kTile];
        float xr[NI], yr[NI], zr[NI], B[NI], ax[NI], ay[NI], az[NI];
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            xr[q] = (float)(xi[q] - c.x);
            yr[q] = (float)(yi[q] - c.y);
            zr[q] = (float)(zi[q] - c.z);
            // conservative FP32 bound: (h_i + h_max)^2 widened by 1e-5 so that
            // FP32 rounding of r2 cannot hide a pair inside the radius
            const float b = (float)((hi[q] + c.w) * (1.0 + 1e-5));
            B[q] = b * b;
            ax[q] = ay[q] = az[q] = 0.0f;
        }
        const int64_t tend = min(j1, t0 + kTile);
        const int cnt = (int)(tend - t0);
        const float4 *__restrict__ tr = jrel + t0;
        bool near = false;
        int j = 0;
        for (; j + UNR <= cnt; j += UNR) {
            float4 pj[UNR];
#pragma unroll
            for (int u = 0; u < UNR; ++u) pj[u] = tr[j + u];
#pragma unroll
            for (int u = 0; u < UNR; ++u)
#pragma unroll
                for (int q = 0; q < NI; ++q) mixed_pair(pj[u], xr[q], yr[q], zr[q], B[q], near, ax[q], ay[q], az[q]);
        }
        for (; j < cnt; ++j) {
            const float4 pj = tr[j];
#pragma unroll
            for (int q = 0; q < NI; ++q) mixed_pair(pj, xr[q], yr[q], zr[q], B[q], near, ax[q], ay[q], az[q]);
        }
        // rare: some lane had a pair within its bound -> redo those pairs in FP64
        if (__builtin_expect(near, 0)) {
            for (int64_t jj = t0; jj < tend; ++jj) {
                const float4 pr = jrel[jj];
                const double4 pd = jrec[jj];
#pragma unroll
                for (int q = 0; q < NI; ++q) {
                    const float dx = pr.x - xr[q], dy = pr.y - yr[q], dz = pr.z - zr[q];
                    const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                    if (r2 < B[q]) {
                        const double ddx = pd.x - xi[q], ddy = pd.y - yi[q], ddz = pd.z - zi[q];
                        const double rr2 = fma(ddx, ddx, fma(ddy, ddy, ddz * ddz));
                        double w = inv_r3(rr2, k.c15);
                        const double beta = hi[q] + soft[jj];
                        if (rr2 < beta * beta) w = softening_exact(sqrt(rr2), beta);
                        const double s = pd.w * w;
                        fx[q] = fma(s, ddx, fx[q]);
                        fy[q] = fma(s, ddy, fy[q]);
                        fz[q] = fma(s, ddz, fz[q]);
                    }
                }
            }
        }
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            fx[q] += (double)ax[q];
            fy[q] += (double)ay[q];
            fz[q] += (double)az[q];
        }
    }

#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int64_t r = row_base + q * kBlock + tid;
        if (r < k.nrows) {
            double *out = part + (size_t)split * 3u * (size_t)k.nrows;
            out[r] = fx[q];
            out[k.nrows + r] = fy[q];
            out[2 * k.nrows + r] = fz[q];
        }
    }
}

// ---------------------------------------------------------------------------
// mixed-precision S1xR2 kernel (nearest z-image, optionally with the tabulated
// Ewald correction): the R3 scheme -- FP32 pair arithmetic on tile-recentred
// positions, FP32 sums inside a tile, FP64 across tiles, FP64 redo of the
// pairs inside the softening bound -- with the z-image wrap in FP32 and the
// correction (D_rho, D_z) interpolated in FP32 from an FP32 copy of the table
// (forces_cuda.cu:819-863 with :188-455).
// ---------------------------------------------------------------------------
template <int V, int NI, int UNR>
__device__ __forceinline__ void body_mixed_z(const PairArgs &a, const int bx, const int split) {
    const double4 *__restrict__ irec = a.irec;
    const double *__restrict__ isoft = a.isoft;
    const double4 *__restrict__ jrec = a.jrec;
    const double *__restrict__ soft = a.soft;
    const float4 *__restrict__ jrel = a.jrel;
    const double4 *__restrict__ tiles = a.tiles;
    const double *__restrict__ table = a.table;
    const float2 *__restrict__ tab32 = a.tab32;
    const double4 *__restrict__ ext = a.tile_ext;
    double *__restrict__ part = a.part;
    KScalars k = a.k;
    k.c15 = in_vgpr(a.k.c15);
    const int tid = threadIdx.x;
    const int64_t row_base = (int64_t)bx * (kBlock * NI);
    const int64_t j0 = (int64_t)split * k.jchunk;  // multiple of kTile
    const int64_t j1 = min(k.N, j0 + k.jchunk);

    double xi[NI], yi[NI], zi[NI], hi[NI], fx[NI], fy[NI], fz[NI];
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int64_t r = min(row_base + q * kBlock + tid, k.nrows - 1);
        const double4 p = irec[k.id_min + r];
        xi[q] = p.x;
        yi[q] = p.y;
        zi[q] = p.z;
        hi[q] = isoft[k.id_min + r];
        fx[q] = fy[q] = fz[q] = 0.0;
    }

    // TSC: the rho rows of each source tile in LDS, as in body_f64 (FP32
    // nodes: 4992 of them, 39 KB, up to 38 z runs of 131), with the sources
    // in input order (xy-compact tiles on column-ordered input).  At N =
    // 524288: 300 -> 431 G pairs/s, pair-sum p99 error 1.5e-5 -> 2.0e-5
    // (comoving term included).  CIC kept Morton tiles and global reads:
    // with the window it ran at 582 against 681.
    constexpr bool SWIN = V == PV_S1R2_TSC;
    constexpr bool SUBT = V == PV_S1R2_CIC || V == PV_S1R2_TSC;  // sub_tiles(): jrel per 8-source sub-tile
    __shared__ __align__(16) float2 s1win[SWIN ? 2 * kS1R2WinNodes : 1];
    __shared__ int s1rng[4];
    if (SWIN) {
        if (tid < 4) s1rng[tid] = (tid & 1) ? INT32_MIN : INT32_MAX;
        __syncthreads();
    }

    const int ntiles = (int)((j1 - j0 + kTile - 1) / kTile);  // 32-bit loop bounds: SALU tests
    for (int ti = 0; ti < ntiles; ++ti) {
        const int64_t t0 = j0 + (int64_t)ti * kTile;
        const double4 c = tiles[t0 / kTile];
        // each row's image nearest the tile centre on the periodic axes, so
        // that a close pair across the box edge rounds like any close pair
        // (the per-pair wrap below then fires only for distant pairs)
        double xw[NI], yw[NI], zw[NI];
        float xr[NI], yr[NI], zr[NI], B[NI], ax[NI], ay[NI], az[NI];
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            xw[q] = xi[q];
            yw[q] = yi[q];
            zw[q] = zi[q];
            if (V == PV_T3_NEAREST) {
                xw[q] = near_image(xw[q], c.x, k);
                yw[q] = near_image(yw[q], c.y, k);
            }
            zw[q] = near_image(zw[q], c.z, k);
            xr[q] = (float)(xw[q] - c.x);
            yr[q] = (float)(yw[q] - c.y);
            zr[q] = (float)(zw[q] - c.z);
            const float b = (float)((hi[q] + c.w) * (1.0 + 1e-5));
            B[q] = b * b;
            ax[q] = ay[q] = az[q] = 0.0f;
        }
        const int64_t tend = min(j1, t0 + kTile);
        const int cnt = (int)(tend - t0);
        const float4 *__restrict__ tr = jrel + t0;
        S1R2Win32 sw{s1win, 0, 0, false};
        if (SWIN) {
            static_assert(!SWIN || NI == 1, "one row per lane");
            const double4 te = ext[t0 / kTile];
            const double axd = fabs(xi[0] - c.x), ayd = fabs(yi[0] - c.y);
            const double gx = fmax(axd - te.x, 0.0), gy = fmax(ayd - te.y, 0.0);
            const double ex = axd + te.x, ey = ayd + te.y;
            const int lo = (int)floor(fmin(sqrt(fma(gx, gx, gy * gy)) * k.inv_drho, k.last_r)) - 1;
            const int hi = (int)floor(fmin(sqrt(fma(ex, ex, ey * ey)) * k.inv_drho, k.last_r)) + 2;
            int *rg = s1rng + 2 * (ti & 1);
            atomicMin(&rg[0], lo);
            atomicMax(&rg[1], hi);
            __syncthreads();  // ranges complete; every wave is done with the previous window
            const int w0 = max(rg[0], -1), w1 = min(rg[1], k.nrho);
            if (tid < 2) s1rng[2 * ((ti + 1) & 1) + tid] = tid ? INT32_MIN : INT32_MAX;  // next tile's slot
            const unsigned nz3 = (unsigned)(k.nz + 3);
            sw.w0 = w0;
            sw.nw = w1 - w0 + 1;
            sw.ok = (int64_t)sw.nw * nz3 <= 2 * kS1R2WinNodes;
            if (sw.ok) {
                const float2 *src = s1r2_row32(tab32, k, w0);
                const unsigned nn = (unsigned)sw.nw * nz3;
                for (unsigned o = tid; o < nn; o += kBlock) s1win[o] = src[o];
            }
            __syncthreads();  // the window is complete
        }
        if (V == PV_S1R2_NEAREST || V == PV_T3_NEAREST) {
            // Far tile (decided in FP64, with margins far above the FP32
            // rounding of the displacements): every lane sees the whole tile
            // on one side of each wrap and outside 1.001 x its bound
            constexpr bool XY = V == PV_T3_NEAREST;
            const double4 te = ext[t0 / kTile];
            bool far = true, shifted = false;
            float sx[NI], sy[NI], sz[NI];
#pragma unroll
            for (int q = 0; q < NI; ++q) {
                double hx = 0.0, hy = 0.0, hz = 0.0;
                far = far && tile_shift(zw[q], c.z, te.z, k, hz, 1e-5);
                if (XY)
                    far = far && tile_shift(xw[q], c.x, te.x, k, hx, 1e-5) && tile_shift(yw[q], c.y, te.y, k, hy, 1e-5);
                far = far && box_dist2(xw[q] - hx, yw[q] - hy, zw[q] - hz, c, te) > (double)B[q] * (1.0 + 1e-3);
                sx[q] = (float)hx;  // 0, -L or +L: (float)(-L) is -Lf
                sy[q] = (float)hy;
                sz[q] = (float)hz;
                shifted = shifted || hx != 0.0 || hy != 0.0 || hz != 0.0;
            }
            if (__all(far)) {
                if (__any(shifted))
                    mixed_far_tile_z<true, XY, XY, NI, UNR>(tr, cnt, xr, yr, zr, sx, sy, sz, ax, ay, az, fx, fy, fz);
                else
                    mixed_far_tile_z<false, XY, XY, NI, UNR>(tr, cnt, xr, yr, zr, sx, sy, sz, ax, ay, az, fx, fy, fz);
#pragma unroll
                for (int q = 0; q < NI; ++q) {
                    fx[q] += (double)ax[q];
                    fy[q] += (double)ay[q];
                    fz[q] += (double)az[q];
                }
                continue;
            }
        }
        if (SUBT) {
            // S1R2 CIC / TSC: per sub-tile of kSub sources, the row's FP32
            // offset from the sub-tile's centre (its z image nearest that
            // centre) and FP32 sums over kSub pairs, added to the FP64
            // accumulators after each sub-tile.  Against whole-tile offsets
            // and sums this cut the error against FP64 at N = 524288 with the
            // comoving term (CIC p99 1.5e-5 -> 8.9e-6, TSC 2.0e-5 -> 9.2e-6;
            // the TSC tiles span half the box in z, so their offsets carried
            // ulp(Lz/4)), for 4-7% of the speed (1.76x / 1.64x FP64).
            for (int s0 = 0; s0 < cnt; s0 += kSub) {
                const int scnt = min(kSub, cnt - s0);
                const double4 cs = a.sub[(t0 + s0) / kSub];
                float xs[NI], ys[NI], zs[NI];
#pragma unroll
                for (int q = 0; q < NI; ++q) {
                    xs[q] = (float)(xi[q] - cs.x);
                    ys[q] = (float)(yi[q] - cs.y);
                    zs[q] = (float)(near_image(zi[q], cs.z, k) - cs.z);
                    ax[q] = ay[q] = az[q] = 0.0f;
                }
                const float4 *__restrict__ ts = tr + s0;
                bool near = false;
                if (scnt == kSub) {
#pragma unroll
                    for (int j = 0; j < kSub; j += UNR) {
                        float4 pj[UNR];
#pragma unroll
                        for (int u = 0; u < UNR; ++u) pj[u] = ts[j + u];
#pragma unroll
                        for (int u = 0; u < UNR; ++u)
#pragma unroll
                            for (int q = 0; q < NI; ++q)
                                mixed_pair_z<V, SWIN>(k, tab32, pj[u], xs[q], ys[q], zs[q], B[q], near, ax[q], ay[q],
                                                      az[q], sw);
                    }
                } else {
                    for (int j = 0; j < scnt; ++j) {
                        const float4 pj = ts[j];
#pragma unroll
                        for (int q = 0; q < NI; ++q)
                            mixed_pair_z<V, SWIN>(k, tab32, pj, xs[q], ys[q], zs[q], B[q], near, ax[q], ay[q], az[q],
                                                  sw);
                    }
                }
                if (__builtin_expect(near, 0)) {
                    for (int jj = 0; jj < scnt; ++jj) {
                        const float4 pr = ts[jj];
#pragma unroll
                        for (int q = 0; q < NI; ++q) {
                            float dx, dy, dz;
                            bool bnd;
                            if (mixed_r2_z<V>(k, pr, xs[q], ys[q], zs[q], dx, dy, dz, bnd) < B[q] || bnd) {
                                const double b = hi[q] + c.w;
                                const int64_t jg = t0 + s0 + jj;
                                pair_f64<V>(k, table, soft, jg, jrec[jg], xi[q], yi[q], zi[q], hi[q], b * b, fx[q],
                                            fy[q], fz[q]);
                            }
                        }
                    }
                }
#pragma unroll
                for (int q = 0; q < NI; ++q) {
                    fx[q] += (double)ax[q];
                    fy[q] += (double)ay[q];
                    fz[q] += (double)az[q];
                }
            }
            continue;
        }
        bool near = false;
        int j = 0;
        for (; j + UNR <= cnt; j += UNR) {
            float4 pj[UNR];
#pragma unroll
            for (int u = 0; u < UNR; ++u) pj[u] = tr[j + u];
#pragma unroll
            for (int u = 0; u < UNR; ++u)
#pragma unroll
                for (int q = 0; q < NI; ++q)
                    mixed_pair_z<V, SWIN>(k, tab32, pj[u], xr[q], yr[q], zr[q], B[q], near, ax[q], ay[q], az[q], sw);
        }
        for (; j < cnt; ++j) {
            const float4 pj = tr[j];
#pragma unroll
            for (int q = 0; q < NI; ++q)
                mixed_pair_z<V, SWIN>(k, tab32, pj, xr[q], yr[q], zr[q], B[q], near, ax[q], ay[q], az[q], sw);
        }
        if (__builtin_expect(near, 0)) {
            for (int64_t jj = t0; jj < tend; ++jj) {
                const float4 pr = jrel[jj];
#pragma unroll
                for (int q = 0; q < NI; ++q) {
                    float dx, dy, dz;
                    bool bnd;
                    if (mixed_r2_z<V>(k, pr, xr[q], yr[q], zr[q], dx, dy, dz, bnd) < B[q] || bnd) {
                        const double b = hi[q] + c.w;
                        pair_f64<V>(k, table, soft, jj, jrec[jj], xi[q], yi[q], zi[q], hi[q], b * b, fx[q],
                                    fy[q], fz[q]);
                    }
                }
            }
        }
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            fx[q] += (double)ax[q];
            fy[q] += (double)ay[q];
            fz[q] += (double)az[q];
        }
    }

#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int64_t r = row_base + q * kBlock + tid;
        if (r < k.nrows) {
            double *out = part + (size_t)split * 3u * (size_t)k.nrows;
            out[r] = fx[q];
            out[k.nrows + r] = fy[q];
            out[2 * k.nrows + r] = fz[q];
        }
    }
}

// ---------------------------------------------------------------------------
// kernels: one evaluation per launch (grid row-blocks x splits), or several
// evaluations of one variant packed into one launch (flat grid, each
// workgroup finds its evaluation among at most kMaxPack segments)
// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// T3 Ewald pair kernel with a table window in LDS.  Rows and sources are in z
// pencils (order_kernels.hip: key = cell column (x, y), then z), so a
// workgroup's 256 rows cover a few adjacent cell columns and one run of
// sources covers one column.  The table rows that any of their stencils can
// reach then form a small (x, y) window of full z runs (5 x 9 rows of the
// folded 63^3 table: 70 KB; serpentine pencils keep the workgroups that
// cross a column change to 6 x 8).  At each change of source column the workgroup
// copies that window into LDS between two barriers (the source loop is the
// same for every wave, so both barriers are reached by all); each pair then
// reads its 16 stencil rows from LDS, which feeds 128 B per clock against the
// 64 B per clock of the vector-L1 path the global reads take.  A lane whose
// stencil leaves the window (a coordinate rounded across a cell edge) reads
// that pair from global memory, and a window that does not fit (workgroups
// whose rows wrap around the box) leaves the whole run on the global path, so
// every read stays in bounds.  Same arithmetic on the same values as the
// global kernel: the sums are bitwise equal.
// ---------------------------------------------------------------------------
constexpr int kT3WinDoubles = 10080;  // 78.75 KB of LDS per workgroup: two workgroups per CU
                                      // (a 6 x 8 window of 63^3 rows)
__device__ __forceinline__ void body_t3_win(const PairArgs &a, const int bx, const int split) {
    __shared__ __align__(16) double win[kT3WinDoubles];
    __shared__ int brange[4];
    const double4 *__restrict__ irec = a.irec;
    const double *__restrict__ isoft = a.isoft;
    const double4 *__restrict__ jrec = a.jrec;
    const double *__restrict__ soft = a.soft;
    const double4 *__restrict__ tiles = a.tiles;
    const double *__restrict__ table = a.table;
    const uint32_t *__restrict__ keys = a.keys;
    KScalars k = a.k;
    k.c15 = in_vgpr(a.k.c15);
    const int tid = threadIdx.x;
    const int64_t row_base = (int64_t)bx * kBlock;
    const int64_t j0 = (int64_t)split * k.jchunk;  // multiple of kTile
    const int64_t j1 = min(k.N, j0 + k.jchunk);
    // rows are the sorted particles (id_min = 0, nrows = N)
    const int64_t r = min(row_base + tid, k.nrows - 1);
    const double4 p = irec[r];
    const double xi = p.x, yi = p.y, zi = p.z, hi = isoft[r];
    double fx = 0.0, fy = 0.0, fz = 0.0;
    const uint32_t kr = keys[r];
    if (tid == 0) {
        brange[0] = INT32_MAX;
        brange[1] = -1;
        brange[2] = INT32_MAX;
        brange[3] = -1;
    }
    __syncthreads();
    const int rbx = (int)(kr >> 20), rby = pencil_y(kr, k.ng);
    atomicMin(&brange[0], rbx);
    atomicMax(&brange[1], rbx);
    atomicMin(&brange[2], rby);
    atomicMax(&brange[3], rby);
    __syncthreads();
    const int bxmin = brange[0], bxmax = brange[1], bymin = brange[2], bymax = brange[3];
    const int Ng = k.ng, lo = k.t3_lo;
    const unsigned NY = (unsigned)(Ng - lo), NZ = (unsigned)(Ng + 3), NZ3 = 3u * NZ, WS = t3_win_stride(NZ3 + 2u);

    int cur = -1;  // cell column of the sources the window was built for
    bool wok = false;
    int fx0 = 0, nxw = 0, fy0 = 0, nyw = 0;
    const int ntiles = (int)((j1 - j0 + kTile - 1) / kTile);  // 32-bit loop bounds: SALU tests
    for (int ti = 0; ti < ntiles; ++ti) {
        const int64_t t0 = j0 + (int64_t)ti * kTile;
        const double b = hi + tiles[t0 / kTile].w;
        const double B = b * b;
        const int cnt = (int)min((int64_t)kTile, j1 - t0);
        for (int u = 0; u < cnt; ++u) {
            const int64_t j = t0 + u;
            const uint32_t kj = keys[j];
            const int pk = (int)(kj >> 10);
            if (pk != cur) {
                cur = pk;
                wok = t3_win_axis(pk >> 10, pk >> 10, bxmin, bxmax, Ng, lo, fx0, nxw) &&
                      t3_win_axis(pencil_y(kj, Ng), pencil_y(kj, Ng), bymin, bymax, Ng, lo, fy0, nyw) &&
                      (int64_t)nxw * nyw * WS <= kT3WinDoubles;
                __syncthreads();  // every wave is done with the previous window
                if (wok) {
                    for (int wa = 0; wa < nxw; ++wa)
                        for (int wc = 0; wc < nyw; ++wc) {
                            const double *src = table + ((unsigned)(fx0 + wa) * NY + (unsigned)(fy0 + wc)) * NZ3;
                            double *dst = win + (unsigned)(wa * nyw + wc) * WS;
                            for (unsigned o = tid; o < NZ3 + 2u; o += kBlock) {
                                if (o < NZ3) {
                                    const unsigned z = o / 3u, c = o - 3u * z;
                                    dst[c < 2u ? 2u * z + c : 2u * NZ + z] = src[o];
                                } else {
                                    dst[o] = 0.0;  // the two pad entries after the z run
                                }
                            }
                        }
                }
                __syncthreads();  // the window is complete
            }
            const double4 pj = jrec[j];
            double dx = pj.x - xi, dy = pj.y - yi, dz = pj.z - zi;
            // forces_cuda.cu:622-627: d - L*d/|d| when |d| > L/2
            if (fabs(dx) > k.halfL) dx -= copysign(k.L, dx);
            if (fabs(dy) > k.halfL) dy -= copysign(k.L, dy);
            if (fabs(dz) > k.halfL) dz -= copysign(k.L, dz);
            const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
            const double w = pair_w_tile(r2, B, hi, soft, j, k);
            T3Stencil st;
            t3_stencil(k, dx, dy, dz, st);
            bool in = wok;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                in = in && (st.mx[q] - (unsigned)fx0 < (unsigned)nxw) && (st.my[q] - (unsigned)fy0 < (unsigned)nyw);
            double Dx, Dy, Dz;
            if (in) {
                const bool odd = (st.iz0 & 1) != 0;
                const double wz5[5] = {odd ? 0.0 : st.wz[0], odd ? st.wz[0] : st.wz[1], odd ? st.wz[1] : st.wz[2],
                                       odd ? st.wz[2] : st.wz[3], odd ? st.wz[3] : 0.0};
                const unsigned za = 2u * NZ + ((unsigned)st.iz0 & ~1u);
                t3_contract_win(
                    st, wz5,
                    [&](int i, int jj, double *vxy, double *vz) {
                        const double *w0 =
                            win + ((st.mx[i] - (unsigned)fx0) * (unsigned)nyw + (st.my[jj] - (unsigned)fy0)) * WS;
                        const double2 *xy = (const double2 *)w0 + st.iz0;  // 16-byte aligned (x, y) nodes
                        const double2 *zz = (const double2 *)(w0 + za);    // 16-byte aligned z pairs
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const double2 a = xy[q];
                            vxy[2 * q] = a.x;
                            vxy[2 * q + 1] = a.y;
                        }
#pragma unroll
                        for (int h = 0; h < 3; ++h) {
                            const double2 b = zz[h];
                            vz[2 * h] = b.x;
                            vz[2 * h + 1] = b.y;
                        }
                    },
                    Dx, Dy, Dz);
            }
            else
                t3_contract(
                    st,
                    [&](int i, int jj, double *v) {
                        t3_load_aos(table + ((st.mx[i] * NY + st.my[jj]) * NZ + (unsigned)st.iz0) * 3u, v);
                    },
                    Dx, Dy, Dz);
            fx = fma(pj.w, fma(w, dx, -Dx), fx);
            fy = fma(pj.w, fma(w, dy, -Dy), fy);
            fz = fma(pj.w, fma(w, dz, -Dz), fz);
        }
    }
    const int64_t rr = row_base + tid;
    if (rr < k.nrows) {
        double *out = a.part + (size_t)split * 3u * (size_t)k.nrows;
        out[rr] = fx;
        out[k.nrows + rr] = fy;
        out[2 * k.nrows + rr] = fz;
    }
}

// ---------------------------------------------------------------------------
// T3 Ewald pair kernel for tables larger than an XCD's L2 (the folded 127^3
// table of IS_PERIODIC = 3 is 12.8 MB against 4 MB of L2 per XCD), with rows
// and sources in z pencils.  The source columns (table cell columns in x)
// are dealt out to the eight XCDs by the table x nodes their pairs read: for
// the row block's first x column c0, XCD k takes the source columns whose
// displacement column (c - c0 + Ng/2) mod Ng lies in [k Ng/8, (k+1) Ng/8), so
// the pairs an XCD evaluates read one slab of the table (~20 x nodes of 127:
// ~4 MB), which its L2 can hold, instead of all of it.  Workgroups are
// dispatched to the XCDs round robin, so workgroup id = 8 * row block + k
// runs on XCD k; its sums are split k of the row block's partial sums (eight
// splits, reduced in fixed order).  Every source column falls in exactly one
// slab, so each pair is evaluated once; the pair arithmetic is pair_f64's.
// ---------------------------------------------------------------------------
constexpr int kXcds = 8;

// first index of the sorted keys at or above v (scalar binary search)
__device__ __forceinline__ int64_t keys_lower_bound(const uint32_t *__restrict__ keys, int64_t n, uint32_t v) {
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (keys[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ void body_t3_slab(const PairArgs &a, const int id) {
    const int bx = id / kXcds, slab = id % kXcds;
    const double4 *__restrict__ irec = a.irec;
    const double *__restrict__ isoft = a.isoft;
    const double4 *__restrict__ jrec = a.jrec;
    const double *__restrict__ soft = a.soft;
    const double4 *__restrict__ tiles = a.tiles;
    const double *__restrict__ table = a.table;
    const uint32_t *__restrict__ keys = a.keys;
    KScalars k = a.k;
    k.c15 = in_vgpr(a.k.c15);
    const int tid = threadIdx.x;
    const int64_t row_base = (int64_t)bx * kBlock;
    // rows are the sorted particles (id_min = 0, nrows = N)
    const int64_t r = min(row_base + tid, k.nrows - 1);
    const double4 p = irec[r];
    const double xi = p.x, yi = p.y, zi = p.z, hi = isoft[r];
    double fx = 0.0, fy = 0.0, fz = 0.0;
    const int Ng = k.ng;
    const int c0 = (int)(keys[row_base] >> 20);  // x column of the block's first row
    const int lo_k = slab * Ng / kXcds, hi_k = (slab + 1) * Ng / kXcds;
    const int cs = imodp(c0 - Ng / 2 + lo_k, Ng), ncol = hi_k - lo_k;
    for (int part = 0; part < 2; ++part) {
        // source columns [ca, cb): the slab's columns, in two runs where they wrap
        const int ca = part == 0 ? cs : 0;
        const int cb = part == 0 ? min(Ng, cs + ncol) : cs + ncol - Ng;
        if (cb <= ca) continue;
        const int64_t j0 = keys_lower_bound(keys, k.N, (uint32_t)ca << 20);
        const int64_t j1 = (cb >= Ng) ? k.N : keys_lower_bound(keys, k.N, (uint32_t)cb << 20);
        for (int64_t t0 = (j0 / kTile) * kTile; t0 < j1; t0 += kTile) {
            const double b = hi + tiles[t0 / kTile].w;
            const double B = b * b;
            const int u0 = (int)(max(j0, t0) - t0), u1 = (int)(min(j1, t0 + kTile) - t0);
            const double4 *__restrict__ tj = jrec + t0;
            for (int u = u0; u < u1; ++u)
                pair_f64<PV_T3_EWALD>(k, table, soft, t0 + u, tj[u], xi, yi, zi, hi, B, fx, fy, fz);
        }
    }
    const int64_t rr = row_base + tid;
    if (rr < k.nrows) {
        double *out = a.part + (size_t)slab * 3u * (size_t)k.nrows;
        out[rr] = fx;
        out[k.nrows + rr] = fy;
        out[2 * k.nrows + rr] = fz;
    }
}

// ---------------------------------------------------------------------------
// Mixed-precision T3 Ewald pair kernel.  Each displacement is formed and
// wrapped in FP64 (forces_cuda.cu:620-627) and rounded to FP32 once: the
// sources are in z pencils, whose 64-source tiles span the box in z, so
// tile-recentred FP32 positions would carry errors of ulp(L/2) on close
// pairs.  r^2, r^-3 and the tricubic correction are FP32, the correction read
// from an FP32 copy of the device table with one 16-byte (Dx, Dy, Dz, 0) word
// per node, so a stencil row is four aligned 16-byte reads.  Pairs within
// 1.00001 x the softening bound are zeroed in FP32 and redone in FP64 (FP64
// table); FP32 sums run over one 64-source tile and are added to FP64
// accumulators.  WIN: rows and sources in pencils and the table window of
// body_t3_win staged in LDS (16 bytes a node: at most 3264 nodes, 51 KB,
// three workgroups per CU); a lane whose stencil leaves the window reads the
// global FP32 table, so both forms give the same sums bitwise.  With every
// workgroup on the window it is bound by LDS bank conflicts like the FP64
// kernel (33 against 34 G pairs/s at 64^3); a third of the workgroups on the
// global table takes it to 38-39.
// ---------------------------------------------------------------------------
constexpr int kT3WinNodes32 = 3264;
// Row blocks with bx % 3 < 2 use the window and the others read the global
// FP32 table, so that the LDS and the vector-L1 path both carry taps: at 64^3
// 38-39 G pairs/s, against 33.1 with every block on the window (LDS-bound) and
// 26.0 with none (vector-L1-bound).  Shares of 4/7, 5/7 and 7/9 measured 38.0,
// 37.7 and 37.3; shares over an even count (1/2, 3/4) left the global blocks
// on a few XCDs and ran at 26.  Rows padded to 256 bytes ran at 31.5.
constexpr unsigned kT3WinNum32 = 2u, kT3WinDen32 = 3u;

template <bool WIN>
__device__ __forceinline__ void body_t3_mixed(const PairArgs &a, const int bx, const int split) {
    __shared__ __align__(16) float4 win[WIN ? kT3WinNodes32 : 1];
    __shared__ int brange[4];
    const double4 *__restrict__ irec = a.irec;
    const double *__restrict__ isoft = a.isoft;
    const double4 *__restrict__ jrec = a.jrec;
    const double *__restrict__ soft = a.soft;
    const double4 *__restrict__ tiles = a.tiles;
    const double *__restrict__ table = a.table;
    const float4 *__restrict__ T32 = a.t3tab32;
    const uint32_t *__restrict__ keys = a.keys;
    KScalars k = a.k;
    k.c15 = in_vgpr(a.k.c15);
    const int tid = threadIdx.x;
    const int64_t row_base = (int64_t)bx * kBlock;
    const int64_t j0 = (int64_t)split * k.jchunk;  // multiple of kTile
    const int64_t j1 = min(k.N, j0 + k.jchunk);
    const int64_t r = min(row_base + tid, k.nrows - 1);
    const double4 p = irec[k.id_min + r];
    const double xi = p.x, yi = p.y, zi = p.z, hi = isoft[k.id_min + r];
    double fx = 0.0, fy = 0.0, fz = 0.0;
    const int Ng = k.ng, lo = k.t3_lo;
    const unsigned NY = (unsigned)(Ng - lo), NZ = (unsigned)(Ng + 3);
    int bxmin = 0, bxmax = 0, bymin = 0, bymax = 0;
    const bool win_share = (unsigned)bx % kT3WinDen32 < kT3WinNum32;
    if (WIN) {
        // rows are the sorted particles (id_min = 0, nrows = N)
        if (tid == 0) {
            brange[0] = INT32_MAX;
            brange[1] = -1;
            brange[2] = INT32_MAX;
            brange[3] = -1;
        }
        __syncthreads();
        const uint32_t kr = keys[r];
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

    int cur = -1;  // cell column of the sources the window was built for
    bool wok = false;
    int fx0 = 0, nxw = 0, fy0 = 0, nyw = 0;
    const int ntiles = (int)((j1 - j0 + kTile - 1) / kTile);  // 32-bit loop bounds: SALU tests
    for (int ti = 0; ti < ntiles; ++ti) {
        const int64_t t0 = j0 + (int64_t)ti * kTile;
        const double hb = hi + tiles[t0 / kTile].w;
        const float bf = (float)(hb * (1.0 + 1e-5));
        const float B = bf * bf;
        const int cnt = (int)min((int64_t)kTile, j1 - t0);
        float ax = 0.0f, ay = 0.0f, az = 0.0f;
        bool near = false;
        for (int u = 0; u < cnt; ++u) {
            const int64_t j = t0 + u;
            if (WIN) {
                const uint32_t kj = keys[j];
                const int pk = (int)(kj >> 10);
                if (pk != cur) {  // the same for every wave: both barriers are reached by all
                    cur = pk;
                    wok = win_share && t3_win_axis(pk >> 10, pk >> 10, bxmin, bxmax, Ng, lo, fx0, nxw) &&
                          t3_win_axis(pencil_y(kj, Ng), pencil_y(kj, Ng), bymin, bymax, Ng, lo, fy0, nyw) &&
                          (int64_t)nxw * nyw * NZ <= kT3WinNodes32;
                    __syncthreads();  // every wave is done with the previous window
                    if (wok) {
                        const unsigned nn = (unsigned)(nxw * nyw) * NZ;
                        for (unsigned o = tid; o < nn; o += kBlock) {
                            const unsigned row = o / NZ, z = o - row * NZ;
                            const unsigned wa = row / (unsigned)nyw, wc = row - wa * (unsigned)nyw;
                            win[o] = T32[(((unsigned)fx0 + wa) * NY + (unsigned)fy0 + wc) * NZ + z];
                        }
                    }
                    __syncthreads();  // the window is complete
                }
            }
            const double4 pj = jrec[j];
            float dx, dy, dz;
            const float r2 = t3_mixed_disp(k, pj, xi, yi, zi, dx, dy, dz);
            const bool nr = r2 < B;  // left to the FP64 redo (r2 may be 0 here)
            near = near || nr;
            const float y = __builtin_amdgcn_rsqf(r2);
            const float y3 = nr ? 0.0f : (y * y) * y;
            const float m = nr ? 0.0f : (float)pj.w;
            T3Stencil32 st;
            t3_stencil_f32(k, dx, dy, dz, st);
            bool in = WIN && wok;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                in = in && (st.mx[q] - (unsigned)fx0 < (unsigned)nxw) && (st.my[q] - (unsigned)fy0 < (unsigned)nyw);
            float Dx, Dy, Dz;
            if (in)
                t3_contract_f32(
                    st,
                    [&](int i, int jj, float4 *n) {
                        const float4 *w0 =
                            win + ((st.mx[i] - (unsigned)fx0) * (unsigned)nyw + (st.my[jj] - (unsigned)fy0)) * NZ +
                            (unsigned)st.iz0;
#pragma unroll
                        for (int q = 0; q < 4; ++q) n[q] = w0[q];
                    },
                    Dx, Dy, Dz);
            else
                t3_contract_f32(
                    st,
                    [&](int i, int jj, float4 *n) {
                        const float4 *g = T32 + (st.mx[i] * NY + st.my[jj]) * NZ + (unsigned)st.iz0;
#pragma unroll
                        for (int q = 0; q < 4; ++q) n[q] = g[q];
                    },
                    Dx, Dy, Dz);
            ax = fmaf(m, fmaf(y3, dx, -Dx), ax);
            ay = fmaf(m, fmaf(y3, dy, -Dy), ay);
            az = fmaf(m, fmaf(y3, dz, -Dz), az);
        }
        if (__builtin_expect(near, 0)) {
            for (int u = 0; u < cnt; ++u) {
                const int64_t jj = t0 + u;
                const double4 pj = jrec[jj];
                float dx, dy, dz;
                if (t3_mixed_disp(k, pj, xi, yi, zi, dx, dy, dz) < B)
                    pair_f64<PV_T3_EWALD>(k, table, soft, jj, pj, xi, yi, zi, hi, hb * hb, fx, fy, fz);
            }
        }
        fx += (double)ax;
        fy += (double)ay;
        fz += (double)az;
    }
    const int64_t rr = row_base + tid;
    if (rr < k.nrows) {
        double *out = a.part + (size_t)split * 3u * (size_t)k.nrows;
        out[rr] = fx;
        out[k.nrows + rr] = fy;
        out[2 * k.nrows + rr] = fz;
    }
}

enum BodyKind : int { BK_F64 = 0, BK_MIXED_R3 = 1, BK_MIXED_Z = 2, BK_T3_WIN = 3, BK_T3_MIXED = 4, BK_T3_WIN_MIXED = 5,
                      BK_T3_SLAB = 6 };

template <int BK, int V, int NI, int UNR>
__device__ __forceinline__ void run_body(const PairArgs &a, int bx, int by) {
    if (BK == BK_F64) body_f64<V, NI, UNR>(a, bx, by);
    else if (BK == BK_T3_WIN) body_t3_win(a, bx, by);
    else if (BK == BK_T3_SLAB) body_t3_slab(a, bx);
    else if (BK == BK_T3_MIXED) body_t3_mixed<false>(a, bx, by);
    else if (BK == BK_T3_WIN_MIXED) body_t3_mixed<true>(a, bx, by);
    else if (BK == BK_MIXED_R3) body_mixed_r3<NI, UNR>(a, bx, by);
    else body_mixed_z<V, NI, UNR>(a, bx, by);
}

// The mixed R3 kernel is held to 80 VGPRs (6 waves per SIMD; no spills),
// 1% faster than the 84 the compiler picks on its own (measured at N = 2^21).
// The mixed S1R2 nearest-image kernel is held to 128 (4 waves): 6% faster
// than at its own 132 VGPRs and 3 waves (N = 524288); the mixed T3 one (one
// row per lane) to 80 (6 waves; 52 bytes of spills, still 5% faster than
// at 4 waves).  The
// mixed T3 window kernel is held to 168 (3 waves, which its 51 KB of LDS
// allows).
template <int BK, int V, int NI, int UNR>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(
    (BK == BK_MIXED_R3 || (BK == BK_F64 && (V == PV_T3_NEAREST || V == PV_S1R2_NEAREST)))
        ? 6
        : ((BK == BK_MIXED_Z && (V == PV_S1R2_NEAREST || V == PV_T3_NEAREST)) ? (V == PV_T3_NEAREST ? 6 : 4)
                                                                                : (BK == BK_T3_WIN_MIXED ? 3 : 1)))))
void pair_kernel(const PairArgs a) {
    run_body<BK, V, NI, UNR>(a, blockIdx.x, blockIdx.y);
}

template <int BK, int V, int NI, int UNR>
__global__ __launch_bounds__(kBlock) void pair_kernel_packed(const PackSeg *__restrict__ segs, int nseg) {
    const int b = blockIdx.x;
    int s = 0;
    for (int q = 1; q < nseg; ++q)
        if (segs[q].blk_begin <= b) s = q;
    const PackSeg &g = segs[s];
    const int local = b - g.blk_begin;
    run_body<BK, V, NI, UNR>(g.a, local % g.nbx, local / g.nbx);
}

__global__ void table_f32_kernel(const double *__restrict__ T, float2 *__restrict__ T32, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) T32[i] = make_float2((float)T[2 * i], (float)T[2 * i + 1]);
}

// T3 device layout (three doubles a node) to 16-byte FP32 nodes (Dx, Dy, Dz, 0).
__global__ void t3_f32_kernel(const double *__restrict__ T, float4 *__restrict__ T32, int64_t nodes) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nodes) T32[i] = make_float4((float)T[3 * i], (float)T[3 * i + 1], (float)T[3 * i + 2], 0.0f);
}

// ---------------------------------------------------------------------------
// fixed-order reduction of the splits + external term, AoS output
// ---------------------------------------------------------------------------
// perm (or null): partial-sum row r belongs to input row perm[r] (rows taken
// in spatial order; id_min is 0 then).
__global__ __launch_bounds__(64) void reduce_kernel(const double *__restrict__ part,
                                                     const double4 *__restrict__ jrec,
                                                     const uint32_t *__restrict__ perm,
                                                     const double *__restrict__ radial,
                                                     double *__restrict__ F, int64_t nrows,
                                                     int64_t id_min, int splits, int ext_mode,
                                                     double ext_coeff, double Rsim,
                                                     int radial_size) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nrows) return;
    const int64_t r = perm ? (int64_t)perm[k] : k;  // output row
    double f[3] = {0.0, 0.0, 0.0};
    // Bound by the latency of its loads where there are few rows, so those of
    // kAhead splits are on the way at once and a workgroup has 64 rows (47
    // splits of N = 3000: 17 us one split after another, 8.0 ahead, 6.2 with 64
    // rows instead of 256); the additions stay in split order
    constexpr int kAhead = 8;
    for (int s0 = 0; s0 < splits; s0 += kAhead) {
        double v[kAhead][3];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const double *p = part + (size_t)min(s0 + u, splits - 1) * 3u * (size_t)nrows + k;
#pragma unroll
            for (int c = 0; c < 3; ++c) v[u][c] = p[(size_t)c * (size_t)nrows];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
#pragma unroll
            for (int c = 0; c < 3; ++c) f[c] = s0 + u < splits ? f[c] + v[u][c] : f[c];
    }
    add_external(f, jrec[id_min + r], radial, ext_mode, ext_coeff, Rsim, radial_size);
    F[3 * r + 0] = f[0];
    F[3 * r + 1] = f[1];
    F[3 * r + 2] = f[2];
}

// ---------------------------------------------------------------------------
// layout kernels
// ---------------------------------------------------------------------------
__global__ void pack_kernel(const double *__restrict__ x, const double *__restrict__ M,
                            const double *__restrict__ h, double4 *__restrict__ jrec,
                            double *__restrict__ soft, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    jrec[i] = make_double4(x[3 * i], x[3 * i + 1], x[3 * i + 2], M[i]);
    soft[i] = h[i];
}

__global__ void pack_positions_kernel(const double *__restrict__ x, double4 *__restrict__ jrec,
                                      int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double m = jrec[i].w;
    jrec[i] = make_double4(x[3 * i], x[3 * i + 1], x[3 * i + 2], m);
}

__global__ __launch_bounds__(256) void check_finite_kernel(const double *__restrict__ x, int64_t count,
                                                           int *__restrict__ flag) {
    bool bad = false;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
        bad = bad || !isfinite(x[i]);
    if (bad) *flag = 1;
}

__global__ void unpack_positions_kernel(const double4 *__restrict__ jrec, double *__restrict__ x,
                                        int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double4 p = jrec[i];
    x[3 * i] = p.x;
    x[3 * i + 1] = p.y;
    x[3 * i + 2] = p.z;
}

// One wave64 per source tile: the tile's bounding-box centre and largest
// softening length (double4 (cx, cy, cz, h_max)); with MIXED also the FP32
// offsets of each source from that centre plus its mass.  A non-null `scaled`
// receives each source as (x, y, z, -1.5 m), the records mr3_scaled reads; it
// may be jrec itself (each lane reads its record before it stores, and the
// padding lanes that re-read the first record of a tile store nothing).
template <bool MIXED, bool SUB = false>
__global__ __launch_bounds__(kTile) void tiles_kernel(const double4 *jrec,
                                                     const double *__restrict__ soft,
                                                     double4 *__restrict__ tiles,
                                                     float4 *__restrict__ jrel, double4 *__restrict__ ext,
                                                     double4 *scaled, double4 *__restrict__ sub, int64_t n) {
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x;
    const int64_t i = t * kTile + lane;
    const bool ok = i < n;
    // padding lanes repeat the first source of their sub-tile, or of the tile
    // (t*kTile < n) when the whole sub-tile is padding
    const int64_t g0 = i - (lane % kSub);
    const int64_t src = ok ? i : (g0 < n ? g0 : t * kTile);
    const double4 p = jrec[src];
    double lo[3] = {p.x, p.y, p.z}, hi[3] = {p.x, p.y, p.z};
    double hm = soft[src];
#pragma unroll
    for (int m = kTile / 2; m > 0; m >>= 1) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = fmin(lo[a], __shfl_xor(lo[a], m, kTile));
            hi[a] = fmax(hi[a], __shfl_xor(hi[a], m, kTile));
        }
        hm = fmax(hm, __shfl_xor(hm, m, kTile));
    }
    const double cx = 0.5 * (lo[0] + hi[0]), cy = 0.5 * (lo[1] + hi[1]), cz = 0.5 * (lo[2] + hi[2]);
    if (lane == 0) tiles[t] = make_double4(cx, cy, cz, hm);
    // half extents, rounded up so that centre +- extent contains every source
    if (ext && lane == 0)
        ext[t] = make_double4((hi[0] - lo[0]) * (0.5 + 1e-15), (hi[1] - lo[1]) * (0.5 + 1e-15),
                              (hi[2] - lo[2]) * (0.5 + 1e-15), 0.0);
    if (MIXED && !SUB && ok)
        jrel[i] = make_float4((float)(p.x - cx), (float)(p.y - cy), (float)(p.z - cz), (float)p.w);
    if (SUB) {
        // the bounding-box centre of each group of kSub consecutive sources,
        // and each source's FP32 offset from its group's centre
        double sl[3] = {p.x, p.y, p.z}, sh[3] = {p.x, p.y, p.z};
#pragma unroll
        for (int m = kSub / 2; m > 0; m >>= 1)
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                sl[a] = fmin(sl[a], __shfl_xor(sl[a], m, kTile));
                sh[a] = fmax(sh[a], __shfl_xor(sh[a], m, kTile));
            }
        const double sx = 0.5 * (sl[0] + sh[0]), sy = 0.5 * (sl[1] + sh[1]), sz = 0.5 * (sl[2] + sh[2]);
        if (ok && lane % kSub == 0) sub[i / kSub] = make_double4(sx, sy, sz, 0.0);
        if (ok) jrel[i] = make_float4((float)(p.x - sx), (float)(p.y - sy), (float)(p.z - sz), (float)p.w);
    }
    if (scaled && ok) scaled[i] = make_double4(p.x, p.y, p.z, -1.5 * p.w);
}

// Sources per inner-loop step (scalar-loaded together), chosen by measurement
// on the N = 2^21 R3 workload together with the rows per lane: FP64 1 row x 4
// sources (80 VGPRs, 6 waves per SIMD), mixed 2 rows x 8 sources.
constexpr int unroll_of(int v, int precision) {
    return precision == STEPS_PREC_MIXED ? ((v == PV_R3 || v == PV_S1R2_NEAREST || v == PV_T3_NEAREST) ? 8 : 2)
                                         : ((v == PV_R3 || v == PV_T3_NEAREST || v == PV_S1R2_NEAREST) ? 4 : 1);
}

template <int BK, int V>
hipError_t launch_pair_t(const PairArgs *a, const PackSeg *segs, int nseg, unsigned gx, unsigned gy,
                         hipStream_t st) {
    constexpr int prec = (BK == BK_F64 || BK == BK_T3_WIN || BK == BK_T3_SLAB) ? STEPS_PREC_FP64 : STEPS_PREC_MIXED;
    constexpr int NI = rows_per_lane(V, prec);
    constexpr int UNR = unroll_of(V, prec);
    if (segs)
        hipLaunchKernelGGL((pair_kernel_packed<BK, V, NI, UNR>), dim3(gx), dim3(kBlock), 0, st, segs, nseg);
    else
        hipLaunchKernelGGL((pair_kernel<BK, V, NI, UNR>), dim3(gx, gy), dim3(kBlock), 0, st, *a);
    return hipGetLastError();
}

// Runtime (variant, precision) -> kernel instantiation; one evaluation (a)
// on a gx x gy grid, or nseg packed evaluations (segs, device) on gx blocks.
hipError_t launch_pair(int variant, int precision, const PairArgs *a, const PackSeg *segs, int nseg, unsigned gx,
                       unsigned gy, hipStream_t st) {
    if (precision == STEPS_PREC_MIXED) {
        switch (variant) {
        case PV_R3: return launch_pair_t<BK_MIXED_R3, PV_R3>(a, segs, nseg, gx, gy, st);
        case PV_T3_NEAREST: return launch_pair_t<BK_MIXED_Z, PV_T3_NEAREST>(a, segs, nseg, gx, gy, st);
        case PV_T3_EWALD: return launch_pair_t<BK_T3_MIXED, PV_T3_EWALD>(a, segs, nseg, gx, gy, st);
        case PV_S1R2_NEAREST: return launch_pair_t<BK_MIXED_Z, PV_S1R2_NEAREST>(a, segs, nseg, gx, gy, st);
        case PV_S1R2_CIC: return launch_pair_t<BK_MIXED_Z, PV_S1R2_CIC>(a, segs, nseg, gx, gy, st);
        case PV_S1R2_TSC: return launch_pair_t<BK_MIXED_Z, PV_S1R2_TSC>(a, segs, nseg, gx, gy, st);
        default: return hipErrorInvalidValue;
        }
    }
    switch (variant) {
    case PV_R3: return launch_pair_t<BK_F64, PV_R3>(a, segs, nseg, gx, gy, st);
    case PV_T3_NEAREST: return launch_pair_t<BK_F64, PV_T3_NEAREST>(a, segs, nseg, gx, gy, st);
    case PV_T3_EWALD: return launch_pair_t<BK_F64, PV_T3_EWALD>(a, segs, nseg, gx, gy, st);
    case PV_S1R2_NEAREST: return launch_pair_t<BK_F64, PV_S1R2_NEAREST>(a, segs, nseg, gx, gy, st);
    case PV_S1R2_NGP: return launch_pair_t<BK_F64, PV_S1R2_NGP>(a, segs, nseg, gx, gy, st);
    case PV_S1R2_CIC: return launch_pair_t<BK_F64, PV_S1R2_CIC>(a, segs, nseg, gx, gy, st);
    case PV_S1R2_TSC: return launch_pair_t<BK_F64, PV_S1R2_TSC>(a, segs, nseg, gx, gy, st);
    case PV_S1R2_IMAGES: return launch_pair_t<BK_F64, PV_S1R2_IMAGES>(a, segs, nseg, gx, gy, st);
    default: return hipErrorInvalidValue;
    }
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

bool is_mixed(const EvalPlan &p) { return p.precision == STEPS_PREC_MIXED && mixed_supported(p.variant); }

// The mixed kernels read spatially ordered sources (Morton order; their FP32
// offsets need compact tiles) except the S1R2 TSC one, whose table window
// needs tiles compact in xy (input order), and the R3 one below N = 65536; the R3 and
// nearest-image FP64 kernels from N = 65536 on (their far-tile test gains 7%
// for R3 at N = 2^21); the T3 Ewald kernel sources in z pencils.  Below
// N = 65536 the ~16 launches of the ordering cost more than the pair kernels
// save: the mixed R3 force at N = 16384 took 0.32-0.34 ms with it against
// 0.24-0.25 ms for FP64.
constexpr int64_t kR3SortMinN = 65536;
bool sorted_sources(const EvalPlan &p) {
    const bool far_tiles = p.variant == PV_R3 || p.variant == PV_T3_NEAREST || p.variant == PV_S1R2_NEAREST;
    // pair-symmetric S1R2 table kernels take rows and sources in input order
    if (is_s1r2_lookup(p.variant) && sym_selected(p)) return false;
    const bool mixed_sorted = is_mixed(p) && p.variant != PV_S1R2_TSC && !(p.variant == PV_R3 && p.N < kR3SortMinN);
    return mixed_sorted || (far_tiles && p.N >= kR3SortMinN) || p.variant == PV_T3_EWALD;
}
bool pencil_order(const EvalPlan &p) { return p.variant == PV_T3_EWALD; }
// The mixed S1R2 CIC / TSC kernels take their FP32 source offsets relative to
// the centres of 8-source sub-tiles (tiles_kernel<true, true>).
bool sub_tiles(const EvalPlan &p) {
    return is_mixed(p) && (p.variant == PV_S1R2_CIC || p.variant == PV_S1R2_TSC);
}
size_t sub_bytes(const EvalPlan &p) {
    return align256((size_t)std::max<int64_t>((p.N + kSub - 1) / kSub, 1) * sizeof(double4));
}
// The FP64 R3 and nearest-image kernels read source records whose mass slot
// holds -1.5 m (mr3_scaled): the sorted copy, scaled in place, or a scaled
// copy of the input-order records.
bool scaled_sources(const EvalPlan &p) {
    return !is_mixed(p) && (p.variant == PV_R3 || p.variant == PV_T3_NEAREST || p.variant == PV_S1R2_NEAREST);
}
// The T3 Ewald kernel also takes its rows in that order when it evaluates
// every particle, and so do the nearest-image FP64 kernels (Morton order: a
// wave's rows then sit in one small region, so whole tiles pass the far /
// no-wrap test; in input order a wave of a lattice spans the box); the
// reduction scatters the sums back to input order.
bool sorted_rows(const EvalPlan &p) {
    const bool nearest = p.variant == PV_T3_NEAREST || p.variant == PV_S1R2_NEAREST;
    return (pencil_order(p) || nearest) && sorted_sources(p) && p.id_min == 0 && p.nrows == p.N;
}
// The LDS-window T3 kernel needs rows in pencils and room for a 5 x 5 window
// of full z runs (Ng <= 127); packed launches keep the global kernel.  On
// finer tables a workgroup's 256 rows span many more table columns, its
// windows rarely fit and it ran slower than the global kernel (127^3 table
// on the 64^3 lattice: 5.67 against 5.87 G pairs/s), so it serves Ng <= 100.
bool t3_window(const EvalPlan &p) {
    return p.variant == PV_T3_EWALD && sorted_rows(p) && !is_mixed(p) && p.t3_ng <= 100 &&
           (int64_t)t3_win_stride(3u * (unsigned)(p.t3_ng + 3) + 2u) * 25 <= kT3WinDoubles;
}
// The same for the mixed T3 kernel (16-byte nodes; Ng <= 127).
bool t3_window_mixed(const EvalPlan &p) {
    return p.variant == PV_T3_EWALD && sorted_rows(p) && is_mixed(p) &&
           (int64_t)(p.t3_ng + 3) * 25 <= kT3WinNodes32;
}

// The XCD-slab T3 kernel (body_t3_slab) takes the tables the window does not
// serve, up to Ng = 160 (a slab of the folded table: Ng/8 + 4 x nodes of
// (Ng - Ng/2) y nodes x (Ng + 3) z nodes x 24 bytes, 4.4 MB at Ng = 127), for
// full evaluations of at least 4096 particles (eight non-empty splits).
}  // namespace
bool t3_slab_plan(const EvalPlan &p) {
    return p.variant == PV_T3_EWALD && p.precision == STEPS_PREC_FP64 && p.t3_ng > 100 && p.t3_ng <= 160 &&
           p.id_min == 0 && p.nrows == p.N && p.N >= 4096;
}
namespace {
bool t3_slab(const EvalPlan &p) { return t3_slab_plan(p) && sorted_rows(p) && p.splits == kXcds; }

size_t s1r2_f32_entries(const EvalPlan &p) {
    return (is_mixed(p) && is_s1r2_lookup(p.variant)) ? s1r2_device_nodes(p.s1r2_nrho, p.s1r2_nz) : 0;
}
// Nodes of the FP32 T3 table of the mixed kernel (one float4 each), sized for
// the unfolded layout so that the scratch size does not depend on the table.
size_t t3_f32_nodes(const EvalPlan &p) {
    return (is_mixed(p) && p.variant == PV_T3_EWALD) ? t3_device_entries(p.t3_ng, 0) / 3 : 0;
}
// Bytes of the FP32 table copy of a mixed table kernel (S1R2 or T3).
size_t table32_bytes(const EvalPlan &p) {
    return std::max(s1r2_f32_entries(p) * sizeof(float2), t3_f32_nodes(p) * sizeof(float4));
}

// Pieces of an evaluation's scratch buffer, in the order tile_extra_bytes
// counts them.
struct ScratchView {
    double *part;
    double4 *tiles;
    double4 *tile_ext;
    double4 *sub;
    float4 *jrel;
    float2 *tab32;
    double4 *jrec_s;
    double *soft_s;
    void *order;
};

ScratchView scratch_view(const EvalPlan &p, double *partials) {
    ScratchView v;
    const int64_t nt = (p.N + kTile - 1) / kTile;
    const size_t n = (size_t)std::max<int64_t>(p.N, 1);
    const size_t tb = align256((size_t)std::max<int64_t>(nt, 1) * sizeof(double4));
    v.part = partials;
    v.tiles = (double4 *)((char *)partials + align256(partial_bytes(p)));
    v.tile_ext = (double4 *)((char *)v.tiles + tb);
    v.sub = (double4 *)((char *)v.tile_ext + tb);
    v.jrel = (float4 *)((char *)v.sub + sub_bytes(p));
    v.tab32 = (float2 *)((char *)v.jrel + align256(n * sizeof(float4)));
    v.jrec_s = (double4 *)((char *)v.tab32 + align256(table32_bytes(p)));
    v.soft_s = (double *)((char *)v.jrec_s + align256(n * sizeof(double4)));
    v.order = (char *)v.soft_s + align256(n * sizeof(double));
    return v;
}

PairArgs make_args(const EvalPlan &p, const DeviceParticles &dp, const ScratchView &v) {
    PairArgs a{};
    const bool sorted = sorted_sources(p);
    a.irec = sorted_rows(p) ? v.jrec_s : dp.jrec;
    a.isoft = sorted_rows(p) ? v.soft_s : dp.soft;
    a.jrec = (sorted || scaled_sources(p)) ? v.jrec_s : dp.jrec;
    a.soft = sorted ? v.soft_s : dp.soft;
    a.jrel = v.jrel;
    a.tiles = v.tiles;
    a.tile_ext = v.tile_ext;
    a.sub = v.sub;
    a.table = (p.variant == PV_T3_EWALD) ? p.t3 : (is_s1r2_lookup(p.variant) ? p.s1r2 : nullptr);
    a.tab32 = v.tab32;
    a.t3tab32 = (const float4 *)v.tab32;  // the same scratch region: one mixed table per evaluation
    a.keys = (sorted && pencil_order(p)) ? spatial_order_keys(v.order, p.N) : nullptr;
    a.part = v.part;
    a.k = make_scalars(p);
    return a;
}

// What the pair-symmetric kernels read and write (launch_sym_pairs / _finish).
SymBuffers sym_buffers(const EvalPlan &p, const DeviceParticles &dp, double *partials) {
    const ScratchView v = scratch_view(p, partials);
    const PairArgs a = make_args(p, dp, v);
    const bool sorted = sorted_sources(p);
    return SymBuffers{a.jrec, a.soft, a.tiles, a.tile_ext, a.table, a.t3tab32, a.jrel, a.keys,
                      sorted ? spatial_order_perm(v.order, p.N) : nullptr, dp.jrec, v.part};
}

unsigned row_blocks(const EvalPlan &p) {
    const int64_t rpb = (int64_t)kBlock * rows_per_lane(p.variant, p.precision);
    return (unsigned)((p.nrows + rpb - 1) / rpb);
}

bool has_pairs(const EvalPlan &p) { return p.nrows > 0 && p.N > 0; }

}  // namespace

// The reference table is antisymmetric in each axis (ewald_space.cc:288-383
// fills it from one O_h wedge): the node mirrored in x, Ng-1-ix, holds
// (-Tx, Ty, Tz), likewise in y.  Components that vanish by symmetry (Tx on
// the plane x = 0, Ty on y = 0) hold rounding noise instead of zero
// (|T| ~ 1e-22 against max|T| ~ 4e-4 for the 63^3 table); two such entries
// count as equal when both are below 2^-52 max|T|.  The plane a mirror maps
// onto itself (odd Ng) is read directly, never negated.  The fold is used
// only when every node passes, so a folded read differs from the stored
// value by at most 2^-51 max|T|, and only in a component that vanishes by
// symmetry.
static bool t3_antisymmetric_xy(const double *T, int ng) {
    const size_t n = (size_t)ng;
    double tmax = 0.0;
    for (size_t i = 0; i < n * n * n * 3u; ++i) tmax = std::max(tmax, std::fabs(T[i]));
    if (!(tmax < INFINITY)) return false;  // NaN or infinite entries: no fold
    const double eps0 = std::ldexp(tmax, -52);
    auto same = [eps0](double b, double a) {
        return b == a || (std::fabs(a) <= eps0 && std::fabs(b) <= eps0);
    };
    auto at = [&](size_t ix, size_t iy, size_t iz) { return T + ((ix * n + iy) * n + iz) * 3u; };
    for (size_t ix = 0; ix < n; ++ix)
        for (size_t iy = 0; iy < n; ++iy)
            for (size_t iz = 0; iz < n; ++iz) {
                const double *a = at(ix, iy, iz), *bx = at(n - 1 - ix, iy, iz), *by = at(ix, n - 1 - iy, iz);
                if (!((2 * ix + 1 == n || same(bx[0], -a[0])) && same(bx[1], a[1]) && same(bx[2], a[2])))
                    return false;
                if (!(same(by[0], a[0]) && (2 * iy + 1 == n || same(by[1], -a[1])) && same(by[2], a[2])))
                    return false;
            }
    return true;
}

T3Symmetry t3_symmetry(const double *T, int ng) {
    T3Symmetry s;
    const size_t n = (size_t)ng, n3 = n * n * n;
    // eight running maxima: a one-shot call with a new table waits for this
    double top[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    size_t k = 0;
    for (; k + 8 <= n3 * 3u; k += 8)
        for (int l = 0; l < 8; ++l) top[l] = std::max(top[l], std::fabs(T[k + l]));
    for (; k < n3 * 3u; ++k) top[0] = std::max(top[0], std::fabs(T[k]));
    const double tmax = *std::max_element(top, top + 8);
    if (!(tmax < INFINITY)) return s;
    const double eps0 = std::ldexp(tmax, -52);
    auto differ = [eps0](double b, double a) {
        return !(b == a) & !((std::fabs(a) <= eps0) & (std::fabs(b) <= eps0));
    };
    bool bad = false;
    for (size_t i = 0; 2 * i < n3; ++i) {  // node n3 - 1 - i is node i seen through the centre
        const double *a = T + 3u * i, *b = T + 3u * (n3 - 1 - i);
        bad |= differ(b[0], -a[0]) | differ(b[1], -a[1]) | differ(b[2], -a[2]);
    }
    if (bad) return s;
    s.odd = true;
    for (const double *row = T; row < T + 3u * n3; row += 3u * n)
        for (size_t z = 0; 2 * z < n; ++z) {
            const double *a = row + 3u * z, *b = row + 3u * (n - 1 - z);
            bad |= differ(b[0], a[0]) | differ(b[1], a[1]) | differ(b[2], -a[2]);
        }
    s.mirror_z = !bad;
    return s;
}

int t3_layout_lo(const double *T, int ng) { return t3_antisymmetric_xy(T, ng) ? ng / 2 : 0; }

int t3_device_layout(const double *T, int ng, std::vector<double> &out) {
    const int lo = t3_layout_lo(T, ng);
    const size_t n = (size_t)ng, nx = (size_t)(ng - lo), nz = n + 3;
    out.resize(t3_device_entries(ng, lo));
    for (size_t mx = 0; mx < nx; ++mx)
        for (size_t my = 0; my < nx; ++my) {
            const double *src = T + (((size_t)lo + mx) * n + (size_t)lo + my) * n * 3u;
            double *dst = out.data() + (mx * nx + my) * nz * 3u;
            for (size_t z = 0; z < nz; ++z) {
                const size_t iz = (z + n - 1) % n;  // layout z = node z + 1, periodic
                for (int c = 0; c < 3; ++c) dst[z * 3 + c] = src[iz * 3 + c];
            }
        }
    return lo;
}

bool s1r2_table_odd(const double *T, int nrho, int nz, double L, double Rsim) {
    double tmax = 0.0;
    for (size_t i = 0; i < (size_t)nrho * nz * 2u; ++i) tmax = std::max(tmax, std::fabs(T[i]));
    if (!(tmax < INFINITY)) return false;
    const double ulp16 = std::ldexp(1.0, -49), drho = kRadialExtent * Rsim / (double)std::max(1, nrho - 1);
    for (int ir = 0; ir < nrho; ++ir)
        for (int iz = 0; 2 * iz < nz; ++iz) {
            const double *a = T + ((size_t)ir * nz + iz) * 2u, *b = T + ((size_t)ir * nz + (nz - 1 - iz)) * 2u;
            const double rho = ir * drho, z = ((double)iz + 0.5) * (L / nz) - 0.5 * L, r2 = rho * rho + z * z;
            const double tol = ulp16 * std::max(tmax, r2 > 0.0 ? 1.0 / r2 : 0.0);
            if (!(std::fabs(a[0] - b[0]) <= tol && std::fabs(a[1] + b[1]) <= tol)) return false;
        }
    return true;
}

void s1r2_device_layout(const double *T, int nrho, int nz, std::vector<double> &out) {
    const size_t nr = (size_t)nrho + 2, nzl = (size_t)nz + 3;
    out.resize(nr * nzl * 2u);
    for (size_t r = 0; r < nr; ++r) {
        const size_t ir = std::min<size_t>(r == 0 ? 0 : r - 1, (size_t)nrho - 1);  // clamped edges
        for (size_t z = 0; z < nzl; ++z) {
            const size_t iz = (z + (size_t)nz - 1) % (size_t)nz;  // entry z holds z node z - 1, periodic
            const double *src = T + (ir * (size_t)nz + iz) * 2u;  // reference layout [(ir*Nz + iz)*2 + c]
            out[(r * nzl + z) * 2u] = src[0];
            out[(r * nzl + z) * 2u + 1] = src[1];
        }
    }
}

size_t partial_bytes(const EvalPlan &p) {
    return std::max((size_t)p.splits * 3u * (size_t)std::max<int64_t>(p.nrows, 1) * sizeof(double), sym_bytes(p));
}

// Scratch after the partial sums (same buffer, 256-byte aligned pieces, in
// ScratchView order): tiles and their half extents [ceil(N/64)] double4; for
// spatially ordered sources (mixed path, R3) also jrel [N] float4, the FP32
// S1R2 table [nrho*nz] float2, the ordered copies (jrec_s double4 [N],
// soft_s double [N]) and the ordering's own scratch.
size_t tile_extra_bytes(const EvalPlan &p) {
    const int64_t nt = (p.N + kTile - 1) / kTile;
    const size_t n = (size_t)std::max<int64_t>(p.N, 1);
    size_t b = 2 * align256((size_t)std::max<int64_t>(nt, 1) * sizeof(double4)) + sub_bytes(p);
    if (sorted_sources(p) || is_mixed(p) || scaled_sources(p)) {  // FP32 records relative to the tiles, FP32 table
        b += align256(n * sizeof(float4));
        b += align256(table32_bytes(p));
    }
    if (sorted_sources(p) || scaled_sources(p)) b += align256(n * sizeof(double4)) + align256(n * sizeof(double));
    if (sorted_sources(p)) {
        b += align256(order_scratch_bytes(p.N));
    }
    return b + 256;
}

hipError_t launch_forces_prepare(const EvalPlan &p, const DeviceParticles &dp, double *partials,
                                 hipStream_t st) {
    if (p.bh) return hipErrorInvalidValue;  // launch_forces runs the octree whole
    if (!has_pairs(p)) return hipSuccess;
    const ScratchView v = scratch_view(p, partials);
    const unsigned nt = (unsigned)((p.N + kTile - 1) / kTile);
    hipError_t e;
    const int64_t n32 = (int64_t)s1r2_f32_entries(p);
    if (n32 > 0) {
        hipLaunchKernelGGL(table_f32_kernel, dim3((unsigned)((n32 + 255) / 256)), dim3(256), 0, st, p.s1r2,
                           v.tab32, n32);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if (t3_f32_nodes(p) > 0) {
        const int64_t nodes = (int64_t)(t3_device_entries(p.t3_ng, p.t3_lo) / 3);  // the layout in use
        hipLaunchKernelGGL(t3_f32_kernel, dim3((unsigned)((nodes + 255) / 256)), dim3(256), 0, st, p.t3,
                           (float4 *)v.tab32, nodes);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if (sorted_sources(p)) {
        if ((e = launch_spatial_order(dp.jrec, dp.soft, p.N, v.order, v.jrec_s, v.soft_s, st,
                                      pencil_order(p) ? p.L : 0.0, pencil_order(p) ? p.t3_ng : 0)) != hipSuccess)
            return e;
        double4 *scaled = scaled_sources(p) ? v.jrec_s : nullptr;  // in place
        if (sub_tiles(p))
            hipLaunchKernelGGL((tiles_kernel<true, true>), dim3(nt), dim3(kTile), 0, st, v.jrec_s, v.soft_s, v.tiles,
                               v.jrel, v.tile_ext, scaled, v.sub, p.N);
        else if (is_mixed(p))
            hipLaunchKernelGGL((tiles_kernel<true>), dim3(nt), dim3(kTile), 0, st, v.jrec_s, v.soft_s, v.tiles,
                               v.jrel, v.tile_ext, scaled, v.sub, p.N);
        else
            hipLaunchKernelGGL((tiles_kernel<false>), dim3(nt), dim3(kTile), 0, st, v.jrec_s, v.soft_s, v.tiles,
                               v.jrel, v.tile_ext, scaled, v.sub, p.N);
    } else {
        // tile extents too: the R3 kernel's far-tile test reads them (on unsorted
        // tiles it rarely passes, and the per-pair loop runs), and so do the
        // S1R2 table windows; the mixed TSC kernel takes its FP32 records
        // relative to input-order tiles
        double4 *scaled = scaled_sources(p) ? v.jrec_s : nullptr;
        if (sub_tiles(p))
            hipLaunchKernelGGL((tiles_kernel<true, true>), dim3(nt), dim3(kTile), 0, st, dp.jrec, dp.soft, v.tiles,
                               v.jrel, v.tile_ext, scaled, v.sub, p.N);
        else if (is_mixed(p))
            hipLaunchKernelGGL((tiles_kernel<true>), dim3(nt), dim3(kTile), 0, st, dp.jrec, dp.soft, v.tiles, v.jrel,
                               v.tile_ext, scaled, v.sub, p.N);
        else
            hipLaunchKernelGGL((tiles_kernel<false>), dim3(nt), dim3(kTile), 0, st, dp.jrec, dp.soft, v.tiles,
                               v.jrel, v.tile_ext, scaled, v.sub, p.N);
    }
    return hipGetLastError();
}

hipError_t launch_forces_pairs(const EvalPlan &p, const DeviceParticles &dp, double *partials, hipStream_t st) {
    if (!has_pairs(p)) return hipSuccess;
    if (sym_selected(p)) return launch_sym_pairs(p, sym_buffers(p, dp, partials), st);
    const PairArgs a = make_args(p, dp, scratch_view(p, partials));
    if (t3_window(p)) return launch_pair_t<BK_T3_WIN, PV_T3_EWALD>(&a, nullptr, 0, row_blocks(p), (unsigned)p.splits, st);
    if (t3_slab(p)) return launch_pair_t<BK_T3_SLAB, PV_T3_EWALD>(&a, nullptr, 0, row_blocks(p) * kXcds, 1, st);
    if (t3_window_mixed(p))
        return launch_pair_t<BK_T3_WIN_MIXED, PV_T3_EWALD>(&a, nullptr, 0, row_blocks(p), (unsigned)p.splits, st);
    return launch_pair(p.variant, is_mixed(p) ? STEPS_PREC_MIXED : STEPS_PREC_FP64, &a, nullptr, 0, row_blocks(p),
                       (unsigned)p.splits, st);
}

hipError_t launch_forces_finish(const EvalPlan &p, const DeviceParticles &dp, double *partials, double *F,
                                hipStream_t st) {
    if (p.nrows <= 0) return hipSuccess;
    if (sym_selected(p)) return launch_sym_finish(p, sym_buffers(p, dp, partials), F, st);
    const int splits = (p.N > 0) ? p.splits : 0;
    const uint32_t *perm =
        (sorted_rows(p) && has_pairs(p)) ? spatial_order_perm(scratch_view(p, partials).order, p.N) : nullptr;
    hipLaunchKernelGGL(reduce_kernel, dim3((unsigned)((p.nrows + 63) / 64)), dim3(64), 0, st, partials,
                       dp.jrec, perm, p.radial, F, p.nrows, p.id_min, splits, p.ext_mode, p.ext_coeff, p.Rsim,
                       p.radial_size);
    return hipGetLastError();
}

hipError_t launch_forces(const EvalPlan &p, const DeviceParticles &dp, double *partials, double *F, hipStream_t st,
                         hipEvent_t ev_begin, hipEvent_t ev_pair_end, hipEvent_t ev_end) {
    hipError_t e;
    if (p.bh) {  // tree build and traversal between the first two events
        if (ev_begin && (e = hipEventRecord(ev_begin, st)) != hipSuccess) return e;
        if ((e = launch_bh_forces(p, dp, partials, F, st, nullptr)) != hipSuccess) return e;
        if (ev_pair_end && (e = hipEventRecord(ev_pair_end, st)) != hipSuccess) return e;
        if (ev_end && (e = hipEventRecord(ev_end, st)) != hipSuccess) return e;
        return hipSuccess;
    }
    if ((e = launch_forces_prepare(p, dp, partials, st)) != hipSuccess) return e;
    if (ev_begin && (e = hipEventRecord(ev_begin, st)) != hipSuccess) return e;
    if ((e = launch_forces_pairs(p, dp, partials, st)) != hipSuccess) return e;
    if (ev_pair_end && (e = hipEventRecord(ev_pair_end, st)) != hipSuccess) return e;
    if ((e = launch_forces_finish(p, dp, partials, F, st)) != hipSuccess) return e;
    if (ev_end && (e = hipEventRecord(ev_end, st)) != hipSuccess) return e;
    return hipSuccess;
}

size_t pack_desc_bytes() { return (std::max(sizeof(PackSeg), sym_desc_bytes()) + 15) & ~(size_t)15; }

const void *pack_kind(const EvalPlan &p) {
    static const char one_sided = 0;  // the group's variant and precision say which kernel
    if (!has_pairs(p)) return nullptr;
    return sym_selected(p) ? sym_pack_kind(p) : &one_sided;
}

int64_t pack_describe(const EvalPlan &p, const DeviceParticles &dp, double *partials, void *host_descs, int idx,
                      int64_t blk_begin) {
    if (sym_selected(p)) return sym_describe(p, sym_buffers(p, dp, partials), host_descs, idx, blk_begin);
    PackSeg g;
    g.a = make_args(p, dp, scratch_view(p, partials));
    g.nbx = std::max(1u, row_blocks(p));
    g.blk_begin = (int)blk_begin;
    ((PackSeg *)host_descs)[idx] = g;
    return (int64_t)g.nbx * p.splits;
}

hipError_t launch_pair_packed(const EvalPlan &p, const void *dev_descs, int nseg, int64_t total_blocks,
                              hipStream_t st) {
    if (nseg <= 0 || total_blocks <= 0) return hipSuccess;
    if (nseg > kMaxPack || total_blocks > INT32_MAX) return hipErrorInvalidValue;
    if (sym_selected(p)) return launch_sym_packed(p, dev_descs, nseg, total_blocks, st);
    return launch_pair(p.variant, p.precision, nullptr, (const PackSeg *)dev_descs, nseg, (unsigned)total_blocks, 1,
                       st);
}

hipError_t launch_pack(const double *x, const double *M, const double *soft, int64_t n,
                       DeviceParticles &dp, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(pack_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, M,
                       soft, dp.jrec, dp.soft, n);
    return hipGetLastError();
}

hipError_t launch_check_finite(const double *x, int64_t count, int *flag, hipStream_t st) {
    if (count <= 0) return hipSuccess;
    const unsigned nb = (unsigned)std::min<int64_t>(4096, (count + 255) / 256);
    hipLaunchKernelGGL(check_finite_kernel, dim3(nb), dim3(256), 0, st, x, count, flag);
    return hipGetLastError();
}

hipError_t launch_pack_positions(const double *x, int64_t n, DeviceParticles &dp,
                                 hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(pack_positions_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                       x, dp.jrec, n);
    return hipGetLastError();
}

hipError_t launch_unpack_positions(const DeviceParticles &dp, double *x, hipStream_t st) {
    if (dp.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(unpack_positions_kernel, dim3((unsigned)((dp.n + 255) / 256)), dim3(256), 0,
                       st, dp.jrec, x, dp.n);
    return hipGetLastError();
}

}  // namespace steps
