// pme.h -- smooth PME of Gaussian charges and point dipoles: spread, convolution, gathers.
//
// Per atom: u = r H^-1 (FP64), w = K frac(u), base = floor(w), f = w - base (rounded to real);
// theta / dtheta (and for forces d2theta) of order P are recomputed from f in registers by every
// kernel (no per-atom spline storage).  Grid point (base + k) mod K gets weight theta[k].
//   Q(g) = sum_i q_i t1 t2 t3 + e_i1 d1 t2 t3 + e_i2 t1 d2 t3 + e_i3 t1 t2 d3,  e_i = d_i H^-1 K
// (pgm_jax/md/pme.py:306-337).  phi = dE_rec/dQ comes from r2c FFT -> multiply by
// Gc = 2 G / w3 -> c2r FFT (unnormalised), pme.py:373-376.
#pragma once

#include "common.h"
#include "tiles.h"

namespace pgm {

struct PMEGeom {
    double hinv[9];      // H^-1
    double escale[9];    // H^-1 with column b scaled by K_b: e = d . escale
    int K[3];
};

template <typename real, int P>
PGM_DEV void stencil(const double *__restrict__ pos, int i, const PMEGeom &g, int *base, real *f) {
    const double x = pos[3 * i], y = pos[3 * i + 1], z = pos[3 * i + 2];
    const double *hi = g.hinv;
    const double u[3] = {x * hi[0] + y * hi[3] + z * hi[6], x * hi[1] + y * hi[4] + z * hi[7], x * hi[2] + y * hi[5] + z * hi[8]};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const double w = (u[a] - floor(u[a])) * (double)g.K[a];
        const double b = floor(w);
        base[a] = (int)b;
        f[a] = (real)(w - b);
    }
}

// bspline of order P at f, evaluated in FP64 and rounded to real.  FP32 recursions lose a few units in the
// last place of every weight, with the same sign for the whole grid: at 32,768 waters the field's error
// against float64 was 3.4e-7 with them and is 2.6e-7 with the weights rounded once; the spread's time did
// not change.
template <typename real, int P, bool D2> PGM_DEV void bspline_rounded(real f, real *th, real *dth, real *d2th) {
    double t[P], d[P], d2[P];
    bspline<double, P, D2>((double)f, t, d, d2);
#pragma unroll
    for (int k = 0; k < P; ++k) {
        th[k] = (real)t[k];
        dth[k] = (real)d[k];
        if (D2) d2th[k] = (real)d2[k];
    }
}

template <typename real>
PGM_DEV void scaled_dipole(const real4<real> &d, const PMEGeom &g, real *e) {
#pragma unroll
    for (int b = 0; b < 3; ++b) e[b] = d.x * (real)g.escale[b] + d.y * (real)g.escale[3 + b] + d.z * (real)g.escale[6 + b];
}

template <typename T> __global__ void k_fill(size_t n, T *__restrict__ p, T v) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Spread: one thread per (atom, x offset); 36 atomic adds each (v1 of the spread; deterministic
// order is not guaranteed).  dq = (d, q); WITHQ includes the charges.
template <typename real, int P, bool WITHQ>
__global__ __launch_bounds__(256) void k_spread(int n, const double *__restrict__ pos, const real4<real> *__restrict__ dq,
                                                PMEGeom g, real *__restrict__ grid, const int *__restrict__ conv_it, int iter) {
    if (conv_it && iter >= *conv_it) return;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = t / P, ix = t - i * P;
    if (i >= n) return;
    int base[3];
    real f[3];
    stencil<real, P>(pos, i, g, base, f);
    real t1[P], d1[P], t2[P], d2[P], t3[P], d3[P];
    bspline<real, P, false>(f[0], t1, d1, nullptr);
    bspline<real, P, false>(f[1], t2, d2, nullptr);
    bspline<real, P, false>(f[2], t3, d3, nullptr);
    const real4<real> d = dq[i];
    real e[3];
    scaled_dipole<real>(d, g, e);
    const real q = WITHQ ? d.w : real(0);
    const real a1 = q * t1[ix] + e[0] * d1[ix];
    const real b1 = e[1] * t1[ix];
    const real c1 = e[2] * t1[ix];
    const int K1 = g.K[0], K2 = g.K[1], K3 = g.K[2];
    int gx = base[0] + ix;
    gx -= gx >= K1 ? K1 : 0;
#pragma unroll
    for (int iy = 0; iy < P; ++iy) {
        const real A = a1 * t2[iy] + b1 * d2[iy];
        const real C = c1 * t2[iy];
        int gy = base[1] + iy;
        gy -= gy >= K2 ? K2 : 0;
        real *line = grid + ((size_t)gx * K2 + gy) * K3;
#pragma unroll
        for (int iz = 0; iz < P; ++iz) {
            int gz = base[2] + iz;
            gz -= gz >= K3 ? K3 : 0;
            unsafeAtomicAdd(line + gz, A * t3[iz] + C * d3[iz]);
        }
    }
}

// ---------------------------------------------------------------------------- tiled spread
// Atomic-free, deterministic spread.  The grid is cut into tiles (T_a points per axis, every tile at
// least P-1 wide, at least three tiles per axis); every atom belongs to the tile holding its stencil
// base.  Atoms are sorted by tile once per geometry (k_pme_bin to k_pme_order).  One
// wave per tile sums its atoms' stencils on the tile's block of (T+P-1)^3 points on the matrix cores
// (k_spread_tiles), and k_merge_table (or the forward planes of the fused transform) sums, for
// every grid point, the (up to 8) blocks that cover it in a fixed order.
// Tiles are numbered by the fine key = cube index * 8 + octant, so that consecutive keys are near each
// other in space.
PGM_DEV int fine_key(const int (&u8)[3], const PMETiles &t) {
    const int oct = ((u8[0] & 1) << 2) | ((u8[1] & 1) << 1) | (u8[2] & 1);
    return (((u8[0] >> 1) * t.nc[1] + (u8[1] >> 1)) * t.nc[2] + (u8[2] >> 1)) * 8 + oct;
}

// Sorting the atoms by tile (key = bead * t8.ntiles + fine key of the stencil base), in four launches:
//   k_pme_bin    each atom's key and its arrival number in the tile (an integer atomic on the tile's count)
//   k_pme_scan   the tiles' ranges (exclusive scan of the counts, one workgroup), the counts cleared again
//   k_pme_place  the atoms into their tiles' ranges, in arrival order
//   k_pme_order  one wave per tile: the atoms of the tile in index order (whatever the arrival order, so
//                the order of every sum is fixed) with their stencils
// A radix sort of (key, atom), tile bounds and stencils took eleven launches, 150 us at 98,304 atoms.
template <typename real> PGM_DEV int tile_base(const double *__restrict__ pos, int i, const PMEGeom &g, const PMETiles &t8, int (&u8)[3], real (&f)[3]) {
    int base[3], loc = 0;
    stencil<real, 4>(pos, i, g, base, f);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int bb = base[a] >= g.K[a] ? base[a] - g.K[a] : base[a];
        const int u = bb / t8.T[a];
        u8[a] = u < t8.nt[a] ? u : t8.nt[a] - 1;
        loc |= (bb - u8[a] * t8.T[a]) << (5 * a);
    }
    return loc;  // the base relative to its tile, packed (lx | ly << 5 | lz << 10)
}
__global__ void k_pme_bin(int n, int nper, const double *__restrict__ pos, PMEGeom g, PMETiles t8, int *__restrict__ key,
                          int *__restrict__ arrival, int *__restrict__ count) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int u8[3];
    double f[3];
    (void)tile_base<double>(pos, i, g, t8, u8, f);
    const int k = (i / nper) * t8.ntiles + fine_key(u8, t8);
    key[i] = k;
    arrival[i] = atomicAdd(count + k, 1);
}

// One workgroup, 2.3 us per 1,024 tiles, where the library's sort of the atoms does not depend on the tiles: beyond
// PME_SCAN_SMALL tiles the counts are taken with four atoms a tile and more, beyond PME_SCAN_MAX never.  Spread
// of the PME object, counts / library sort [us]: 200^3 (17,576 tiles) 300 atoms 152 / 160, 30,000: 162 / 178; 256^3
// (32,768) 300: 355 / 386, 3,000: 356 / 337, 100,000: 389 / 394, 300,000: 429 / 503; 384^3 (110,592) 30,000:
// 1021 / 919, 300,000: 1180 / 1145, 1,000,000: 1330 / 1338.  Four waves: a workgroup of sixteen waited 160 us for
// a CU with room beside the record pass.
constexpr int PME_SCAN_SMALL = 20000, PME_SCAN_MAX = 1 << 17, PME_SCAN_THREADS = 256;
// k_pme_order compares the m atoms of a tile with one another, m^2 / 64 steps of a wave: tiles that may hold
// more than PME_ORDER_MAX (8^3 points 0.16 nm apart in water) leave the sort to the library too.  Spread of the
// PME object on 48^3, 216 tiles, counts / library sort [us]: 100 atoms a tile 78 / 120, 200: 151 / 181, 400:
// 330 / 220, 800: 931 / 369, 6,400: 36,000 / 2,310.
constexpr int PME_ORDER_MAX = 256;
__global__ __launch_bounds__(PME_SCAN_THREADS) void k_pme_scan(int nk, int *__restrict__ count, int2 *__restrict__ range) {
    constexpr int NW = PME_SCAN_THREADS / WAVE;
    __shared__ int wsum[NW];
    const int lane = threadIdx.x % WAVE, wv = threadIdx.x / WAVE;
    int carry = 0;
    for (int k0 = 0; k0 < nk; k0 += 4 * PME_SCAN_THREADS) {
        const int k = k0 + 4 * threadIdx.x;
        int c[4], sum = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            c[u] = k + u < nk ? count[k + u] : 0;
            sum += c[u];
        }
        int incl = sum;
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) {
            const int t = __shfl_up(incl, o, WAVE);
            if (lane >= o) incl += t;
        }
        __syncthreads();
        if (lane == WAVE - 1) wsum[wv] = incl;
        __syncthreads();
        int before = carry, total = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            if (w < wv) before += wsum[w];
            total += wsum[w];
        }
        int s = before + incl - sum;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (k + u < nk) {
                range[k + u] = make_int2(s, s + c[u]);
                s += c[u];
                count[k + u] = 0;
            }
        carry += total;
    }
}

__global__ void k_pme_place(int n, const int *__restrict__ key, const int *__restrict__ arrival, const int2 *__restrict__ range,
                            int *__restrict__ slot) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) slot[range[key[i]].x + arrival[i]] = i;
}

// Tile coordinates of octant oct of a cube whose packed coordinates (u0 | u1 << 10 | u2 << 20) are org; false
// for an octant past the grid.
PGM_DEV bool octant_tile(int org, int oct, const PMETiles &t, int (&u8)[3]) {
    u8[0] = 2 * (org & 1023) + (oct >> 2);
    u8[1] = 2 * ((org >> 10) & 1023) + ((oct >> 1) & 1);
    u8[2] = 2 * (org >> 20) + (oct & 1);
    return u8[0] < t.nt[0] && u8[1] < t.nt[1] && u8[2] < t.nt[2];
}

// The stencil of a sorted atom: the offsets f in [0, 1) along the axes (rounded to real, the arguments of
// bspline) and the base point relative to its tile, packed (lx | ly << 5 | lz << 10) in the bits of w.
// 16 bytes per atom (FP32): the spread and the gather evaluate the splines from it (about 60
// instructions per axis) rather than read 6 P stored weights per atom, whose rows of 144 bytes made each
// of the gather's 36 loads touch one cache line per lane.
PGM_DEV float pack_loc(int v, float) { return __int_as_float(v); }
PGM_DEV double pack_loc(int v, double) { return __longlong_as_double((long long)v); }
PGM_DEV int unpack_loc(float v) { return __float_as_int(v); }
PGM_DEV int unpack_loc(double v) { return (int)__double_as_longlong(v); }

template <typename real>
PGM_DEV real4<real> atom_stencil(const double *__restrict__ pos, int i, const PMEGeom &g, const PMETiles &t8) {
    int u8[3];
    real f[3];
    const int loc = tile_base<real>(pos, i, g, t8, u8, f);
    real4<real> v;
    v.x = f[0];
    v.y = f[1];
    v.z = f[2];
    v.w = pack_loc(loc, real(0));
    return v;
}

template <typename real>
__global__ __launch_bounds__(256) void k_pme_order(int nk, const int2 *__restrict__ range, const int *__restrict__ slot,
                                                   const double *__restrict__ pos, PMEGeom g, PMETiles t8, int *__restrict__ sidx,
                                                   real4<real> *__restrict__ sten) {
    const int lane = threadIdx.x % WAVE, k = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (k >= nk) return;
    const int2 rg = range[k];
    for (int s = rg.x + lane; __ballot(s < rg.y); s += WAVE) {
        const int i = s < rg.y ? slot[s] : 0;
        int rank = 0;  // atoms of the tile with a smaller index
        for (int t0 = rg.x; t0 < rg.y; t0 += WAVE) {
            const int m = min(WAVE, rg.y - t0);
            const int other = lane < m ? slot[t0 + lane] : 0;
            for (int j = 0; j < m; ++j) rank += __builtin_amdgcn_readlane(other, j) < i ? 1 : 0;
        }
        if (s < rg.y) {
            sidx[rg.x + rank] = i;
            sten[rg.x + rank] = atom_stencil<real>(pos, i, g, t8);
        }
    }
}

// The same from a library sort of (key, atom): ranges from the sorted keys, stencils in sorted order.
// Thread s in [0, n] looks at the keys either side of position s (key -1 before the first, the tile
// count after the last): position s is the start of every tile k with key[s-1] < k <= key[s] and the
// end of tile k - 1, so every tile's start and end is written once and an empty tile gets an empty
// range.
template <typename real>
__global__ void k_pme_sorted(int n, const int *__restrict__ skey, int nk, const int *__restrict__ sidx, const double *__restrict__ pos,
                             PMEGeom g, PMETiles t8, int2 *__restrict__ range, real4<real> *__restrict__ sten) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s > n) return;
    const int p8 = s > 0 ? skey[s - 1] : -1, c8 = s < n ? skey[s] : nk;
    for (int k = p8 + 1; k <= c8; ++k) {
        if (k < nk) range[k].x = s;
        if (k > 0 && k <= nk) range[k - 1].y = s;
    }
    if (s < n) sten[s] = atom_stencil<real>(pos, sidx[s], g, t8);
}

// Tiled spread on the matrix cores: one wave per tile (fine key; block b * t.ntiles + key for bead b).
// On the tile's block the sum over its atoms is, for every y, a product of two thin matrices,
//   Q[x][z] = sum_a X1[x][a] (Y[y][a] Z[a][z]) + X2[x][a] (Y'[y][a] e2 Z[a][z] + Y[y][a] e3 Z'[a][z]),
//   X1 = q theta_x + e1 theta'_x,  X2 = theta_x,
// with the weights zero outside an atom's P points: 16 x 16 x 4 matrix instructions over four atoms at
// a time (x the rows, z the columns; FP32 or FP64), the block held in accumulators of at most 15 rows y
// until it is stored.  The atoms come in chunks of SPREAD_CHUNK: 3 x SPREAD_CHUNK lanes evaluate one
// axis' spline of one atom each into dense rows in LDS.  All rows y are taken for every four atoms: a
// test per row, to skip those out of reach, takes the independent products out of one stream and costs
// more than it saves (50 us).  No atomics and a fixed order: bitwise reproducible.
//
// Bound by the chain of one wave: at 4,096 tiles of 24 atoms four waves a SIMD are all there are, the matrix
// cores are busy for 8.3 of 25.6 us, the VALU for a third, and 45 MB of blocks are written.  Measured per launch (FP32, alone) at 32,768 waters and 128^3 / 512 waters and 32^3: 24.1 / 9.8
// us; the earlier form, one atom at a time with a read-add-write of its 216 points in LDS, 26.8 / 13.7 us;
// summing the eight tiles of a cube in LDS first (22 MB written) 30.0 / 19.3 us.
constexpr int SPREAD_CHUNK = 16;
constexpr int SPREAD_ROW = 17;  // LDS row of one atom's dense weights (16 points; odd: no bank conflicts)
constexpr int SPREAD_PLANES = 7;  // X1, X2, Y, Y', Z, e2 Z, e3 Z'

template <typename real> struct mfma_acc;
template <> struct mfma_acc<float> { typedef float type __attribute__((ext_vector_type(4))); };
template <> struct mfma_acc<double> { typedef double type __attribute__((ext_vector_type(4))); };
PGM_DEV mfma_acc<float>::type mfma_16x16x4(float a, float b, mfma_acc<float>::type c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
PGM_DEV mfma_acc<double>::type mfma_16x16x4(double a, double b, mfma_acc<double>::type c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// Row of result register r of lane group grp = lane / 16 (lane l holds column l % 16).
template <typename real> PGM_DEV int mfma_row(int grp, int r) { return sizeof(real) == 4 ? 4 * grp + r : grp + 4 * r; }

// LDS of one wave of the spread, in 16-byte units.
template <typename real> constexpr int spread_lds16() {
    return (SPREAD_PLANES * SPREAD_CHUNK * SPREAD_ROW * (int)sizeof(real) + 15) / 16;
}
template <typename real> struct SpreadArgs {
    PMETiles t;
    PMEGeom g;
    const int *corg;
    const int2 *range;
    const int *sidx;
    const real4<real> *sten;
    real *blocks;
};

// Tile `tile` (bead * t.ntiles + key) by one wave, its rows in w4.
template <typename real, int P, bool WITHQ>
PGM_DEV void spread_tile(const SpreadArgs<real> &A, int tile, float4 *w4, const real4<real> *__restrict__ dq,
                         const int *__restrict__ conv_it, int iter) {
    const PMETiles &t = A.t;
    const PMEGeom &g = A.g;
    const int *__restrict__ corg = A.corg;
    const int2 *__restrict__ range = A.range;
    const int *__restrict__ sidx = A.sidx;
    const real4<real> *__restrict__ sten = A.sten;
    real *__restrict__ blocks = A.blocks;
    const int bead = tile / t.ntiles, key = tile - bead * t.ntiles;
    if (cg_done(conv_it, bead, iter)) return;
    int u8[3];
    if (!octant_tile(corg[key >> 3], key & 7, t, u8)) return;  // no merge reads the block
    using acc_t = typename mfma_acc<real>::type;
    constexpr int MAXB = P + 7;  // block rows at most (T <= 8)
    constexpr int PLANE = SPREAD_CHUNK * SPREAD_ROW, NZ = spread_lds16<real>();
    real *w = reinterpret_cast<real *>(w4);
    const int lane = threadIdx.x % WAVE, grp = lane / 16, m = lane % 16;
    const int2 rg = range[tile];
    const int s0 = rg.x, s1 = rg.y;
    acc_t D[MAXB];
#pragma unroll
    for (int y = 0; y < MAXB; ++y) D[y] = acc_t{0, 0, 0, 0};
    const int ax = lane / SPREAD_CHUNK, a = lane % SPREAD_CHUNK;  // this lane's axis (0..2) and atom of a chunk
    real4<real> st{}, d{};
    if (ax < 3 && s0 + a < s1) {
        st = sten[s0 + a];
        d = dq[sidx[s0 + a]];
    }
    for (int c0 = s0; c0 < s1; c0 += SPREAD_CHUNK) {
        const int mc = min(SPREAD_CHUNK, s1 - c0);
        const bool on = ax < 3 && a < mc;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the previous chunk's rows have been read
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < NZ; k += WAVE)
            if (k + lane < NZ) w4[k + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (on) {
            const int l = (unpack_loc(st.w) >> (5 * ax)) & 31;
            double th[P], dth[P], e[3];
            bspline<double, P, false>((double)(ax == 0 ? st.x : (ax == 1 ? st.y : st.z)), th, dth, nullptr);
#pragma unroll
            for (int b = 0; b < 3; ++b) e[b] = (double)d.x * g.escale[b] + (double)d.y * g.escale[3 + b] + (double)d.z * g.escale[6 + b];
            const double q = WITHQ ? (double)d.w : 0.0;
            real *row = w + a * SPREAD_ROW + l;
            if (ax == 0) {
#pragma unroll
                for (int k = 0; k < P; ++k) {
                    row[k] = (real)(q * th[k] + e[0] * dth[k]);
                    row[PLANE + k] = (real)th[k];
                }
            } else if (ax == 1) {
#pragma unroll
                for (int k = 0; k < P; ++k) {
                    row[2 * PLANE + k] = (real)th[k];
                    row[3 * PLANE + k] = (real)dth[k];
                }
            } else {
#pragma unroll
                for (int k = 0; k < P; ++k) {
                    row[4 * PLANE + k] = (real)th[k];
                    row[5 * PLANE + k] = (real)(e[1] * th[k]);
                    row[6 * PLANE + k] = (real)(e[2] * dth[k]);
                }
            }
        }
        if (ax < 3 && c0 + SPREAD_CHUNK + a < s1) {  // the next chunk's atoms, in flight with the products
            st = sten[c0 + SPREAD_CHUNK + a];
            d = dq[sidx[c0 + SPREAD_CHUNK + a]];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int a0 = 0; a0 < mc; a0 += 4) {
            const real *row = w + (a0 + grp) * SPREAD_ROW;
            const real x1 = row[m], x2 = row[PLANE + m];
            const real z0 = row[4 * PLANE + m], z1 = row[5 * PLANE + m], z2 = row[6 * PLANE + m];
#pragma unroll
            for (int y = 0; y < MAXB; ++y) {
                const real ty = row[2 * PLANE + y], dy = row[3 * PLANE + y];
                D[y] = mfma_16x16x4(x1, ty * z0, D[y]);
                D[y] = mfma_16x16x4(x2, dy * z1 + ty * z2, D[y]);
            }
        }
    }
    real *out = blocks + (size_t)tile * t.bsize + m;
#pragma unroll
    for (int y = 0; y < MAXB; ++y) {
        if (y < t.B[1]) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int x = mfma_row<real>(grp, r);
                if (x < t.B[0]) out[(x * t.B[1] + y) * PME_ZROW] = D[y][r];
            }
        }
    }
}

template <typename real, int P, bool WITHQ>
__global__ __launch_bounds__(64, sizeof(real) == 4 ? 4 : 2) void k_spread_tiles(SpreadArgs<real> A, const real4<real> *__restrict__ dq,
                                                     const int *__restrict__ conv_it, int iter) {
    __shared__ float4 w4[spread_lds16<real>()];
    spread_tile<real, P, WITHQ>(A, blockIdx.x, w4, dq, conv_it, iter);
}

// Block merge: grid point value = sum of the tiles' blocks covering it -- along each axis its own tile
// (local l) and, when l <= P-2, the previous one (local l + width of that tile), in a fixed order
// (deterministic).  Table driven: for grid coordinate g along axis a, tab_a[2 g] is the offset (in reals)
// of the point in the axis part of its own tile's block -- A_a(u) bsize + l stride_a with A_0(u) =
// ((u >> 1) nc1 nc2 8 + (u & 1) 4), A_1(u) = ((u >> 1) nc2 8 + (u & 1) 2), A_2(u) = ((u >> 1) 8 + (u & 1)),
// strides B1 PME_ZROW, PME_ZROW, 1 -- and tab_a[2 g + 1] the same for the previous tile (local l + its
// width) when l <= P-2, else PME_NO_BLOCK.  Both the fine key and the in-block offset are sums over the axes, so a
// grid point's up to 8 block values are blocks[bead base + X + Y + Z] over the axes' candidates, summed
// in a fixed order.
// Launch: x = z-line (blockDim.x points), y = K2 rows, z = K1 planes times beads.
template <typename real>
__global__ __launch_bounds__(128) void k_merge_table(int K1, int K2, int K3, size_t bead_blocks, const unsigned *__restrict__ tab,
                                                     const real *__restrict__ blocks, real *__restrict__ grid,
                                                     const int *__restrict__ conv_it, int iter) {
    const int gz = blockIdx.x * blockDim.x + threadIdx.x;
    const int gy = blockIdx.y;
    const int gx = blockIdx.z % K1, bead = blockIdx.z / K1;
    if (gz >= K3 || cg_done(conv_it, bead, iter)) return;
    const unsigned *tx = tab, *ty = tab + 2 * K1, *tz = tab + 2 * (K1 + K2);
    const unsigned X[2] = {tx[2 * gx], tx[2 * gx + 1]}, Y[2] = {ty[2 * gy], ty[2 * gy + 1]}, Z[2] = {tz[2 * gz], tz[2 * gz + 1]};
    const real *b = blocks + bead_blocks * bead;
    real acc = real(0);
#pragma unroll
    for (int i0 = 0; i0 < 2; ++i0)
#pragma unroll
        for (int i1 = 0; i1 < 2; ++i1)
#pragma unroll
            for (int i2 = 0; i2 < 2; ++i2)
                if (X[i0] != PME_NO_BLOCK && Y[i1] != PME_NO_BLOCK && Z[i2] != PME_NO_BLOCK) acc += b[(size_t)X[i0] + Y[i1] + Z[i2]];
    grid[(((size_t)bead * K1 + gx) * K2 + gy) * K3 + gz] = acc;
}

// Convolution on the half spectrum: F[Q] *= Gc; with ENERGY also sum (w3/2) Gc |F[Q]|^2 per block
// (= sum G |F[Q]|^2 with G of pme.py:243-267), FP64.  Grid (blocks per bead, beads): bead b's
// transform at cgrid + 2 b nc, its partials at epart[b * gridDim.x + blockIdx.x].
template <typename real, bool ENERGY>
__global__ __launch_bounds__(256) void k_convolve(size_t nc, int K3h, int K3even, real *__restrict__ cgrid,
                                                  const real *__restrict__ Gc, double *__restrict__ epart,
                                                  const int *__restrict__ conv_it, int iter) {
    if (cg_done(conv_it, blockIdx.y, iter)) return;
    __shared__ double lds[16];
    const size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    cgrid += 2 * nc * blockIdx.y;
    double e[1] = {0.0};
    if (s < nc) {
        const real gc = Gc[s];
        const real re = cgrid[2 * s], im = cgrid[2 * s + 1];
        if (ENERGY) {
            const int k3 = (int)(s % (size_t)K3h);
            const double w = (k3 == 0 || (K3even && k3 == K3h - 1)) ? 0.5 : 1.0;
            e[0] = w * (double)gc * ((double)re * re + (double)im * im);
        }
        cgrid[2 * s] = re * gc;
        cgrid[2 * s + 1] = im * gc;
    }
    if (ENERGY) {
        block_sum<1>(e, lds);
        if (threadIdx.x == 0) epart[blockIdx.y * gridDim.x + blockIdx.x] = e[0];
    }
}

// Reciprocal-space part of the strain derivative that comes from the influence function: for
// G(m*, V) = exp(-pi^2 |m*|^2 / beta^2) / (2 pi V |m*|^2) B(m), with m* = H^-1 m moving as
// -eps^T m* and V as (1 + tr eps), dG/d eps_ab = G [2 (pi^2/beta^2 + 1/|m*|^2) m*_a m*_b - delta_ab].
// Per block: the six sums of w Gc |F Q|^2 2 (pi^2/beta^2 + 1/|m*|^2) m*_a m*_b (xx yy zz xy xz yz)
// and E_rec = sum w Gc |F Q|^2, from the unconvolved transform (w = 1/2 on the k3 = 0 and Nyquist
// planes of the half spectrum, 1 elsewhere).  cgrid is only read.
struct RecipGeom {
    double hinv[9];   // H^-1: m* = H^-1 (m1, m2, m3)
    int K[3];
    double pb2;       // pi^2 / beta^2
};

template <typename real>
__global__ __launch_bounds__(256) void k_convolve_virial(size_t nc, RecipGeom rg, const real *__restrict__ cgrid,
                                                         const real *__restrict__ Gc, double *__restrict__ vpart) {
    __shared__ double lds[7 * 16];
    const size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    if (s < nc) {
        const int K1 = rg.K[0], K2 = rg.K[1], K3 = rg.K[2], K3h = K3 / 2 + 1;
        const int k3 = (int)(s % (size_t)K3h);
        const int k2 = (int)((s / (size_t)K3h) % (size_t)K2);
        const int k1 = (int)(s / ((size_t)K3h * K2));
        const double f1 = k1 <= (K1 - 1) / 2 ? k1 : k1 - K1;
        const double f2 = k2 <= (K2 - 1) / 2 ? k2 : k2 - K2;
        const double f3 = k3;
        const double *h = rg.hinv;
        const double mx = h[0] * f1 + h[1] * f2 + h[2] * f3;
        const double my = h[3] * f1 + h[4] * f2 + h[5] * f3;
        const double mz = h[6] * f1 + h[7] * f2 + h[8] * f3;
        const double msq = mx * mx + my * my + mz * mz;
        const double re = (double)cgrid[2 * s], im = (double)cgrid[2 * s + 1];
        const double w = (k3 == 0 || (K3 % 2 == 0 && k3 == K3h - 1)) ? 0.5 : 1.0;
        const double e = w * (double)Gc[s] * (re * re + im * im);
        if (msq > 0.0) {
            const double c = 2.0 * e * (rg.pb2 + 1.0 / msq);
            acc[0] = c * mx * mx;
            acc[1] = c * my * my;
            acc[2] = c * mz * mz;
            acc[3] = c * mx * my;
            acc[4] = c * mx * mz;
            acc[5] = c * my * mz;
            acc[6] = e;
        }
    }
    block_sum<7>(acc, lds);
    if (threadIdx.x == 0)
        for (int k = 0; k < 7; ++k) vpart[7 * blockIdx.x + k] = acc[k];
}

// Gather of the dipole gradient (pme.py:378-388): g_a = sum phi * (derivative spline along a),
// dU/dd = escale . g; then combined with the row field according to `mode`:
//   0 FIELD   out = -(row + rec - c_self d)                          [+ sum |alpha out| per block]
//   1 AV      out = d / alpha + row + rec - c_self d                 [+ sum d . out per block]
//   2 FUSED   out = -(row + rec - c_self d) - x0 / alpha             (d = p + x0, extra = x0)
//   3 PLAIN   out = b - (d / alpha + row + rec - c_self d)           (d = x0, extra = b)
//   4 REC     out = dU_rec/dd alone
enum { MODE_FIELD = 0, MODE_AV = 1, MODE_FUSED = 2, MODE_PLAIN = 3, MODE_REC = 4 };

// out[i] from rec = dU_rec/dd (rx, ry, rz) and the row field, by `mode` (see above); acc gets the
// per-atom contribution to the block partial of MODE_FIELD / MODE_AV.
template <typename real>
PGM_DEV void combine_out(int mode, int i, real rx, real ry, real rz, const real4<real> *__restrict__ dq,
                         const real4<real> *__restrict__ row, const real *__restrict__ alpha,
                         const real4<real> *__restrict__ extra, real cself, real4<real> *__restrict__ out, double &acc) {
    const real4<real> d = dq[i];
    const real4<real> rw = row[i];
    const real tx = rw.x + rx - cself * d.x;  // dU/dd (direct + reciprocal + self)
    const real ty = rw.y + ry - cself * d.y;
    const real tz = rw.z + rz - cself * d.z;
    real4<real> o;
    o.w = 0;
    const real ia = alpha[i] != real(0) ? real(1) / alpha[i] : real(0);  // 0: not polarizable
    if (mode == MODE_FIELD) {
        o.x = -tx;
        o.y = -ty;
        o.z = -tz;
        const real a = alpha[i];
        acc = fabs((double)(a * o.x)) + fabs((double)(a * o.y)) + fabs((double)(a * o.z));
    } else if (mode == MODE_AV) {
        o.x = d.x * ia + tx;
        o.y = d.y * ia + ty;
        o.z = d.z * ia + tz;
        acc = (double)(d.x * o.x) + (double)(d.y * o.y) + (double)(d.z * o.z);
    } else if (mode == MODE_FUSED) {
        const real4<real> x0 = extra[i];
        o.x = -tx - x0.x * ia;
        o.y = -ty - x0.y * ia;
        o.z = -tz - x0.z * ia;
    } else if (mode == MODE_REC) {
        o.x = rx;
        o.y = ry;
        o.z = rz;
    } else {
        const real4<real> b = extra[i];
        o.x = b.x - (d.x * ia + tx);
        o.y = b.y - (d.y * ia + ty);
        o.z = b.z - (d.z * ia + tz);
    }
    out[i] = o;
}

// One wave copies the potential on a tile's (T + P - 1)^3 block (periodic wrap) into blk, 16 bytes per lane
// and load where the rows allow it (VEC: K3 and T2 multiples of 16 / sizeof(real)), and waits for its writes.
template <typename real, int P, bool VEC>
PGM_DEV void load_tile_block(const PMETiles &t, const PMEGeom &g, const int *u8, const real *__restrict__ phi, real *blk, int lane) {
    constexpr int V = VEC ? 16 / (int)sizeof(real) : 1, LPR = 16 / V, RPI = WAVE / LPR;  // reals, lanes per row, rows per load
    constexpr int SZ = (P + 7) | 1;
    const int K1 = g.K[0], K2 = g.K[1], K3 = g.K[2], BY = t.B[1], BZ = t.B[2], nrow = t.B[0] * BY;
    const int bz = V * (lane % LPR);
    int gz = u8[2] * t.T[2] + bz;
    gz -= gz >= K3 ? K3 : 0;
    const int o0 = u8[0] * t.T[0], o1 = u8[1] * t.T[1];
    const unsigned magic = 65536u / (unsigned)BY + 1u;  // row / BY for row < 256
    constexpr int BATCH = 8;
    for (int r0 = lane / LPR; r0 < nrow; r0 += BATCH * RPI) {
        real v[BATCH][V];
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            const int rr = r0 + u * RPI < nrow ? r0 + u * RPI : 0;
            const int bx = (int)(((unsigned)rr * magic) >> 16), by = rr - bx * BY;
            int gx = o0 + bx, gy = o1 + by;
            gx -= gx >= K1 ? K1 : 0;
            gy -= gy >= K2 ? K2 : 0;
            const real *src = phi + ((size_t)gx * K2 + gy) * K3 + gz;
            if constexpr (V == 4) {
                const float4 q = *reinterpret_cast<const float4 *>(src);
                v[u][0] = q.x, v[u][1] = q.y, v[u][2] = q.z, v[u][3] = q.w;
            } else if constexpr (V == 2) {
                const double2 q = *reinterpret_cast<const double2 *>(src);
                v[u][0] = q.x, v[u][1] = q.y;
            } else {
                v[u][0] = bz < BZ ? *src : real(0);
            }
        }
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
            if (r0 + u * RPI < nrow)
#pragma unroll
                for (int k = 0; k < V; ++k)
                    if (bz + k < BZ) blk[(r0 + u * RPI) * SZ + bz + k] = v[u][k];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Tiled gather + combine: one wave per tile (fine key), GATHER_WAVES waves per workgroup.  The wave copies
// the potential on the tile's (T + P - 1)^3 block (periodic wrap) into its part of the LDS, 16 bytes
// per lane and load where the rows allow it (VEC: K3 and T2 multiples of 16 / sizeof(real)), then two
// neighbouring lanes per atom (sorted order s, atom sidx[s]) sum its stencil from LDS, the first
// (P+1)/2 x planes and the rest, and the first lane's combine_out writes the result.  Per-workgroup
// partials of MODE_FIELD / MODE_AV go to part[blockIdx.x].  The potential of bead b is at phi + b K1 K2 K3.
// Bound by latency and LDS reads: 16.8 us alone at 32,768 waters, the VALU issuing for 44 % of it and the waves
// waiting for as much (51 MB read and written, a tile's block being 4 times its points).  Measured against one 512-thread workgroup per 16^3 points reading
// stored splines (FP32, alone): 22 us at 32,768 waters and 128^3, 10.4 us at 64 waters and 32^3.
template <typename real> constexpr int gather_waves() { return sizeof(real) == 4 ? 4 : 2; }
template <typename real, int P, bool VEC>
__global__ __launch_bounds__(WAVE * gather_waves<real>()) void k_gather_tiles(PMETiles t, const int *__restrict__ corg, PMEGeom g,
                                                      const int2 *__restrict__ range, const int *__restrict__ sidx,
                                                      const real4<real> *__restrict__ sten,
                                                      const real *__restrict__ phi, const real4<real> *__restrict__ dq,
                                                      const real4<real> *__restrict__ row, const real *__restrict__ alpha,
                                                      const real4<real> *__restrict__ extra, real cself, int mode,
                                                      real4<real> *__restrict__ out, double *__restrict__ part,
                                                      const int *__restrict__ conv_it, int iter) {
    constexpr int GW = gather_waves<real>();
    const int bead = (blockIdx.x * GW) / t.ntiles;  // t.ntiles is a multiple of 8
    if (cg_done(conv_it, bead, iter)) return;
    constexpr int MAXB = P + 7, SZ = MAXB | 1;
    __shared__ real blk_all[GW][MAXB * MAXB * SZ];
    __shared__ double lds[16];
    const int lane = threadIdx.x % WAVE, wv = threadIdx.x / WAVE;
    const int tile = blockIdx.x * GW + wv;
    real *blk = blk_all[wv];
    const int BY = t.B[1];
    const int2 rg = range[tile];
    const int s0 = rg.x, s1 = rg.y, lt = tile - bead * t.ntiles;
    const int half = lane & 1;
    double acc[1] = {0.0};
    int u8[3];
    if (s0 < s1 && octant_tile(corg[lt >> 3], lt & 7, t, u8)) {
        phi += (size_t)bead * g.K[0] * g.K[1] * g.K[2];
        int s = s0 + (lane >> 1);
        real4<real> st{};
        int atom = 0;
        if (s < s1) {  // in flight with the block
            st = sten[s];
            atom = sidx[s];
        }
        load_tile_block<real, P, VEC>(t, g, u8, phi, blk, lane);
        constexpr int PH = (P + 1) / 2;  // x planes of the first lane of a pair
        while (__ballot(s < s1)) {
            if (s < s1) {
                real t1[P], d1[P], t2[P], d2[P], t3[P], d3[P];
                bspline_rounded<real, P, false>(st.x, t1, d1, nullptr);
                bspline_rounded<real, P, false>(st.y, t2, d2, nullptr);
                bspline_rounded<real, P, false>(st.z, t3, d3, nullptr);
                const int lc = unpack_loc(st.w);
                const int lx = lc & 31, ly = (lc >> 5) & 31, lz = (lc >> 10) & 31;
                real g1 = 0, g2 = 0, g3 = 0;
#pragma unroll
                for (int ixh = 0; ixh < PH; ++ixh) {
                    const int ix = half ? PH + ixh : ixh;
                    if (ix >= P) break;
                    // spline weights picked with compile-time indices (registers, not scratch)
                    const int ih = PH + ixh < P ? PH + ixh : P - 1;
                    const real d1x = half ? d1[ih] : d1[ixh], t1x = half ? t1[ih] : t1[ixh];
                    real s_tt = 0, s_dt = 0, s_td = 0;
#pragma unroll
                    for (int iy = 0; iy < P; ++iy) {
                        const real *line = blk + ((lx + ix) * BY + (ly + iy)) * SZ + lz;
                        real lt = 0, ld = 0;
#pragma unroll
                        for (int iz = 0; iz < P; ++iz) {
                            const real w = line[iz];
                            lt += w * t3[iz];
                            ld += w * d3[iz];
                        }
                        s_tt += lt * t2[iy];
                        s_dt += lt * d2[iy];
                        s_td += ld * t2[iy];
                    }
                    g1 += s_tt * d1x;
                    g2 += s_dt * t1x;
                    g3 += s_td * t1x;
                }
                g1 += __shfl_xor(g1, 1, WAVE);
                g2 += __shfl_xor(g2, 1, WAVE);
                g3 += __shfl_xor(g3, 1, WAVE);
                if (!half) {
                    const double *es = g.escale;
                    const real rx = (real)es[0] * g1 + (real)es[1] * g2 + (real)es[2] * g3;
                    const real ry = (real)es[3] * g1 + (real)es[4] * g2 + (real)es[5] * g3;
                    const real rz = (real)es[6] * g1 + (real)es[7] * g2 + (real)es[8] * g3;
                    double c = 0.0;
                    combine_out<real>(mode, atom, rx, ry, rz, dq, row, alpha, extra, cself, out, c);
                    acc[0] += c;
                }
            }
            s += WAVE / 2;
            if (s < s1) {
                st = sten[s];
                atom = sidx[s];
            }
        }
    }
    if (part) {
        block_sum<1>(acc, lds);
        if (threadIdx.x == 0) part[blockIdx.x] = acc[0];
    }
}

template <typename real, int P>
__global__ __launch_bounds__(256) void k_gather_combine(int n, const double *__restrict__ pos, PMEGeom g,
                                                        const real *__restrict__ phi, const real4<real> *__restrict__ dq,
                                                        const real4<real> *__restrict__ row, const real *__restrict__ alpha,
                                                        const real4<real> *__restrict__ extra, real cself, int mode,
                                                        real4<real> *__restrict__ out, double *__restrict__ part,
                                                        const int *__restrict__ conv_it, int iter) {
    if (conv_it && iter >= *conv_it) return;
    __shared__ double lds[16];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double acc[1] = {0.0};
    if (i < n) {
        int base[3];
        real f[3];
        stencil<real, P>(pos, i, g, base, f);
        real t1[P], d1[P], t2[P], d2[P], t3[P], d3[P];
        bspline<real, P, false>(f[0], t1, d1, nullptr);
        bspline<real, P, false>(f[1], t2, d2, nullptr);
        bspline<real, P, false>(f[2], t3, d3, nullptr);
        const int K1 = g.K[0], K2 = g.K[1], K3 = g.K[2];
        real g1 = 0, g2 = 0, g3 = 0;
#pragma unroll
        for (int ix = 0; ix < P; ++ix) {
            int gx = base[0] + ix;
            gx -= gx >= K1 ? K1 : 0;
            real s_tt = 0, s_dt = 0, s_td = 0;  // sums over (iy, iz) of phi t2 t3, phi d2 t3, phi t2 d3
#pragma unroll
            for (int iy = 0; iy < P; ++iy) {
                int gy = base[1] + iy;
                gy -= gy >= K2 ? K2 : 0;
                const real *line = phi + ((size_t)gx * K2 + gy) * K3;
                real lt = 0, ld = 0;
#pragma unroll
                for (int iz = 0; iz < P; ++iz) {
                    int gz = base[2] + iz;
                    gz -= gz >= K3 ? K3 : 0;
                    const real v = line[gz];
                    lt += v * t3[iz];
                    ld += v * d3[iz];
                }
                s_tt += lt * t2[iy];
                s_dt += lt * d2[iy];
                s_td += ld * t2[iy];
            }
            g1 += s_tt * d1[ix];
            g2 += s_dt * t1[ix];
            g3 += s_td * t1[ix];
        }
        const double *es = g.escale;
        const real rx = (real)es[0] * g1 + (real)es[1] * g2 + (real)es[2] * g3;
        const real ry = (real)es[3] * g1 + (real)es[4] * g2 + (real)es[5] * g3;
        const real rz = (real)es[6] * g1 + (real)es[7] * g2 + (real)es[8] * g3;
        combine_out<real>(mode, i, rx, ry, rz, dq, row, alpha, extra, cself, out, acc[0]);
    }
    if (part) {
        block_sum<1>(acc, lds);
        if (threadIdx.x == 0) part[blockIdx.x] = acc[0];
    }
}

// phi-weighted sums S[wx][wy][wz] with w = 0 (theta), 1 (dtheta), 2 (d2theta):
// gd_a = S(d along a), gw_a = q S(d along a) + sum_b e_b S(d along a, d along b / d2 if a == b).
template <typename real>
PGM_DEV void force_out(int i, const real4<real> &d, const PMEGeom &g, double s100, double s010, double s001, double s200, double s020,
                       double s002, double s110, double s101, double s011, const double *__restrict__ dd,
                       const double *__restrict__ rowf, double cself, double *__restrict__ rec_dr, double *__restrict__ gp,
                       double *__restrict__ rec_dd) {
    real e[3];
    scaled_dipole<real>(d, g, e);
    const real q = d.w;
    const double gd[3] = {s100, s010, s001};
    const double qq = (double)q, e0 = (double)e[0], e1 = (double)e[1], e2 = (double)e[2];
    const double gw[3] = {qq * s100 + e0 * s200 + e1 * s110 + e2 * s101, qq * s010 + e0 * s110 + e1 * s020 + e2 * s011,
                          qq * s001 + e0 * s101 + e1 * s011 + e2 * s002};
    const double *es = g.escale;
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        const double rdd = es[3 * b] * gd[0] + es[3 * b + 1] * gd[1] + es[3 * b + 2] * gd[2];
        rec_dr[3 * i + b] = es[3 * b] * gw[0] + es[3 * b + 1] * gw[1] + es[3 * b + 2] * gw[2];
        gp[3 * i + b] = KE * (rowf[3 * i + b] + rdd - cself * dd[3 * i + b]);
        if (rec_dd) rec_dd[3 * i + b] = rdd;
    }
}

// Force gather: dU_rec/dd and dU_rec/dr at fixed q, d (the autodiff of pme.py:390-411 written
// out, with the second spline derivative), FP64 outputs; also gp = KE (rowf + dU_rec/dd - c_self d),
// the total dE/dd of the atom for the covalent-frame pull-back.  rec_dd (optional) receives
// dU_rec/dd itself (for the strain derivative).
template <typename real, int P>
__global__ __launch_bounds__(256) void k_gather_forces(int n, int nper, const double *__restrict__ pos, PMEGeom g,
                                                       const real *__restrict__ phi, const real4<real> *__restrict__ dq,
                                                       const double *__restrict__ dd, const double *__restrict__ rowf,
                                                       double cself, double *__restrict__ rec_dr, double *__restrict__ gp,
                                                       double *__restrict__ rec_dd) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int base[3];
    real f[3];
    stencil<real, P>(pos, i, g, base, f);
    real t[3][P], dt[3][P], d2t[3][P];
#pragma unroll
    for (int a = 0; a < 3; ++a) bspline_rounded<real, P, true>(f[a], t[a], dt[a], d2t[a]);
    const real4<real> d = dq[i];
    const int K1 = g.K[0], K2 = g.K[1], K3 = g.K[2];
    phi += (size_t)(i / nper) * K1 * K2 * K3;
    double s100 = 0, s010 = 0, s001 = 0, s200 = 0, s020 = 0, s002 = 0, s110 = 0, s101 = 0, s011 = 0;
#pragma unroll
    for (int ix = 0; ix < P; ++ix) {
        int gx = base[0] + ix;
        gx -= gx >= K1 ? K1 : 0;
        real a_0 = 0, a_y = 0, a_z = 0, a_yy = 0, a_zz = 0, a_yz = 0;
#pragma unroll
        for (int iy = 0; iy < P; ++iy) {
            int gy = base[1] + iy;
            gy -= gy >= K2 ? K2 : 0;
            const real *line = phi + ((size_t)gx * K2 + gy) * K3;
            real l0 = 0, l1 = 0, l2 = 0;
#pragma unroll
            for (int iz = 0; iz < P; ++iz) {
                int gz = base[2] + iz;
                gz -= gz >= K3 ? K3 : 0;
                const real v = line[gz];
                l0 += v * t[2][iz];
                l1 += v * dt[2][iz];
                l2 += v * d2t[2][iz];
            }
            a_0 += l0 * t[1][iy];
            a_y += l0 * dt[1][iy];
            a_z += l1 * t[1][iy];
            a_yy += l0 * d2t[1][iy];
            a_zz += l2 * t[1][iy];
            a_yz += l1 * dt[1][iy];
        }
        s100 += (double)(a_0 * dt[0][ix]);
        s010 += (double)(a_y * t[0][ix]);
        s001 += (double)(a_z * t[0][ix]);
        s200 += (double)(a_0 * d2t[0][ix]);
        s020 += (double)(a_yy * t[0][ix]);
        s002 += (double)(a_zz * t[0][ix]);
        s110 += (double)(a_y * dt[0][ix]);
        s101 += (double)(a_z * dt[0][ix]);
        s011 += (double)(a_yz * t[0][ix]);
    }
    force_out<real>(i, d, g, s100, s010, s001, s200, s020, s002, s110, s101, s011, dd, rowf, cself, rec_dr, gp, rec_dd);
}

// The force gather on tiles: the block and the two lanes per atom of k_gather_tiles, with the second
// derivatives of the splines and k_gather_forces' sums and outputs.
// Bound like k_gather_tiles (19 us alone at 32,768 waters).  Against one thread per atom on the grid in memory (k_gather_forces, which
// untiled grids keep): forces of 9,001 waters 375 -> 345 us, strain of 2,744 waters 303 -> 270, compute of 1,331 waters
// at order 8 1049 -> 1000.
template <typename real, int P, bool VEC>
__global__ __launch_bounds__(WAVE * gather_waves<real>()) void k_gather_forces_tiles(
    PMETiles t, const int *__restrict__ corg, PMEGeom g, const int2 *__restrict__ range, const int *__restrict__ sidx,
    const real4<real> *__restrict__ sten, const real *__restrict__ phi, const real4<real> *__restrict__ dq,
    const double *__restrict__ dd, const double *__restrict__ rowf, double cself, double *__restrict__ rec_dr,
    double *__restrict__ gp, double *__restrict__ rec_dd) {
    constexpr int GW = gather_waves<real>();
    const int bead = (blockIdx.x * GW) / t.ntiles;  // t.ntiles is a multiple of 8
    constexpr int MAXB = P + 7, SZ = MAXB | 1;
    __shared__ real blk_all[GW][MAXB * MAXB * SZ];
    const int lane = threadIdx.x % WAVE, wv = threadIdx.x / WAVE;
    const int tile = blockIdx.x * GW + wv;
    real *blk = blk_all[wv];
    const int BY = t.B[1];
    const int2 rg = range[tile];
    const int s1 = rg.y, lt = tile - bead * t.ntiles;
    const int half = lane & 1;
    int u8[3];
    if (rg.x >= s1 || !octant_tile(corg[lt >> 3], lt & 7, t, u8)) return;
    load_tile_block<real, P, VEC>(t, g, u8, phi + (size_t)bead * g.K[0] * g.K[1] * g.K[2], blk, lane);
    constexpr int PH = (P + 1) / 2;  // x planes of the first lane of a pair
    for (int s = rg.x + (lane >> 1); s < s1; s += WAVE / 2) {
        const real4<real> st = sten[s];
        const int i = sidx[s];
        real tx[P], dx[P], d2x[P], ty[P], dy[P], d2y[P], tz[P], dz[P], d2z[P];
        bspline_rounded<real, P, true>(st.x, tx, dx, d2x);
        bspline_rounded<real, P, true>(st.y, ty, dy, d2y);
        bspline_rounded<real, P, true>(st.z, tz, dz, d2z);
        const int lc = unpack_loc(st.w);
        const int lx = lc & 31, ly = (lc >> 5) & 31, lz = (lc >> 10) & 31;
        double s100 = 0, s010 = 0, s001 = 0, s200 = 0, s020 = 0, s002 = 0, s110 = 0, s101 = 0, s011 = 0;
#pragma unroll
        for (int ixh = 0; ixh < PH; ++ixh) {
            const int ix = half ? PH + ixh : ixh;
            if (ix >= P) break;
            const int ih = PH + ixh < P ? PH + ixh : P - 1;
            const real t_x = half ? tx[ih] : tx[ixh], d_x = half ? dx[ih] : dx[ixh], d2_x = half ? d2x[ih] : d2x[ixh];
            real a_0 = 0, a_y = 0, a_z = 0, a_yy = 0, a_zz = 0, a_yz = 0;
#pragma unroll
            for (int iy = 0; iy < P; ++iy) {
                const real *line = blk + ((lx + ix) * BY + (ly + iy)) * SZ + lz;
                real l0 = 0, l1 = 0, l2 = 0;
#pragma unroll
                for (int iz = 0; iz < P; ++iz) {
                    const real v = line[iz];
                    l0 += v * tz[iz];
                    l1 += v * dz[iz];
                    l2 += v * d2z[iz];
                }
                a_0 += l0 * ty[iy];
                a_y += l0 * dy[iy];
                a_z += l1 * ty[iy];
                a_yy += l0 * d2y[iy];
                a_zz += l2 * ty[iy];
                a_yz += l1 * dy[iy];
            }
            s100 += (double)(a_0 * d_x);
            s010 += (double)(a_y * t_x);
            s001 += (double)(a_z * t_x);
            s200 += (double)(a_0 * d2_x);
            s020 += (double)(a_yy * t_x);
            s002 += (double)(a_zz * t_x);
            s110 += (double)(a_y * d_x);
            s101 += (double)(a_z * d_x);
            s011 += (double)(a_yz * t_x);
        }
        s100 += __shfl_xor(s100, 1, WAVE);
        s010 += __shfl_xor(s010, 1, WAVE);
        s001 += __shfl_xor(s001, 1, WAVE);
        s200 += __shfl_xor(s200, 1, WAVE);
        s020 += __shfl_xor(s020, 1, WAVE);
        s002 += __shfl_xor(s002, 1, WAVE);
        s110 += __shfl_xor(s110, 1, WAVE);
        s101 += __shfl_xor(s101, 1, WAVE);
        s011 += __shfl_xor(s011, 1, WAVE);
        if (!half)
            force_out<real>(i, dq[i], g, s100, s010, s001, s200, s020, s002, s110, s101, s011, dd, rowf, cself, rec_dr, gp, rec_dd);
    }
}

}  // namespace pgm
