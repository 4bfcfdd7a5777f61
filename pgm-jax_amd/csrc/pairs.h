// pairs.h -- neighbour rows and the real-space pair kernels of the pGM force field.
//
// Rows: for every atom i, the partners j with |min_image(r_i - r_j)| below a cutoff, stored as
// int32 in row-major (N, cap) order; every pair appears in both rows (no scatter, no atomics: the
// per-atom sums are deterministic).  Rows are built from a cell list every few steps with the
// cutoff + skin, and compacted to the cutoff at every force evaluation.
//
// The force pass uses rowl<real>() lanes per atom (lane l takes entries l, l + lanes, ...), so one
// wave64 covers 64/lanes atoms; the partial sums are reduced across the lanes with shuffles: 16 in
// FP32 (measured 7 % faster than 8), 8 in FP64 (3 % faster than 16).  The
// displacement is formed in FP64 from the FP64 positions (exact for intramolecular pairs whatever
// the absolute coordinates) and then rounded to `real`.
#pragma once

#include "common.h"

namespace pgm {

constexpr int ROWL = 16;  // the most lanes per atom of the force pass (buffer sizes)
template <typename real> constexpr int rowl() { return sizeof(real) == 4 ? 16 : 8; }

// Packed per-atom geometry xr: x, y, z [nm] and R^2 (Gaussian radius squared) [nm^2].
// ---------------------------------------------------------------------------- cells
// Cell of every atom in fractional coordinates of the box; key = bead * ncell + (c0 * n1 + c1) * n2 + c2
// (nper atoms per bead).
__global__ void k_cell_keys(int n, int nper, const double *__restrict__ pos, Box box, int3 nc, int *__restrict__ key,
                            int *__restrict__ atom) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double x = pos[3 * i], y = pos[3 * i + 1], z = pos[3 * i + 2];
    const double *hi = box.hinv;  // u_b = sum_a r_a hinv[a][b]
    double u[3] = {x * hi[0] + y * hi[3] + z * hi[6], x * hi[1] + y * hi[4] + z * hi[7], x * hi[2] + y * hi[5] + z * hi[8]};
    int c[3];
    const int ncs[3] = {nc.x, nc.y, nc.z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        double f = u[a] - floor(u[a]);
        int k = (int)(f * ncs[a]);
        c[a] = k < 0 ? 0 : (k >= ncs[a] ? ncs[a] - 1 : k);
    }
    key[i] = (i / nper) * (nc.x * nc.y * nc.z) + (c[0] * nc.y + c[1]) * nc.z + c[2];
    atom[i] = i;
}

__global__ void k_fill_int(int n, int *__restrict__ p, int v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_iota(int n, int *__restrict__ p) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}

// cell_start[c] / cell_end[c] from the sorted keys.
__global__ void k_cell_bounds(int n, const int *__restrict__ skey, int *__restrict__ start, int *__restrict__ end) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int k = skey[s];
    if (s == 0 || skey[s - 1] != k) start[k] = s;
    if (s == n - 1 || skey[s + 1] != k) end[k] = s + 1;
}

// Full rows within rc_list (cutoff + skin) by a search of the neighbouring cells (27, or every
// distinct cell along an axis with fewer than 3 cells) of the atom's own bead.  One thread per atom;
// the partners come in cell order and, within a cell, in atom order (deterministic).
__global__ void k_build_rows(int n, int nper, const double *__restrict__ pos, Box box, int3 nc, const int *__restrict__ satom,
                             const int *__restrict__ cstart, const int *__restrict__ cend, double rc2, int cap,
                             int *__restrict__ rows, int *__restrict__ count, int *__restrict__ maxcount) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double xi = pos[3 * i], yi = pos[3 * i + 1], zi = pos[3 * i + 2];
    const double *hi = box.hinv;
    const double u[3] = {xi * hi[0] + yi * hi[3] + zi * hi[6], xi * hi[1] + yi * hi[4] + zi * hi[7],
                         xi * hi[2] + yi * hi[5] + zi * hi[8]};
    const int ncs[3] = {nc.x, nc.y, nc.z};
    int c[3], lo[3], hiO[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        double f = u[a] - floor(u[a]);
        int k = (int)(f * ncs[a]);
        c[a] = k < 0 ? 0 : (k >= ncs[a] ? ncs[a] - 1 : k);
        lo[a] = ncs[a] >= 3 ? -1 : 0;
        hiO[a] = ncs[a] >= 3 ? 1 : ncs[a] - 1;
    }
    int cnt = 0;
    int *row = rows + (size_t)i * cap;
    const int cell0 = (i / nper) * (nc.x * nc.y * nc.z);
    for (int o0 = lo[0]; o0 <= hiO[0]; ++o0) {
        const int c0 = (c[0] + o0 + ncs[0]) % ncs[0];
        for (int o1 = lo[1]; o1 <= hiO[1]; ++o1) {
            const int c1 = (c[1] + o1 + ncs[1]) % ncs[1];
            for (int o2 = lo[2]; o2 <= hiO[2]; ++o2) {
                const int c2 = (c[2] + o2 + ncs[2]) % ncs[2];
                const int cell = cell0 + (c0 * nc.y + c1) * nc.z + c2;
                const int s0 = cstart[cell], s1 = cend[cell];
                for (int s = s0; s < s1; ++s) {
                    const int j = satom[s];
                    if (j == i) continue;
                    double dx = xi - pos[3 * j], dy = yi - pos[3 * j + 1], dz = zi - pos[3 * j + 2];
                    min_image(dx, dy, dz, box);
                    if (dx * dx + dy * dy + dz * dz < rc2) {
                        if (cnt < cap) row[cnt] = j;
                        ++cnt;
                    }
                }
            }
        }
    }
    count[i] = cnt;
    atomicMax(maxcount, cnt);
}

// The same rows built cell by cell: one workgroup per cell (bead * ncell + cell, atoms in sorted
// order), its atoms the owners (one thread each, in chunks of blockDim), the neighbouring cells'
// positions staged through LDS in chunks of blockDim and tested by every owner.  Cells and atoms are
// visited in k_build_rows's order; each position is read once per workgroup instead of once per
// owner.  With at least three cells per axis (cell heights >= the list cutoff) the only image of j
// within the cutoff of i lies in the neighbour cell as visited, so positions are wrapped into the
// box (r - floor(r H^-1) H, the cell's own fractional coordinates) and the neighbour cell's lattice
// shift is added when staging: one subtraction per pair instead of a minimum image.  Fewer cells
// per axis keep the per-pair minimum image.
__global__ __launch_bounds__(256) void k_build_rows_cells(int ncell_bead, const double *__restrict__ pos, Box box, int3 nc,
                                                          const int *__restrict__ satom, const int *__restrict__ cstart,
                                                          const int *__restrict__ cend, double rc2, int cap,
                                                          int *__restrict__ rows, int *__restrict__ count,
                                                          int *__restrict__ maxcount) {
    __shared__ double4 sp[256];  // staged candidate: position (shifted) and index (as a double)
    const int cell = blockIdx.x;
    const int bead = cell / ncell_bead, lc = cell - bead * ncell_bead;
    const int own0 = cstart[cell], own1 = cend[cell];
    if (own1 <= own0) return;  // empty cell (uniform)
    const int ncs[3] = {nc.x, nc.y, nc.z};
    const int c[3] = {lc / (nc.y * nc.z), (lc / nc.z) % nc.y, lc % nc.z};
    int lo[3], hiO[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        lo[a] = ncs[a] >= 3 ? -1 : 0;
        hiO[a] = ncs[a] >= 3 ? 1 : ncs[a] - 1;
    }
    const bool shifted = ncs[0] >= 3 && ncs[1] >= 3 && ncs[2] >= 3;
    // position wrapped into the box: r - sum_a floor(u_a) h_a, u = r H^-1
    auto wrapped = [&](int j, double &x, double &y, double &z) {
        x = pos[3 * j];
        y = pos[3 * j + 1];
        z = pos[3 * j + 2];
        if (!shifted) return;
        const double *hi = box.hinv, *h = box.h;
        const double n0 = floor(x * hi[0] + y * hi[3] + z * hi[6]), n1 = floor(x * hi[1] + y * hi[4] + z * hi[7]),
                     n2 = floor(x * hi[2] + y * hi[5] + z * hi[8]);
        x -= n0 * h[0] + n1 * h[3] + n2 * h[6];
        y -= n0 * h[1] + n1 * h[4] + n2 * h[7];
        z -= n0 * h[2] + n1 * h[5] + n2 * h[8];
    };
    for (int o0s = own0; o0s < own1; o0s += blockDim.x) {
        const int s = o0s + threadIdx.x;
        const bool owner = s < own1;
        const int i = owner ? satom[s] : 0;
        double xi = 0.0, yi = 0.0, zi = 0.0;
        if (owner) wrapped(i, xi, yi, zi);
        int cnt = 0;
        int *row = rows + (size_t)i * cap;
        for (int q0 = lo[0]; q0 <= hiO[0]; ++q0) {
            const int c0 = (c[0] + q0 + ncs[0]) % ncs[0];
            for (int q1 = lo[1]; q1 <= hiO[1]; ++q1) {
                const int c1 = (c[1] + q1 + ncs[1]) % ncs[1];
                for (int q2 = lo[2]; q2 <= hiO[2]; ++q2) {
                    const int c2 = (c[2] + q2 + ncs[2]) % ncs[2];
                    const int nb = bead * ncell_bead + (c0 * nc.y + c1) * nc.z + c2;
                    const int s0 = cstart[nb], s1 = cend[nb];
                    // lattice shift of the neighbour cell as visited (wrap across a box face)
                    double shx = 0.0, shy = 0.0, shz = 0.0;
                    if (shifted) {
                        const int q[3] = {q0, q1, q2};
#pragma unroll
                        for (int a = 0; a < 3; ++a) {
                            const int w = c[a] + q[a] < 0 ? -1 : (c[a] + q[a] >= ncs[a] ? 1 : 0);
                            shx += w * box.h[3 * a];
                            shy += w * box.h[3 * a + 1];
                            shz += w * box.h[3 * a + 2];
                        }
                    }
                    for (int t0 = s0; t0 < s1; t0 += blockDim.x) {
                        const int m = min((int)blockDim.x, s1 - t0);
                        __syncthreads();
                        if ((int)threadIdx.x < m) {
                            const int j = satom[t0 + threadIdx.x];
                            double x, y, z;
                            wrapped(j, x, y, z);
                            sp[threadIdx.x] = make_double4(x + shx, y + shy, z + shz, (double)j);
                        }
                        __syncthreads();
                        if (owner) {
                            if (shifted) {
                                // eight candidates' distances at a time (their LDS reads in flight
                                // together), then the hits appended in candidate order
                                for (int u0 = 0; u0 < m; u0 += 8) {
                                    double d2[8];
                                    int jj[8];
#pragma unroll
                                    for (int k = 0; k < 8; ++k) {
                                        const int u = u0 + k < m ? u0 + k : m - 1;
                                        const double4 c4 = sp[u];
                                        jj[k] = (int)c4.w;
                                        const double dx = xi - c4.x, dy = yi - c4.y, dz = zi - c4.z;
                                        d2[k] = dx * dx + dy * dy + dz * dz;
                                    }
#pragma unroll
                                    for (int k = 0; k < 8; ++k)
                                        if (u0 + k < m && d2[k] < rc2 && jj[k] != i) {
                                            if (cnt < cap) row[cnt] = jj[k];
                                            ++cnt;
                                        }
                                }
                            } else {
                                for (int u = 0; u < m; ++u) {
                                    const double4 c4 = sp[u];
                                    const int j = (int)c4.w;
                                    if (j == i) continue;
                                    double dx = xi - c4.x, dy = yi - c4.y, dz = zi - c4.z;
                                    min_image(dx, dy, dz, box);
                                    if (dx * dx + dy * dy + dz * dz < rc2) {
                                        if (cnt < cap) row[cnt] = j;
                                        ++cnt;
                                    }
                                }
                            }
                        }
                    }
                }
            }
        }
        if (owner) count[i] = cnt;
        // the largest count: one atomic per wave, and only above the value already there (a
        // same-address atomic per atom serialises in one L2 channel)
        int m = owner ? cnt : 0;
#pragma unroll
        for (int o = WAVE / 2; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, WAVE));
        if (threadIdx.x % WAVE == 0 && m > __hip_atomic_load(maxcount, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(maxcount, m);
    }
}

// Compacted rows within rc: one wave per atom, ballot + prefix count, one pass.  "Near" partners
// (those for which a series branch of the radial kernels may be taken: (a r)^2 or (beta r)^2
// below 1.05, FP64) fill the row from the front, the others from the back (row[cap - 1 - k]);
// count_near[i] and count[i] - count_near[i] give the two parts, so the kernels run the far part on
// the closed form only (no divergent series).  Entry order within each part is the build order.
__global__ __launch_bounds__(256) void k_compact_rows(int n, const double4 *__restrict__ xr, Box box,
                                                      const int *__restrict__ rows_full, const int *__restrict__ count_full,
                                                      int cap_full, double rc2, double beta2, int cap, int *__restrict__ rows,
                                                      int *__restrict__ count, int *__restrict__ count_near) {
    const int lane = threadIdx.x % WAVE;
    const int i = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (i >= n) return;
    const double4 a = xr[i];
    const int cf = count_full[i] < cap_full ? count_full[i] : cap_full;
    const int *rf = rows_full + (size_t)i * cap_full;
    int *rc = rows + (size_t)i * cap;
    int on = 0, of = 0;
    for (int e0 = 0; e0 < cf; e0 += WAVE) {
        const int e = e0 + lane;
        bool kn = false, kf = false;
        int j = 0;
        if (e < cf) {
            j = rf[e];
            const double4 b = xr[j];
            double dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
            min_image(dx, dy, dz, box);
            const double r2 = dx * dx + dy * dy + dz * dz;
            const bool near = r2 < 1.05 * 2.0 * (a.w + b.w) || beta2 * r2 < 1.05;
            kn = r2 < rc2 && near;
            kf = r2 < rc2 && !near;
        }
        const unsigned long long below = (1ull << lane) - 1ull;
        const unsigned long long mn = __ballot(kn), mf = __ballot(kf);
        const int pn = on + __popcll(mn & below), pf = of + __popcll(mf & below);
        if (kn && pn + of < cap) rc[pn] = j;                 // the far part starts at cap - of
        if (kf && on + pf < cap) rc[cap - 1 - pf] = j;
        on += __popcll(mn);
        of += __popcll(mf);
    }
    if (lane == 0) {
        const int tot = on + of < cap ? on + of : cap;
        count_near[i] = on < tot ? on : tot;
        count[i] = tot;
    }
}

// Sliced-ELL layout of the rows used by the CG matvec: entry e of atom i lives at
// ell(e, i) = (e / RL) * (n * RL) + i * RL + e % RL, so RL lanes per atom, 64 / RL atoms per wave,
// read 64 consecutive words per load.
constexpr int RL = 4;
PGM_DEV size_t ell(int e, int i, int n) { return (size_t)(e / RL) * ((size_t)n * RL) + (size_t)i * RL + (e % RL); }

// Pair tensors of the compacted rows, once per geometry: partner index, G1 and G2 of every entry
// (the dipole field needs only these) in the ELL layout, near part (series branches) first, then
// the far part (closed form).  RL lanes per atom.
template <typename real>
__global__ __launch_bounds__(256) void k_pair_tensors(int n, const int *__restrict__ rows, const int *__restrict__ count,
                                                      const int *__restrict__ count_near, int cap,
                                                      const double4 *__restrict__ xr, Box box, real beta, double rce2,
                                                      int *__restrict__ jell, real *__restrict__ G1, real *__restrict__ G2) {
    const int lane = threadIdx.x % RL;
    const int i = blockIdx.x * (blockDim.x / RL) + threadIdx.x / RL;
    if (i >= n) return;
    const double4 a = xr[i];
    const int c = count[i], cn = count_near[i];
    const size_t o = (size_t)i * cap;
    for (int e = lane; e < c; e += RL) {
        const int j = e < cn ? rows[o + e] : rows[o + cap - 1 - (e - cn)];
        const double4 b = xr[j];
        double dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
        min_image(dx, dy, dz, box);
        const real x = (real)dx, y = (real)dy, z = (real)dz;
        const real aij = rsqrt_(real(2) * (real)(a.w + b.w));
        real G[3] = {real(0), real(0), real(0)};
        if (dx * dx + dy * dy + dz * dz < rce2) {  // electrostatics within the elec cutoff only
            if (e < cn)
                pair_G<real, 3>(aij, beta, x * x + y * y + z * z, G);
            else
                pair_G_far<real, 3>(aij, beta, x * x + y * y + z * z, G);
        }
        const size_t q = ell(e, i, n);
        jell[q] = j;
        G1[q] = G[1];
        G2[q] = G[2];
    }
}

// ---------------------------------------------------------------------------- field rows
// out_i = sum_k de_ik/dd_i = sum_k (-q_k G1 - G2 (d_k . x)) x + G1 d_k, x = r_i - r_k
// (minus the direct-space field at atom i; pgm_jax/md/forcefield.py:1395-1402).
// dq holds (d_x, d_y, d_z, q) per atom; WITHQ adds the charge term.
template <typename real, bool WITHQ>
PGM_DEV void row_field_entry(const double4 &a, const double4 &b, const real4<real> &dk, const Box &box, real g1, real g2,
                             real &ex, real &ey, real &ez) {
    double dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
    min_image(dx, dy, dz, box);
    const real x = (real)dx, y = (real)dy, z = (real)dz;
    const real dkx = dk.x * x + dk.y * y + dk.z * z;
    real cf = -g2 * dkx;
    if (WITHQ) cf -= dk.w * g1;
    ex += cf * x + g1 * dk.x;
    ey += cf * y + g1 * dk.y;
    ez += cf * z + g1 * dk.z;
}

// out_i = sum_k de_ik/dd_i = sum_k (-q_k G1 - G2 (d_k . x)) x + G1 d_k, x = r_i - r_k
// (minus the direct-space field at atom i; pgm_jax/md/forcefield.py:1395-1402), with the partner
// indices and G1, G2 precomputed by k_pair_tensors (ELL layout, RL lanes per atom).  dq holds
// (d_x, d_y, d_z, q) per atom; WITHQ adds the charge term.
template <typename real, bool WITHQ>
__global__ __launch_bounds__(256) void k_row_field(int n, int nper, const int *__restrict__ jell, const int *__restrict__ count,
                                                   const real *__restrict__ G1, const real *__restrict__ G2,
                                                   const double4 *__restrict__ xr, const real4<real> *__restrict__ dq, Box box,
                                                   real4<real> *__restrict__ out, const int *__restrict__ conv_it, int iter,
                                                   Ext3 ext = {}) {
    const int lane = threadIdx.x % RL;
    const int i = blockIdx.x * (blockDim.x / RL) + threadIdx.x / RL;
    if (i >= n || cg_done(conv_it, i / nper, iter)) return;
    const double4 a = xr[i];
    const int c = count[i];
    real ex = 0, ey = 0, ez = 0;
    // Entries in batches of RF_UNROLL per lane: the partner indices and kernels of the batch are
    // loaded first, then the partners' positions and dipoles, so the dependent loads of the batch
    // are in flight together instead of one chain per entry.  Slots past the row's end are masked
    // (own index, zero kernels); the summation order per lane is unchanged.
    constexpr int RF_UNROLL = 4;
    for (int e0 = lane; e0 < c; e0 += RF_UNROLL * RL) {
        int j[RF_UNROLL];
        real g1[RF_UNROLL], g2[RF_UNROLL];
#pragma unroll
        for (int u = 0; u < RF_UNROLL; ++u) {
            const int e = e0 + u * RL;
            const bool ok = e < c;
            const size_t q = ell(ok ? e : 0, i, n);
            j[u] = ok ? jell[q] : i;
            g1[u] = ok ? G1[q] : real(0);
            g2[u] = ok ? G2[q] : real(0);
        }
        double4 b[RF_UNROLL];
        real4<real> d[RF_UNROLL];
#pragma unroll
        for (int u = 0; u < RF_UNROLL; ++u) {
            b[u] = xr[j[u]];
            d[u] = dq[j[u]];
        }
#pragma unroll
        for (int u = 0; u < RF_UNROLL; ++u) row_field_entry<real, WITHQ>(a, b[u], d[u], box, g1[u], g2[u], ex, ey, ez);
    }
    ex = group_sum<RL>(ex);
    ey = group_sum<RL>(ey);
    ez = group_sum<RL>(ez);
    if (lane == 0) {
        real4<real> v;
        v.x = ex;
        v.y = ey;
        v.z = ez;
        v.w = 0;
        if (WITHQ) {  // a uniform external field: its dU/dd is -ext
            v.x -= (real)ext.x;
            v.y -= (real)ext.y;
            v.z -= (real)ext.z;
        }
        out[i] = v;
    }
}

// ---------------------------------------------------------------------------- pair forces
// Per atom i, over its row (forcefield.py:2294-2360, :2116-2146):
//   e_ik  = q_i q_k G0 + (q_i d_k.x - q_k d_i.x) G1 - G2 (d_i.x)(d_k.x) + G1 d_i.d_k
//   de/dx = x [-q_i q_k G1 - t G2 + G3 (d_i.x)(d_k.x) - G2 d_i.d_k] + q_i G1 d_k - q_k G1 d_i
//           - G2 (d_i (d_k.x) + d_k (d_i.x)),   t = q_i d_k.x - q_k d_i.x
//   LJ (intermolecular only): eps (s^12 - 2 s^6), s = rmin/r, (1/r) de/dr = 12 eps (s^6 - s^12)/r^2,
//   one FP64 reciprocal of r^2 per pair; the partner's (rmin/2, sqrt eps, molecule) in one 32-byte
//   load (ljp).
// Electrostatic terms stop at the elec cutoff (r^2 < rce2), LJ at the van der Waals cutoff (r^2 < rcv2;
// pgm_jax/md/forcefield.py:1197-1238, 2355): the rows span both.
// Outputs (FP64): g_el = sum de/dx, g_lj, the row field sum de/dd_i, and per-block energy sums
// (each pair counted in both rows: the caller halves them).  With VIRIAL, also the per-block sums
// of (KE de/dx + de_LJ/dx) (x) X, X = x - o_i + o_k with o the offsets of the atoms from their
// molecules' centres of mass: the pair part of the molecular strain derivative (again twice).
#define PAIR_NEAR pair_G_near<4>(a.w + b.w, beta64, r2d, G);
#define PAIR_FAR pair_G_far<real, 4>(rsqrt_n(real(2) * (real)(a.w + b.w)), beta, (real)r2d, G);
#define PAIR_FORCE_ENTRY(GFUN) \
            const double4 b = xr[j]; \
            double dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z; \
            min_image(dx, dy, dz, box); \
            const real x = (real)dx, y = (real)dy, z = (real)dz; \
            const double r2d = dx * dx + dy * dy + dz * dz; \
            real G[4] = {real(0), real(0), real(0), real(0)}; \
            if (r2d < rce2) { GFUN } \
            const real4<real> dk = dq[j]; \
            const real qk = dk.w; \
            const real dix = di.x * x + di.y * y + di.z * z; \
            const real dkx = dk.x * x + dk.y * y + dk.z * z; \
            const real didk = di.x * dk.x + di.y * dk.y + di.z * dk.z; \
            const real t = qi * dkx - qk * dix; \
            const real ep = qi * qk * G[0] + t * G[1] - G[2] * dix * dkx + G[1] * didk; \
            const real radial = -qi * qk * G[1] - t * G[2] + G[3] * dix * dkx - G[2] * didk; \
            const real qiG1 = qi * G[1], qkG1 = qk * G[1]; \
            const real ge0 = radial * x + qiG1 * dk.x - qkG1 * di.x - G[2] * (di.x * dkx + dk.x * dix); \
            const real ge1 = radial * y + qiG1 * dk.y - qkG1 * di.y - G[2] * (di.y * dkx + dk.y * dix); \
            const real ge2 = radial * z + qiG1 * dk.z - qkG1 * di.z - G[2] * (di.z * dkx + dk.z * dix); \
            gx += (double)ge0; \
            gy += (double)ge1; \
            gz += (double)ge2; \
            ee += (double)ep; \
            const real cfield = -qk * G[1] - G[2] * dkx; \
            fx += (double)(cfield * x + G[1] * dk.x); \
            fy += (double)(cfield * y + G[1] * dk.y); \
            fz += (double)(cfield * z + G[1] * dk.z); \
            const double4 ljk = ljp[j]; \
            const double eps = sei * ljk.y; \
            double l0 = 0.0, l1 = 0.0, l2 = 0.0; \
            if ((int)ljk.z != mi && eps != 0.0 && r2d < rcv2) { \
                const double rmin = rhi + ljk.x; \
                const double ir2 = 1.0 / r2d; \
                const double s2 = rmin * rmin * ir2; \
                const double s6 = s2 * s2 * s2; \
                el += eps * (s6 * s6 - 2.0 * s6); \
                const double dl = eps * 12.0 * (s6 - s6 * s6) * ir2; \
                l0 = dl * dx; \
                l1 = dl * dy; \
                l2 = dl * dz; \
            } \
            lx += l0; \
            ly += l1; \
            lz += l2; \
            if (VIRIAL) { \
                const double X[3] = {dx - oi[0] + off[3 * j], dy - oi[1] + off[3 * j + 1], dz - oi[2] + off[3 * j + 2]}; \
                const double v[3] = {KE * (double)ge0 + l0, KE * (double)ge1 + l1, KE * (double)ge2 + l2}; \
                _Pragma("unroll") for (int p_ = 0; p_ < 3; ++p_) \
                _Pragma("unroll") for (int q_ = 0; q_ < 3; ++q_) w[3 * p_ + q_] += v[p_] * X[q_]; \
            }

// Grid (blocks per bead, beads): partials per block of one bead, at blockIdx.y * gridDim.x + blockIdx.x.
template <typename real, bool VIRIAL>
__global__ __launch_bounds__(256) void k_pair_forces(int nper, const int *__restrict__ rows, const int *__restrict__ count,
                                                     const int *__restrict__ count_near, int cap,
                                                     const double4 *__restrict__ xr, const real4<real> *__restrict__ dq, Box box,
                                                     double beta64, double rce2, double rcv2, const double4 *__restrict__ ljp,
                                                     double *__restrict__ g_el,
                                                     double *__restrict__ g_lj, double *__restrict__ rowf,
                                                     double *__restrict__ epart, const double *__restrict__ off,
                                                     double *__restrict__ wpart, Ext3 ext = {}) {
    __shared__ double lds[9 * 16];
    constexpr int RL_ = rowl<real>();
    const real beta = (real)beta64;
    const int lane = threadIdx.x % RL_;
    const int li = blockIdx.x * (blockDim.x / RL_) + threadIdx.x / RL_;
    const int i = blockIdx.y * nper + li;
    const int pb = blockIdx.y * gridDim.x + blockIdx.x;
    double esum[2] = {0.0, 0.0};
    double w[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (li < nper) {
        const double4 a = xr[i];
        const real4<real> di = dq[i];
        const real qi = di.w;
        const double4 lji = ljp[i];
        const double rhi = lji.x, sei = lji.y;
        const int mi = (int)lji.z;
        const int c = count[i];
        const int *row = rows + (size_t)i * cap;
        double oi[3] = {0.0, 0.0, 0.0};
        if (VIRIAL) {
            oi[0] = off[3 * i];
            oi[1] = off[3 * i + 1];
            oi[2] = off[3 * i + 2];
        }
        double gx = 0, gy = 0, gz = 0, lx = 0, ly = 0, lz = 0, fx = 0, fy = 0, fz = 0, ee = 0, el = 0;
        const int cn = count_near[i];
        for (int e = lane; e < cn; e += RL_) {
            const int j = row[e];
            PAIR_FORCE_ENTRY(PAIR_NEAR)
        }
        for (int e = cap - (c - cn) + lane; e < cap; e += RL_) {
            const int j = row[e];
            PAIR_FORCE_ENTRY(PAIR_FAR)
        }
        gx = group_sum<RL_>(gx);
        gy = group_sum<RL_>(gy);
        gz = group_sum<RL_>(gz);
        lx = group_sum<RL_>(lx);
        ly = group_sum<RL_>(ly);
        lz = group_sum<RL_>(lz);
        fx = group_sum<RL_>(fx);
        fy = group_sum<RL_>(fy);
        fz = group_sum<RL_>(fz);
        if (lane == 0) {
            g_el[3 * i] = gx;
            g_el[3 * i + 1] = gy;
            g_el[3 * i + 2] = gz;
            g_lj[3 * i] = lx;
            g_lj[3 * i + 1] = ly;
            g_lj[3 * i + 2] = lz;
            rowf[3 * i] = fx - ext.x;  // a uniform external field: its dU/dd is -ext
            rowf[3 * i + 1] = fy - ext.y;
            rowf[3 * i + 2] = fz - ext.z;
        }
        esum[0] = ee;
        esum[1] = el;
    }
    block_sum<2>(esum, lds);
    if (threadIdx.x == 0) {
        epart[2 * pb] = esum[0];
        epart[2 * pb + 1] = esum[1];
    }
    if (VIRIAL) {
        block_sum<9>(w, lds);
        if (threadIdx.x == 0)
            for (int k = 0; k < 9; ++k) wpart[9 * pb + k] = w[k];
    }
}

// ---------------------------------------------------------------------------- molecule-blocked field rows
// For systems of 3-site molecules (atoms 3I, 3I+1, 3I+2) the CG row field runs on molecule pairs:
// record (I, J) holds the 9 atom pairs (p of I, k of J), real 6p + k = G1 and 6p + 3 + k = G2 (zero beyond
// the cutoff and for p == k when J == I), so one lane fetches J's three positions and dipoles once for
// nine pair terms instead of one gather per pair.  The record's word (mj[I mcap + e]) is
// J | code << 26: code = the lattice shifts (n_a + 1 in two bits per axis) shared by every pair
// within the cutoff, or MOL_OWN_IMAGES when they differ (the pairs then take min_image each).
//
// The 18 reals of the records are stored in chunks of MCH = 16 records of one molecule, in planes of
// 16 bytes per record (FP32: four planes of four reals and one of two; FP64: nine planes of two),
// so the lanes that take consecutive records read (and the record pass writes) whole 256-byte
// segments.  One 72-byte record per lane in a row made every load instruction of a wave touch 36
// cache lines instead of 8.  The layout does not depend on how many lanes share a molecule.
constexpr int MOL_OWN_IMAGES = 63;
constexpr int MOL_REC = 18;  // reals per record: for each atom of I, G1 and G2 of its three pairs
constexpr int MCH = 16;      // records per chunk
// First real of the chunk of record e of molecule I (mcap a multiple of MCH).
PGM_DEV size_t mchunk(int e, int I, int mcap) { return ((size_t)I * (mcap / MCH) + e / MCH) * (size_t)(MCH * MOL_REC); }
// Offset of real t (0..17) of record e within its chunk.
template <typename real> PGM_DEV int mslot(int e, int t) {
    constexpr int V = 16 / (int)sizeof(real);  // reals per plane entry
    constexpr int FULL = MOL_REC / V * V;      // reals in whole planes
    const int s = e % MCH;
    return t < FULL ? (t / V) * (V * MCH) + s * V + t % V : FULL * MCH + s * (MOL_REC - FULL) + (t - FULL);
}
// The 18 reals of record e of the chunk at g, to or from registers.
// STREAM: non-temporal loads, for records that are not read again before they leave the caches.
template <bool STREAM, typename V> PGM_DEV V stream_load(const V *p) {
    if constexpr (STREAM) return __builtin_nontemporal_load(p);
    return *p;
}
template <bool STREAM> PGM_DEV void mload(const float *__restrict__ g, int e, float (&G)[MOL_REC]) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    const int s = e % MCH;
    const f4 *q = reinterpret_cast<const f4 *>(g) + s;
    const f4 a = stream_load<STREAM>(q), b = stream_load<STREAM>(q + MCH), c = stream_load<STREAM>(q + 2 * MCH),
             d = stream_load<STREAM>(q + 3 * MCH);
    const f2 t = stream_load<STREAM>(reinterpret_cast<const f2 *>(g + 16 * MCH) + s);
    const float v[MOL_REC] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x, c.y, c.z, c.w, d.x, d.y, d.z, d.w, t.x, t.y};
#pragma unroll
    for (int k = 0; k < MOL_REC; ++k) G[k] = v[k];
}
template <bool STREAM> PGM_DEV void mload(const double *__restrict__ g, int e, double (&G)[MOL_REC]) {
    typedef double d2 __attribute__((ext_vector_type(2)));
    const d2 *q = reinterpret_cast<const d2 *>(g) + e % MCH;
#pragma unroll
    for (int k = 0; k < MOL_REC / 2; ++k) {
        const d2 v = stream_load<STREAM>(q + k * MCH);
        G[2 * k] = v.x;
        G[2 * k + 1] = v.y;
    }
}
PGM_DEV void mstore(float *__restrict__ g, int e, const float (&A)[9], const float (&B)[9]) {
    const int s = e % MCH;
    float4 *q = reinterpret_cast<float4 *>(g) + s;
    q[0] = make_float4(A[0], A[1], A[2], B[0]);
    q[MCH] = make_float4(B[1], B[2], A[3], A[4]);
    q[2 * MCH] = make_float4(A[5], B[3], B[4], B[5]);
    q[3 * MCH] = make_float4(A[6], A[7], A[8], B[6]);
    reinterpret_cast<float2 *>(g + 16 * MCH)[s] = make_float2(B[7], B[8]);
}
PGM_DEV void mstore(double *__restrict__ g, int e, const double (&A)[9], const double (&B)[9]) {
    double2 *q = reinterpret_cast<double2 *>(g) + e % MCH;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        q[(3 * p) * MCH] = make_double2(A[3 * p], A[3 * p + 1]);
        q[(3 * p + 1) * MCH] = make_double2(A[3 * p + 2], B[3 * p]);
        q[(3 * p + 2) * MCH] = make_double2(B[3 * p + 1], B[3 * p + 2]);
    }
}
// G1 and G2 of atom p's three pairs of record e (p the same for the whole wave).
PGM_DEV void mload_atom(const float *__restrict__ g, int e, int p, float (&G1)[3], float (&G2)[3]) {
    const int s = e % MCH;
    const float4 *q = reinterpret_cast<const float4 *>(g) + s;
    if (p == 0) {
        const float4 a = q[0];
        const float2 b = *reinterpret_cast<const float2 *>(q + MCH);
        G1[0] = a.x, G1[1] = a.y, G1[2] = a.z, G2[0] = a.w, G2[1] = b.x, G2[2] = b.y;
    } else if (p == 1) {
        const float2 a = *(reinterpret_cast<const float2 *>(q + MCH) + 1);
        const float4 b = q[2 * MCH];
        G1[0] = a.x, G1[1] = a.y, G1[2] = b.x, G2[0] = b.y, G2[1] = b.z, G2[2] = b.w;
    } else {
        const float4 a = q[3 * MCH];
        const float2 b = reinterpret_cast<const float2 *>(g + 16 * MCH)[s];
        G1[0] = a.x, G1[1] = a.y, G1[2] = a.z, G2[0] = a.w, G2[1] = b.x, G2[2] = b.y;
    }
}
PGM_DEV void mload_atom(const double *__restrict__ g, int e, int p, double (&G1)[3], double (&G2)[3]) {
    const double2 *q = reinterpret_cast<const double2 *>(g) + e % MCH + 3 * p * MCH;
    const double2 a = q[0], b = q[MCH], c = q[2 * MCH];
    G1[0] = a.x, G1[1] = a.y, G1[2] = b.x, G2[0] = b.y, G2[1] = c.x, G2[2] = c.y;
}

// Candidate partner molecules of molecule I: the molecules of the atoms in the full (cutoff + skin)
// rows of I's three atoms, deduplicated with a bitmap over the bead's molecules in LDS (`words`
// words per wave) and written in increasing order.  One wave per molecule, no block barriers.
__global__ __launch_bounds__(256) void k_mol_rows(int nmol, int nmol_bead, const int *__restrict__ rows_full,
                                                  const int *__restrict__ count_full, int cap_full, int mcap,
                                                  int *__restrict__ mrows, int *__restrict__ mcount, int *__restrict__ maxcount) {
    extern __shared__ unsigned int mol_bits[];
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    const int I = blockIdx.x * (blockDim.x / WAVE) + w;
    if (I >= nmol) return;
    const int words = (nmol_bead + 31) / 32;
    unsigned int *bits = mol_bits + (size_t)w * words;
    for (int k = lane; k < words; k += WAVE) bits[k] = 0u;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int m0 = (I / nmol_bead) * nmol_bead;
    // the three rows in rounds of four entries per lane and atom, all twelve loads issued first
    int cnt3[3], cmax = 0;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        cnt3[p] = min(count_full[3 * I + p], cap_full);
        cmax = max(cmax, cnt3[p]);
    }
    for (int e0 = 0; e0 < cmax; e0 += 4 * WAVE) {
        int v[3][4];
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = e0 + lane + u * WAVE;
                v[p][u] = e < cnt3[p] ? rows_full[(size_t)(3 * I + p) * cap_full + e] : -1;
            }
        // consecutive entries of a row are often the atoms of one molecule (and its neighbours in
        // index): a lane skips a molecule its left neighbour sets, which keeps most same-word LDS
        // atomics out of one instruction
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int J = v[p][u] >= 0 ? v[p][u] / 3 - m0 : -1;
                const int Jl = __shfl_up(J, 1, WAVE);
                if (J >= 0 && (lane == 0 || Jl != J)) atomicOr(&bits[J >> 5], 1u << (J & 31));
            }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int per = (words + WAVE - 1) / WAVE;
    const int w0 = min(words, lane * per), w1 = min(words, w0 + per);
    int cnt = 0;
    for (int k = w0; k < w1; ++k) cnt += __popc(bits[k]);
    int incl = cnt;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const int t = __shfl_up(incl, o, WAVE);
        if (lane >= o) incl += t;
    }
    int pos = incl - cnt;
    const int total = __shfl(incl, WAVE - 1, WAVE);
    int *mrow = mrows + (size_t)I * mcap;
    for (int k = w0; k < w1; ++k) {
        unsigned int b = bits[k];
        while (b) {
            const int t = __ffs(b) - 1;
            b &= b - 1u;
            if (pos < mcap) mrow[pos] = m0 + 32 * k + t;
            ++pos;
        }
    }
    if (lane == 0) {
        mcount[I] = total;
        if (total > __hip_atomic_load(maxcount, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(maxcount, total);
    }
}

// Records of the molecule blocks, once per geometry (the molecule form of k_compact_rows +
// k_pair_tensors): every candidate J of I with at least one atom pair inside the electrostatics
// cutoff (r^2 < rce2; pairs beyond it hold zeros, and rce2 = rc2 without a split cutoff) is kept, in candidate
// order, its G1 / G2 from the FP64 minimum-image displacement.  WPM waves per molecule, one lane per
// candidate, ballot compaction (with WPM = 4 across the waves of the workgroup, in candidate order too).
//
// The lattice shift is found once per molecule pair, from the atoms 0: where that displacement plus the
// extents of the two molecules stays within half the box along every axis, every atom pair has the same
// shift (min_image would apply none to the shifted displacement), and J is moved by it once.  A wave with
// a candidate near half the box, or a molecule split across the box, takes every pair's own minimum
// image (only possible in boxes little wider than two cutoffs, or with such molecules).
//
// The closed form (both screenings with (a r)^2, (beta r)^2 >= 1) is evaluated for all nine pairs; the
// others (the own molecule, hydrogen bonds: a few pairs per molecule) go to a queue in LDS and are
// evaluated at the end, one per lane, so that a wave runs the series once and not once for every near
// pair of its busiest lane (see record_B).
//
// With ROWS the same pass also writes the compacted atom rows of the force pass (what
// k_compact_rows makes from the full atom rows): for atom 3I + p every 3J + k with r^2 < rc^2,
// the near pairs (r^2 < 1.05 * 2 (R_i^2 + R_j^2) or beta^2 r^2 < 1.05, FP64) from the front of the
// row and the others from the back, in (k, candidate) order per wave chunk; count / count_near
// as k_compact_rows gives them.  (Used for FP32 with WPM = 1; the FP64 variant keeps its registers for
// the tensors and leaves the atom rows to k_compact_rows.)
//
// VALU bound: 186 us alone at 32,768 waters (FP32), 89 % of the instructions the SIMDs can issue in that time.
constexpr int MOL_HELD = 64;                // near pairs a wave holds back for a later round
constexpr int MOL_QUEUE = MOL_HELD + 9 * WAVE;  // and those of one round at most

template <typename real>
PGM_DEV void mol_near_pair(int I, int J, int e, int t, const double4 *__restrict__ xr, const Box &box, double rce2, double beta64, int mcap,
                           real *__restrict__ mg) {
    const int p = t / 3, k = t - 3 * p;
    const double4 a = xr[3 * I + p], b = xr[3 * J + k];
    double dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
    min_image(dx, dy, dz, box);
    const double r2d = dx * dx + dy * dy + dz * dz;
    real G[3] = {real(0), real(0), real(0)};
    if (r2d < rce2) {
        const double w2 = 2.0 * (a.w + b.w);
        if constexpr (sizeof(real) == 4) {
            const double y = (double)rsqrt_n((float)w2);  // 1/sqrt to FP32, then one Newton step
            const double2 A = record_B(y * (1.5 - 0.5 * w2 * y * y), r2d), B = record_B(beta64, r2d);
            G[1] = (real)(A.x - B.x);
            G[2] = (real)(A.y - B.y);
        } else {
            pair_G<real, 3>(1.0 / sqrt(w2), beta64, r2d, G);
        }
    }
    real *g = mg + mchunk(e, I, mcap);
    g[mslot<real>(e, 6 * p + k)] = G[1];
    g[mslot<real>(e, 6 * p + 3 + k)] = G[2];
}

template <typename real, bool ROWS, int WPM>
__global__ __launch_bounds__(256, sizeof(real) == 4 ? 4 : 1) void k_mol_tensors(int nmol, const int *__restrict__ mrows, const int *__restrict__ mcount_full,
                                                     int mcap_full, int mcap, const double4 *__restrict__ xr, Box box,
                                                     double rc2, double rce2, double beta64, int *__restrict__ mj, real *__restrict__ mg,
                                                     int *__restrict__ mcount, int *__restrict__ rows, int acap,
                                                     int *__restrict__ acount, int *__restrict__ acount_near, double beta2) {
    static_assert(!ROWS || WPM == 1, "atom rows are compacted by one wave per molecule");
    __shared__ int2 nearq[4][MOL_QUEUE];
    __shared__ int wsum[4];
    const real beta = (real)beta64;
    const int lane = threadIdx.x % WAVE, wv = threadIdx.x / WAVE;
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int I = WPM == 1 ? blk * 4 + wv : blk;
    if (I >= nmol) return;
    int2 *queue = nearq[wv];
    const double4 a[3] = {xr[3 * I], xr[3 * I + 1], xr[3 * I + 2]};
    // half the box less this molecule's extent from its atom 0, per axis
    const double hx = 0.5 * box.h[0] - fmax(fabs(a[1].x - a[0].x), fabs(a[2].x - a[0].x));
    const double hy = 0.5 * box.h[4] - fmax(fabs(a[1].y - a[0].y), fabs(a[2].y - a[0].y));
    const double hz = 0.5 * box.h[8] - fmax(fabs(a[1].z - a[0].z), fabs(a[2].z - a[0].z));
    const int cf = min(mcount_full[I], mcap_full);
    const int *cand = mrows + (size_t)I * mcap_full;
    int kept = 0, qlen = 0;
    int on[3] = {0, 0, 0}, of[3] = {0, 0, 0};  // atom rows: near / far entries so far
    const unsigned long long below = (1ull << lane) - 1ull;
    for (int e0 = WPM == 1 ? 0 : WAVE * wv; e0 < cf || (WPM > 1 && e0 - WAVE * wv < cf); e0 += WAVE * WPM) {
        const int e = e0 + lane;
        bool keep = false, own = false;
        int J = 0, code = MOL_OWN_IMAGES;
        unsigned near = 0u, akeep = 0u, anear = 0u;
        real G1[9], G2[9];
#pragma unroll
        for (int t = 0; t < 9; ++t) G1[t] = G2[t] = real(0);
        double4 b[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) b[k] = make_double4(0.0, 0.0, 0.0, 0.0);
        int n0[3] = {0, 0, 0};
        bool one = true;  // one shift for the nine pairs
        if (e < cf) {
            J = cand[e];
            own = J == I;
#pragma unroll
            for (int k = 0; k < 3; ++k) b[k] = xr[3 * J + k];
            double dx = a[0].x - b[0].x, dy = a[0].y - b[0].y, dz = a[0].z - b[0].z;
            min_image_n(dx, dy, dz, box, n0);
            one = fabs(dx) + fmax(fabs(b[1].x - b[0].x), fabs(b[2].x - b[0].x)) <= hx &&
                  fabs(dy) + fmax(fabs(b[1].y - b[0].y), fabs(b[2].y - b[0].y)) <= hy &&
                  fabs(dz) + fmax(fabs(b[1].z - b[0].z), fabs(b[2].z - b[0].z)) <= hz;
        }
        const auto pair = [&](int p, int k, double r2d) {
            const int t = 3 * p + k;
            if (r2d >= rc2) return;
            if (ROWS) {
                akeep |= 1u << t;
                if (r2d < 1.05 * 2.0 * (a[p].w + b[k].w) || beta2 * r2d < 1.05) anear |= 1u << t;
            }
            if (r2d >= rce2) return;  // records hold the electrostatic pairs only
            keep = true;
            const real r2 = (real)r2d;
            const real aij = rsqrt_n(real(2) * (real)(a[p].w + b[k].w));
            if (!own && aij * aij * r2 >= real(1) && beta * beta * r2 >= real(1)) {
                real G[3];
                pair_G_far<real, 3>(aij, beta, r2, G);
                G1[t] = G[1];
                G2[t] = G[2];
            } else {
                near |= 1u << t;
            }
        };
        const bool small = n0[0] >= -1 && n0[0] <= 1 && n0[1] >= -1 && n0[1] <= 1 && n0[2] >= -1 && n0[2] <= 1;
        if (!__ballot(!one)) {
            const double f0 = n0[0], f1 = n0[1], f2 = n0[2];
            const double sx = f0 * box.h[0] + f1 * box.h[3] + f2 * box.h[6], sy = f1 * box.h[4] + f2 * box.h[7], sz = f2 * box.h[8];
            if (e < cf) {
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const double bx = b[k].x + sx, by = b[k].y + sy, bz = b[k].z + sz;
#pragma unroll
                    for (int p = 0; p < 3; ++p) {
                        const double dx = a[p].x - bx, dy = a[p].y - by, dz = a[p].z - bz;
                        if (!(own && p == k)) pair(p, k, dx * dx + dy * dy + dz * dz);
                    }
                }
                if (!own && small) code = (n0[0] + 1) | ((n0[1] + 1) << 2) | ((n0[2] + 1) << 4);
            }
        } else if (e < cf) {
            bool first = true, same = true;
            int nc[3] = {0, 0, 0};
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    if (own && p == k) continue;
                    double dx = a[p].x - b[k].x, dy = a[p].y - b[k].y, dz = a[p].z - b[k].z;
                    int n[3];
                    min_image_n(dx, dy, dz, box, n);
                    const double r2d = dx * dx + dy * dy + dz * dz;
                    if (r2d < rce2) {
                        if (first) {
                            nc[0] = n[0], nc[1] = n[1], nc[2] = n[2];
                            first = false;
                        } else if (n[0] != nc[0] || n[1] != nc[1] || n[2] != nc[2]) {
                            same = false;
                        }
                    }
                    pair(p, k, r2d);
                }
            const bool sm = nc[0] >= -1 && nc[0] <= 1 && nc[1] >= -1 && nc[1] <= 1 && nc[2] >= -1 && nc[2] <= 1;
            if (!own && same && sm) code = (nc[0] + 1) | ((nc[1] + 1) << 2) | ((nc[2] + 1) << 4);
        }
        if (ROWS) {  // atom rows of the force pass
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                int *rw = rows + (size_t)(3 * I + p) * acap;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const unsigned bit = 1u << (3 * p + k);
                    const bool kn = (akeep & bit) && (anear & bit), kf = (akeep & bit) && !(anear & bit);
                    const unsigned long long mn = __ballot(kn), mf = __ballot(kf);
                    const int pn = on[p] + __popcll(mn & below), pf = of[p] + __popcll(mf & below);
                    if (kn && pn + of[p] < acap) rw[pn] = 3 * J + k;  // the far part starts at acap - of
                    if (kf && on[p] + pf < acap) rw[acap - 1 - pf] = 3 * J + k;
                    on[p] += __popcll(mn);
                    of[p] += __popcll(mf);
                }
            }
        }
        const unsigned long long m = __ballot(keep);
        int slot0 = kept;  // first slot of this wave's records in the round
        if (WPM > 1) {
            __syncthreads();
            if (lane == 0) wsum[wv] = __popcll(m);
            __syncthreads();
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                if (w < wv) slot0 += wsum[w];
                kept += wsum[w];
            }
        } else {
            kept += __popcll(m);
        }
        const int slot_e = slot0 + __popcll(m & below);
        const bool put = keep && slot_e < mcap;
        if (put) {
            mj[(size_t)I * mcap + slot_e] = (int)((unsigned)J | ((unsigned)code << 26));
            mstore(mg + mchunk(slot_e, I, mcap), slot_e, G1, G2);
        }
        if (!put) near = 0u;
        if (__ballot(near != 0u)) {
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                const bool q = (near >> t) & 1u;
                const unsigned long long mq = __ballot(q);
                if (q) queue[qlen + __popcll(mq & below)] = make_int2((slot_e << 4) | t, J);
                qlen += __popcll(mq);
            }
        }
        const bool last = e0 + WAVE * WPM >= cf + (WPM == 1 ? 0 : WAVE * wv);
        if (qlen > MOL_HELD || (last && qlen)) {  // the queued pairs, after the stores of their records
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            __builtin_amdgcn_wave_barrier();
            for (int u = lane; u < qlen; u += WAVE) {
                const int2 q = queue[u];
                mol_near_pair<real>(I, q.y, q.x >> 4, q.x & 15, xr, box, rce2, beta64, mcap, mg);
            }
            __builtin_amdgcn_wave_barrier();
            qlen = 0;
        }
    }
    if (WPM == 1 ? lane == 0 : threadIdx.x == 0) mcount[I] = kept < mcap ? kept : mcap;
    if (ROWS && lane < 3) {
        const int o = on[lane], f = of[lane];
        const int tot = o + f < acap ? o + f : acap;
        acount_near[3 * I + lane] = o < tot ? o : tot;
        acount[3 * I + lane] = tot;
    }
}

// Row field of the molecule blocks: out_i for the three atoms of I (the same sum as k_row_field over
// the pairs within rc, in molecule-pair order).  RLM lanes per molecule take its records in turn.  Bound by the
// record stream in large systems (32,768 waters: 338 MB, with the gathers 362 MB moved, in 78 us, 4.6 TB/s where a
// copy reaches 4.8), by the partners' gathers and latency in smaller ones.
template <typename real> struct RowArgs {
    int nmol, nmol_bead, mcap;
    const int *mj;
    const real *mg;
    const int *mcount;
    const double4 *xr;
    Box box;
    real4<real> *out;
    Ext3 ext;
};

// Workgroup `block` of the row field.
template <typename real, bool WITHQ, int RLM, bool STREAM>
PGM_DEV void row_field_mol(const RowArgs<real> &A, int block, const real4<real> *__restrict__ dq, const int *__restrict__ conv_it,
                           int iter) {
    const int nmol = A.nmol, nmol_bead = A.nmol_bead, mcap = A.mcap;
    const int *__restrict__ mj = A.mj;
    const real *__restrict__ mg = A.mg;
    const int *__restrict__ mcount = A.mcount;
    const double4 *__restrict__ xr = A.xr;
    const Box &box = A.box;
    real4<real> *__restrict__ out = A.out;
    const Ext3 &ext = A.ext;
    const int lane = threadIdx.x % RLM;
    const int I = block * (blockDim.x / RLM) + threadIdx.x / RLM;
    if (I >= nmol || cg_done(conv_it, I / nmol_bead, iter)) return;
    const double4 a[3] = {xr[3 * I], xr[3 * I + 1], xr[3 * I + 2]};
    real acc[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) acc[t] = real(0);
    const int c = mcount[I];
    const int *words = mj + (size_t)I * mcap;
    for (int e = lane; e < c; e += RLM) {
        const unsigned word = (unsigned)words[e];
        const int J = (int)(word & ((1u << 26) - 1u)), code = (int)(word >> 26);
        real G[MOL_REC];
        mload<STREAM>(mg + mchunk(e, I, mcap), e, G);
        double4 b[3];
        real4<real> d[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            b[k] = xr[3 * J + k];
            d[k] = dq[3 * J + k];
        }
        const bool own = code == MOL_OWN_IMAGES;
        if (!own) {  // the lattice shift shared by the record's pairs moves J once, not every difference
            const double n0 = (double)((code & 3) - 1), n1 = (double)(((code >> 2) & 3) - 1), n2 = (double)(((code >> 4) & 3) - 1);
            const double sx = n0 * box.h[0] + n1 * box.h[3] + n2 * box.h[6], sy = n1 * box.h[4] + n2 * box.h[7], sz = n2 * box.h[8];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                b[k].x += sx;
                b[k].y += sy;
                b[k].z += sz;
            }
        }
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                double dx = a[p].x - b[k].x, dy = a[p].y - b[k].y, dz = a[p].z - b[k].z;
                if (own) min_image(dx, dy, dz, box);
                const real x = (real)dx, y = (real)dy, z = (real)dz;
                const real g1 = G[6 * p + k], g2 = G[6 * p + 3 + k];
                const real dkx = d[k].x * x + d[k].y * y + d[k].z * z;
                real cf = -g2 * dkx;
                if (WITHQ) cf -= d[k].w * g1;
                acc[3 * p] += cf * x + g1 * d[k].x;
                acc[3 * p + 1] += cf * y + g1 * d[k].y;
                acc[3 * p + 2] += cf * z + g1 * d[k].z;
            }
    }
#pragma unroll
    for (int t = 0; t < 9; ++t) acc[t] = group_sum<RLM>(acc[t]);
    if (lane == 0)
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            real4<real> v;
            v.x = acc[3 * p];
            v.y = acc[3 * p + 1];
            v.z = acc[3 * p + 2];
            v.w = 0;
            if (WITHQ) {  // a uniform external field: its dU/dd is -ext
                v.x -= (real)ext.x;
                v.y -= (real)ext.y;
                v.z -= (real)ext.z;
            }
            out[3 * I + p] = v;
        }
}

template <typename real, bool WITHQ, int RLM, bool STREAM>
__global__ __launch_bounds__(256) void k_row_field_mol(RowArgs<real> A, const real4<real> *__restrict__ dq,
                                                       const int *__restrict__ conv_it, int iter) {
    row_field_mol<real, WITHQ, RLM, STREAM>(A, xcd_block(blockIdx.x, gridDim.x), dq, conv_it, iter);
}

// ---------------------------------------------------------------------------- molecule-blocked force pass
// The force pass of k_pair_forces (the same per-atom sums g_el, g_lj, rowf and per-block energy
// partials, each pair again counted from both sides) on the molecule-block records, for 3-site
// molecules when the van der Waals cutoff does not exceed the electrostatic one (every LJ pair then
// lies in a record) and no strain derivative is asked for.  A workgroup takes MOL_FORCE_MOLS molecules, one
// wave for each of their three atoms p, MOL_FORCE_LANES lanes per molecule: with p the same over a wave a
// record's six reals of the atom are two coalesced loads, and the waves of the hydrogens (no LJ) never enter
// the LJ branch.  The partners' atoms go through LDS, wave k fetching atom k of the round's 64 partners (one
// round ahead) for all three: one lane per (atom, record) fetching them itself was bound by the gathers, 576
// address cycles per 64 of them (400 us at 32,768 waters).  On the closed-form
// branch ((a r)^2, (b r)^2 >= 1) the other two radial functions follow from G1, G2 and the two Gaussians
// c_a = 2a/sqrt(pi) exp(-a^2 r^2), c_b likewise: G0 = r^2 G1 + (c_a - c_b) and G3 = (5 G2 - ((2a^2)^2 c_a -
// (2b^2)^2 c_b)) / r^2, the recursion B_n = ((2n-1) B_(n-1) - (2a^2)^(n-1) c) / r^2 of the closed
// form read down and up (no erfc).  Pairs off it (a few per atom: its own molecule, hydrogen bonds)
// are queued per atom in LDS and evaluated after the record loop over the molecule's lanes, in FP64 (see
// pair_G_near).  The terms of a record are summed in `real`, then added to FP64 sums.  Grid (blocks per
// bead, beads).  287 us alone at 32,768 waters (FP32): 62 % of the instructions the SIMDs can issue, the rest
// waits (half of the waves' time) that three waves per SIMD do not cover.
#define MOL_FORCE_TERMS(G0_, G1_, G2_, G3_)                                                            \
    {                                                                                                  \
        const real dix = di.x * x + di.y * y + di.z * z;                                               \
        const real dkx = dk.x * x + dk.y * y + dk.z * z;                                               \
        const real didk = di.x * dk.x + di.y * dk.y + di.z * dk.z;                                     \
        const real qk = dk.w;                                                                          \
        const real t = qi * dkx - qk * dix;                                                            \
        pe += qi * qk * (G0_) + t * (G1_) - (G2_) * dix * dkx + (G1_) * didk;                          \
        const real radial = -qi * qk * (G1_) - t * (G2_) + (G3_) * dix * dkx - (G2_) * didk;           \
        const real qiG1 = qi * (G1_), qkG1 = qk * (G1_);                                               \
        pg0 += radial * x + qiG1 * dk.x - qkG1 * di.x - (G2_) * (di.x * dkx + dk.x * dix);             \
        pg1 += radial * y + qiG1 * dk.y - qkG1 * di.y - (G2_) * (di.y * dkx + dk.y * dix);             \
        pg2 += radial * z + qiG1 * dk.z - qkG1 * di.z - (G2_) * (di.z * dkx + dk.z * dix);             \
        const real cfield = -qk * (G1_) - (G2_) * dkx;                                                 \
        pf0 += cfield * x + (G1_) * dk.x;                                                              \
        pf1 += cfield * y + (G1_) * dk.y;                                                              \
        pf2 += cfield * z + (G1_) * dk.z;                                                              \
    }

constexpr int MOL_FORCE_LANES = 8;
constexpr int MOL_FORCE_MOLS = WAVE / MOL_FORCE_LANES;  // molecules per workgroup of three waves
constexpr int MOL_NEAR_QUEUE = 64;  // queued series pairs per molecule and atom: drained above 64 - 3 MOL_FORCE_LANES
template <typename real>
__global__ __launch_bounds__(3 * WAVE, sizeof(real) == 4 ? 3 : 1) void k_pair_forces_mol(int nper, int mcap, const int *__restrict__ mj,
                                                         const real *__restrict__ mg, const int *__restrict__ mcount,
                                                         const double4 *__restrict__ xr, const real4<real> *__restrict__ dq,
                                                         Box box, double beta64, double rce2, double rcv2,
                                                         const double4 *__restrict__ ljp, double *__restrict__ g_el,
                                                         double *__restrict__ g_lj, double *__restrict__ rowf,
                                                         double *__restrict__ epart, Ext3 ext = {}) {
    constexpr int FL = MOL_FORCE_LANES;
    __shared__ double lds[2 * 16];
    __shared__ int nq[3 * MOL_FORCE_MOLS][MOL_NEAR_QUEUE];  // (record index << 2 | k) of the series pairs of an atom
    __shared__ double2 s_xy[2][3][WAVE], s_zr[2][3][WAVE], s_lj[2][3][WAVE];  // partner atoms, shifted; (rmin/2, sqrt eps)
    __shared__ real4<real> s_d[2][3][WAVE];
    const int lane = threadIdx.x % FL, wl = threadIdx.x % WAVE;
    const int p = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int lm = xcd_block(blockIdx.x, gridDim.x) * MOL_FORCE_MOLS + wl / FL;  // molecule of the bead
    const bool in = 3 * lm < nper;
    const int I = blockIdx.y * (nper / 3) + (in ? lm : 0), i = 3 * I + p;
    const int pb = blockIdx.y * gridDim.x + blockIdx.x;
    int *queue = nq[threadIdx.x / FL];
    const double4 a = xr[i];
    const real4<real> di = dq[i];
    const real qi = di.w;
    const double rhi = ljp[i].x, sei = ljp[i].y;
    const real beta = (real)beta64, fb = real(2) * beta * beta;
    double gx = 0, gy = 0, gz = 0, lx = 0, ly = 0, lz = 0, fx = 0, fy = 0, fz = 0, ee = 0, el = 0;
    const int c = in ? mcount[I] : 0;
    int cmax = c;  // the same for the three waves
#pragma unroll
    for (int o = WAVE / 2; o >= FL; o >>= 1) cmax = max(cmax, __shfl_xor(cmax, o, WAVE));
    const int *words = mj + (size_t)I * mcap;
    int qlen = 0;
    // the lattice shift of a record's word, 0 where the pairs take their own images (returns whether)
    const auto shift = [&](unsigned word, double &sx, double &sy, double &sz) {
        const int code = (int)(word >> 26);
        const bool own = code == MOL_OWN_IMAGES;
        const double n0 = own ? 0.0 : (double)((code & 3) - 1), n1 = own ? 0.0 : (double)(((code >> 2) & 3) - 1),
                     n2 = own ? 0.0 : (double)(((code >> 4) & 3) - 1);
        sx = n0 * box.h[0] + n1 * box.h[3] + n2 * box.h[6];
        sy = n1 * box.h[4] + n2 * box.h[7];
        sz = n2 * box.h[8];
        return own;
    };
    unsigned word = 0u;
    const auto stage = [&](int buf, unsigned w) {  // atom p of the partner of word w
        const int j = 3 * (int)(w & ((1u << 26) - 1u)) + p;
        const double4 b = xr[j];
        const real4<real> d = dq[j];
        const double2 l = *reinterpret_cast<const double2 *>(ljp + j);
        double sx, sy, sz;
        shift(w, sx, sy, sz);
        s_xy[buf][p][wl] = make_double2(b.x + sx, b.y + sy);
        s_zr[buf][p][wl] = make_double2(b.z + sz, b.w);
        s_lj[buf][p][wl] = l;
        s_d[buf][p][wl] = d;
    };
    if (lane < c) {
        word = (unsigned)words[lane];
        stage(0, word);
    }
    for (int e0 = 0, buf = 0; e0 < cmax; e0 += FL, buf ^= 1) {
        const int e = e0 + lane;
        __syncthreads();  // this round's partners are in; the other buffer's readers are done
        unsigned next = 0u;
        if (e + FL < c) {
            next = (unsigned)words[e + FL];
            stage(buf ^ 1, next);
        }
        unsigned nearm = 0u;
        if (e < c) {
            const bool own = (int)(word & ((1u << 26) - 1u)) == I, images = (int)(word >> 26) == MOL_OWN_IMAGES;
            real G1[3], G2[3];
            mload_atom(mg + mchunk(e, I, mcap), e, p, G1, G2);
            real pg0 = 0, pg1 = 0, pg2 = 0, pf0 = 0, pf1 = 0, pf2 = 0, pe = 0;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                if (own && k == p) continue;
                const double2 bxy = s_xy[buf][k][wl], bzr = s_zr[buf][k][wl];
                const real4<real> dk = s_d[buf][k][wl];
                double dx = a.x - bxy.x, dy = a.y - bxy.y, dz = a.z - bzr.x;
                if (images) min_image(dx, dy, dz, box);
                const double r2d = dx * dx + dy * dy + dz * dz;
                if (sei != 0.0) {  // LJ, FP64 as in k_pair_forces
                    const double2 lj = s_lj[buf][k][wl];
                    const double eps = sei * lj.y;
                    if (!own && eps != 0.0 && r2d < rcv2) {
                        const double rmin = rhi + lj.x;
                        const double ir2 = 1.0 / r2d;
                        const double s2 = rmin * rmin * ir2;
                        const double s6 = s2 * s2 * s2;
                        el += eps * (s6 * s6 - 2.0 * s6);
                        const double dl = eps * 12.0 * (s6 - s6 * s6) * ir2;
                        lx += dl * dx;
                        ly += dl * dy;
                        lz += dl * dz;
                    }
                }
                if (r2d >= rce2) continue;
                const real x = (real)dx, y = (real)dy, z = (real)dz;
                const real r2 = (real)r2d;
                const real aij = rsqrt_n(real(2) * (real)(a.w + bzr.y));
                const real sa = aij * aij * r2, sb = beta * beta * r2;
                if (sa >= real(1) && sb >= real(1)) {
                    const real ir = rsqrt_n(r2), ir2 = ir * ir;
                    const real ca = real(TWO_OVER_SQRTPI) * aij * exp_neg(sa);
                    const real cb = real(TWO_OVER_SQRTPI) * beta * exp_neg(sb);
                    const real fa = real(2) * aij * aij;
                    const real g1 = G1[k], g2 = G2[k];
                    const real g0 = r2 * g1 + (ca - cb);
                    const real g3 = (real(5) * g2 - (ca * fa * fa - cb * fb * fb)) * ir2;
                    MOL_FORCE_TERMS(g0, g1, g2, g3)
                } else {
                    nearm |= 1u << k;
                }
            }
            gx += (double)pg0;
            gy += (double)pg1;
            gz += (double)pg2;
            fx += (double)pf0;
            fy += (double)pf1;
            fz += (double)pf2;
            ee += (double)pe;
        }
        word = next;
        if (__ballot(nearm != 0u)) {  // queue the series pairs with those of the molecule's other lanes
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const bool q = (nearm >> k) & 1u;
                const unsigned g = (unsigned)(__ballot(q) >> (wl - lane)) & ((1u << FL) - 1u);
                if (q) queue[qlen + __popc(g & ((1u << lane) - 1u))] = (e << 2) | k;
                qlen += __popc(g);
            }
        }
        if (e0 + FL < cmax && !__ballot(qlen > MOL_NEAR_QUEUE - 3 * FL)) continue;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int u = lane; __ballot(u < qlen); u += FL) {  // the queued series pairs, over the molecule's lanes
            if (u < qlen) {
                const int v = queue[u], k = v & 3;
                const unsigned wn = (unsigned)words[v >> 2];
                const int j = 3 * (int)(wn & ((1u << 26) - 1u)) + k;
                const double4 b = xr[j];
                const real4<real> dk = dq[j];
                double sx, sy, sz;
                const bool im = shift(wn, sx, sy, sz);
                double dx = a.x - (b.x + sx), dy = a.y - (b.y + sy), dz = a.z - (b.z + sz);
                if (im) min_image(dx, dy, dz, box);
                const real x = (real)dx, y = (real)dy, z = (real)dz;
                real G[4];
                pair_G_near<4>(a.w + b.w, beta64, dx * dx + dy * dy + dz * dz, G);
                real pg0 = 0, pg1 = 0, pg2 = 0, pf0 = 0, pf1 = 0, pf2 = 0, pe = 0;
                MOL_FORCE_TERMS(G[0], G[1], G[2], G[3])
                gx += (double)pg0;
                gy += (double)pg1;
                gz += (double)pg2;
                fx += (double)pf0;
                fy += (double)pf1;
                fz += (double)pf2;
                ee += (double)pe;
            }
        }
        __builtin_amdgcn_wave_barrier();
        qlen = 0;
    }
    gx = group_sum<FL>(gx);
    gy = group_sum<FL>(gy);
    gz = group_sum<FL>(gz);
    lx = group_sum<FL>(lx);
    ly = group_sum<FL>(ly);
    lz = group_sum<FL>(lz);
    fx = group_sum<FL>(fx);
    fy = group_sum<FL>(fy);
    fz = group_sum<FL>(fz);
    if (in && lane == 0) {
        g_el[3 * i] = gx;
        g_el[3 * i + 1] = gy;
        g_el[3 * i + 2] = gz;
        g_lj[3 * i] = lx;
        g_lj[3 * i + 1] = ly;
        g_lj[3 * i + 2] = lz;
        rowf[3 * i] = fx - ext.x;  // a uniform external field: its dU/dd is -ext
        rowf[3 * i + 1] = fy - ext.y;
        rowf[3 * i + 2] = fz - ext.z;
    }
    double esum[2] = {ee, el};
    block_sum<2>(esum, lds);
    if (threadIdx.x == 0) {
        epart[2 * pb] = esum[0];
        epart[2 * pb + 1] = esum[1];
    }
}
#undef MOL_FORCE_TERMS

}  // namespace pgm
