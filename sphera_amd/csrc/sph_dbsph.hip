// DB-SPH walls (Domain%tipo = "bsph", 3D, explicit RK1, FP64): the wall
// elements ("semi-particles") of a surface mesh take part in the fluid
// particles' Shepard sums, density and momentum, and carry a density and
// pressure of their own from a partial Riemann problem with the fluid.
//
//   k_dbsph_lists     CalcVarLength.f90:134-140,330-340,462-540,842-877 and, in
//                     the step, Euler.f90:185-241 around it: Gamma, the
//                     fluid-wall list, sigma, rhoSPH_new, dShep, FS, and the
//                     density from rhoSPH_new / Gamma with the EoS
//   k_momentum_dbsph  RHS_momentum_equation.f90:173-177 with inter_EqMoto.f90
//                     (DB-SPH pressure term :229-235, wall terms :286-322)
//   k_dbsph_muscl     Gradients_to_MUSCL.f90:47-91 (with the wall terms of
//                     Gradients_to_MUSCL_boundary.f90 when asked for)
//   k_dbsph_walls     BC_wall_elements.f90:71-158
//   k_dbsph_kinematics DBSPH_kinematics.f90 and the wall move of Euler.f90:152-159
//
// Wall elements do not move.  Their cell lists are built once on the host
// (OrdGrid1.f90:108-137): wstart[c-1] .. wstart[c]-1 index wids, the wall
// elements of cell c in ascending id, and wpos holds the same elements in
// that order as (x, y, z, id) so that a cell's candidates are one contiguous
// read.
#pragma once

namespace sph {

constexpr int SPH_MW = 128;   // fluid-wall list capacity per particle
constexpr int SPH_WF = 128;   // fluid neighbours a wall element gathers
constexpr int DB_G = 8;       // lanes per particle in k_dbsph_lists

// k_dbsph_lists's LDS of a particle: a bit for every place of the merged
// sequence, and DB_INTS words
constexpr int DB_INTS = 3 * 28 + SPH_MW;
__host__ __device__ __forceinline__ int db_words(int nmaxpartj, int cap) {
    return ((nmaxpartj < cap ? nmaxpartj : cap) + SPH_MW + 2 * DB_G) / 32 + 1;
}

// wall-element tables: w0 = (x, y, z, weight), w1 = (normal, volume),
// w2 = (velocity, mass)
struct DWall {
    const double4* w0;
    const double4* w1;
    const double4* w2;
    const int* wstart;
    const int* wids;
    const int* wcell;
    const double4* wpos;
};

// MODE 0: the pre-loop's first call (on_going_time_step = -2: Gamma = sigma,
// or 1 without wall neighbours); 1: its second call (Gamma kept, FS set);
// 2: inside Euler after OrdGrid1 (Gamma += dShep dt before the sums, then
// dden / Gamma and the density and pressure of the particle)
// The sums take the cells in the reference's order (y, x, z nest): the fluid
// neighbours of a cell (their list entries carry the stencil code (dx+1) +
// 3(dy+1) + 9(dz+1) and come in this order, ascending pg index in a cell), then
// its wall elements.  Bound by latency: walking the 27 cells one after the
// other, each with its dependent loads, took 139 us at 2,000 particles and 191
// at 70,000.  So DB_G lanes of a particle first find the wall elements of all
// cells side by side and mark their places in the merged sequence, then run
// through that sequence two places a lane at a time: 42 and 114 us.
template <int MODE>
__global__ __launch_bounds__(256) void k_dbsph_lists(
    DPC* Pp, DWall W, const double4* __restrict__ xm, const double4* __restrict__ vel,
    const double2* __restrict__ rp, const int* __restrict__ cell, const uint32_t* __restrict__ nbr,
    const int* __restrict__ nnb,
    const double* __restrict__ gam_in, const double* __restrict__ dsh_in, double* __restrict__ gam_out,
    double* __restrict__ dsh_out, double* __restrict__ sig_out, double* __restrict__ rsph_out,
    int* __restrict__ fs_out, int* __restrict__ nfw, int* __restrict__ fwl, int* __restrict__ wwet,
    double* __restrict__ dden, double2* __restrict__ rp_out, const double* scal, int* iscal) {
    DPC& P = *Pp;
    extern __shared__ uint32_t db_lds[];
    const int np = blockDim.x / DB_G, words = db_words(P.nmaxpartj, P.cap);
    const int q = threadIdx.x / DB_G, g = threadIdx.x % DB_G;
    uint32_t* bm = db_lds + q * (words + DB_INTS);  // merged positions that are wall elements
    int* wa = reinterpret_cast<int*>(bm + words);   // first wall element of cell t
    int* pre = wa + 28;                             // wall elements of the cells before cell t
    int* cnt = pre + 28;                            // fluid entries of the cells up to cell t
    int* ids = cnt + 28;                            // the particle's wall elements
    const int i = xcd_block(gridDim.x) * np + q;
    const int gb = (threadIdx.x & 63) & ~(DB_G - 1);  // the group's first lane
    const uint64_t gmask = (1ull << DB_G) - 1ull;
    if (i >= iscal[IS_N]) return;  // whole groups leave together
    const double4 xi = xm[i];
    const double4 vi = vel[i];  // var == vel at every CalcVarLength of the DB-SPH step
    double gamma = 0.0;
    if (MODE == 2) {  // Euler.f90:185-189
        gamma = gam_in[i] + dsh_in[i] * scal[SC_DT];
        if (P.gamma_lim && gamma >= 1.0) gamma = 1.0;
    } else if (MODE == 1) {
        gamma = gam_in[i];
    }
    int nf = 0;
    const int cap = SPH_MW < P.nmaxpartj ? SPH_MW : P.nmaxpartj;
    int ci, cj, ck;
    d_cell_indices(P, cell[i], ci, cj, ck);
    const size_t N = P.cap;
    const int nn = nnb[i];
    // the wall elements of the 27 cells, in the order of the nest
    int mine = 0;
    for (int t = g; t < 27; t += DB_G) {
        const int c = d_cell_number(P, ci + (t / 3) % 3 - 1, cj + t / 9 - 1, ck + t % 3 - 1);
        const int w0 = c ? W.wstart[c - 1] : 0, n = c ? W.wstart[c] - w0 : 0;
        wa[t] = w0;
        pre[t + 1] = n;
        cnt[t] = 0;
        mine += n;
    }
    if ((__ballot(mine > 0) >> gb) & gmask) {
        for (int w = g; w < words; w += DB_G) bm[w] = 0;
        wave_lds_sync();
        for (int k = g; k < nn; k += DB_G) {  // code (dx+1) + 3(dy+1) + 9(dz+1) -> place in the nest
            const int e = (int)(nbr[nb_index(N, i, k)] >> NB_SHIFT);
            atomicAdd(&cnt[9 * (e / 3 % 3) + 3 * (e % 3) + e / 9], 1);
        }
        wave_lds_sync();
        if (g == 0) {
            int a = 0, b = 0;
            pre[0] = 0;
            for (int t = 0; t < 27; ++t) {
                a += cnt[t];
                cnt[t] = a;
                b += pre[t + 1];
                pre[t + 1] = b;
            }
        }
        wave_lds_sync();
        const int total = pre[27];
        for (int w0 = 0; w0 < total; w0 += DB_G) {
            const int w = w0 + g;
            bool inr = false, wet = false;
            int id = 0, t = 0;
            if (w < total) {
                for (int d = 16; d > 0; d >>= 1)
                    if (t + d < 27 && pre[t + d] <= w) t += d;
                const double4 a = W.wpos[wa[t] + w - pre[t]];
                const double R0 = xi.x - a.x, R1 = xi.y - a.y, R2 = xi.z - a.z;
                const double rij = R0 * R0 + R1 * R1 + R2 * R2;
                if (rij <= P.square_doubleh) {
                    inr = true;
                    id = (int)a.w;
                    const double qh = sqrt(rij) / P.h;
                    wet = (int)qh < 2 && (qh * P.h) <= (1.3 * P.dx + W.w0[id].w / 2.0);
                }
            }
            // in candidate order: the elements within 2h take the next list
            // slots while there are any left
            const uint64_t mk = (__ballot(inr) >> gb) & gmask;
            const int slot = nf + __popcll(mk & ((1ull << g) - 1ull));
            if (inr && slot >= cap) atomicAdd(&iscal[IS_DB_OVERFLOW], 1);
            if (inr && slot < cap) {
                fwl[(size_t)slot * P.cap + i] = id;
                if (wet) wwet[id] = 1;
                ids[slot] = id;
                const int pos = cnt[t] + slot;  // after the fluid entries of its cell
                atomicOr(&bm[pos >> 5], 1u << (pos & 31));
            }
            nf = nf + __popcll(mk);
            if (nf > cap) nf = cap;
        }
        wave_lds_sync();
    }
    // the merged sequence, two places a lane at a time
    double s[3] = {0.0, 0.0, 0.0};  // sigma, rhoSPH_new, dShep
    const int len = nn + nf;
    auto entry = [&](int k) { return k < nn ? (int)(nbr[nb_index(N, i, k)] & NB_MASK) : i; };
    int walls = 0;  // before the current places
    for (int p0 = 0; p0 < len; p0 += 2 * DB_G) {
        const uint32_t mask = nf ? (bm[p0 >> 5] >> (p0 & 31)) & ((1u << (2 * DB_G)) - 1u) : 0u;
        d2 x, y, z, rho, c1 = d2(0.0);
        bool on[2];
        d2 m = d2(0.0), vn = d2(0.0), mw = d2(0.0);
        bool wall[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int o = u * DB_G + g, p = p0 + o;
            const int nw = walls + __popc(mask & ((1u << o) - 1u));
            wall[u] = (mask >> o) & 1u;
            on[u] = p < len;
            if (!wall[u]) {
                const int j = on[u] ? entry(p - nw) : i;
                const double4 xj = xm[j];
                x[u] = xj.x;
                y[u] = xj.y;
                z[u] = xj.z;
                m[u] = xj.w;
                rho[u] = rp[j].x;
                vn[u] = 0.0;
            } else {
                const int id = ids[nw];
                const double4 a = W.w0[id], b = W.w1[id], gv = W.w2[id];
                x[u] = a.x;
                y[u] = a.y;
                z[u] = a.z;
                m[u] = b.w;
                mw[u] = gv.w;
                rho[u] = 1.0;
                c1[u] = a.w;
                vn[u] = b.x * (gv.x - vi.x) + b.y * (gv.y - vi.y) + b.z * (gv.z - vi.z);
            }
        }
        walls += __popc(mask);
        const d2 R0 = xi.x - x, R1 = xi.y - y, R2 = xi.z - z;
        const K64x2 K = kvals64x2(P, R0 * R0 + R1 * R1 + R2 * R2, false, false, true);
        const d2 mW = m * K.W;
        const d2 vol = div64(mW, rho, inv64(rho));
        double t[2][3];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const double k1 = on[u] ? K.W[u] : 0.0;
            t[u][0] = !on[u] ? 0.0 : wall[u] ? mW[u] : vol[u];
            t[u][1] = !on[u] ? 0.0 : wall[u] ? mw[u] * k1 : mW[u];
            t[u][2] = wall[u] ? k1 * c1[u] * vn[u] : 0.0;
        }
        add_lanes<DB_G>(s, t[0]);
        add_lanes<DB_G>(s, t[1]);
    }
    const double sigma = s[0], rsph = s[1], dshep = s[2];
    if (g != 0) return;
    nfw[i] = nf;
    sig_out[i] = sigma;
    rsph_out[i] = rsph;
    dsh_out[i] = dshep;
    int fs = 0;
    if (MODE == 0) {  // CalcVarLength.f90:845-853
        if (nf == 0) {
            gamma = 1.0;
        } else {
            gamma = sigma;
            if (P.gamma_lim) gamma = fmin(gamma, 1.0);
        }
    } else {  // CalcVarLength.f90:854-865
        const double msg = fmin(sigma + 0.05, gamma);
        if (P.fs_allowed && msg != gamma) fs = 1;
    }
    if (MODE == 2) {  // Euler.f90:225-239, then EoS_fluid_loop.f90:59-70
        if (P.gamma_lim && nf == 0) gamma = 1.0;
        dden[i] = dden[i] / gamma;
        double rho;
        if (fs == 0) {
            rho = rsph / gamma;
        } else {
            rho = rsph / sigma;
            if (rho < (0.98 * P.den0)) rho = 0.98 * P.den0;
        }
        rp_out[i] = make_double2(rho, P.eps / P.den0 * (rho - P.den0) + P.prif);
    }
    gam_out[i] = gamma;
    fs_out[i] = fs;
}

// RHS_momentum_equation.f90:173-177 and inter_EqMoto.f90 for bsph: the
// symmetric pressure term -m_j (p_i/rho_i^2 + p_j/rho_j^2) r PartKernel(1)
// (no ALE1 complement), the Monaghan and Morris terms as for SA-SPH, then the
// wall elements' pressure terms; the wall shear and semi-particle Morris
// terms read the VSL gradients and semi-particle viscosities, which are zero
// without the VSL model (slip_ID = 0), and add zeros.  acc = (tpres + tdiss
// + tvisc) / Gamma + g; Euler's vel += dt acc (kodvel = 0) is fused.
// Bound by dependent gathers: list entry, record, sum.  G lanes of a particle,
// a step's gathers during the step before: 2,000 particles 48 -> 21 us, 70,000
// 110 -> 90.
template <int G>
__global__ __launch_bounds__(256) void k_momentum_dbsph(
    DPC* Pp, DWall W, const double4* __restrict__ xm, const double4* __restrict__ vel,
    const double2* __restrict__ rp, const uint32_t* __restrict__ nbr, const int* __restrict__ nnb,
    const int* __restrict__ nfw, const int* __restrict__ fwl, const double* __restrict__ gam,
    const double* __restrict__ wdens, const double* __restrict__ wpres, int* __restrict__ lam_out,
    double4* __restrict__ acc_out, double4* __restrict__ vel_out, const double* scal, const int* iscal) {
    DPC& P = *Pp;
    // G lanes per particle; lane 0 adds their terms in list order
    const int i = (xcd_block(gridDim.x) * 256 + (int)threadIdx.x) / G, g = threadIdx.x % G;
    if (i >= iscal[IS_N]) return;  // whole groups leave together
    const size_t N = P.cap;
    const double h = P.h;
    const double4 vi = vel[i];
    const double2 rpi = rp[i];
    const double4 xi = xm[i];
    const double rhoi = rpi.x, pi = rpi.y;
    double tp[3] = {0.0, 0.0, 0.0};
    double s[12];  // td, tv, rvs, tpa
    for (int c = 0; c < 12; ++c) s[c] = 0.0;
    const double celt = P.celerita + P.celerita;
    const double nui = P.kin_visc, nuj = P.kin_visc;
    const bool morris = nui > 1.0e-12 && nuj > 1.0e-12;
    const double ai = pi / (rhoi * rhoi);
    pair_sums64<G, 12>(nbr, N, i, nnb[i], g, false, 0u, s, [](uint32_t) { return Nb{}; },
        [&](int j) {
            const double4 x = xm[j], v = vel[j];
            const double2 q = rp[j];
            return Nb{x.x, x.y, x.z, v.x, v.y, v.z, q.x, q.y, 0.0, x.w};
        },
        [&](d2 (&t)[12], const Nb& a, const Nb& b, bool, bool) {
            const d2 R0 = xi.x - d2{a.x, b.x}, R1 = xi.y - d2{a.y, b.y}, R2 = xi.z - d2{a.z, b.z};
            const d2 rij = R0 * R0 + R1 * R1 + R2 * R2;
            const K64x2 K = kvals64x2(P, rij, true, false, false);
            const d2 rhoj = {a.rho, b.rho}, pj = {a.p, b.p}, amassj = {a.m, b.m};
            const d2 dv0 = d2{a.u, b.u} - vi.x, dv1 = d2{a.v, b.v} - vi.y, dv2 = d2{a.w, b.w} - vi.z;
            const d2 r2 = rhoj * rhoj;
            const d2 alpha = ai + div64(pj, r2, inv64(r2));
            t[9] = -amassj * alpha * R0 * K.K1;
            t[10] = -amassj * alpha * R1 * K.K1;
            t[11] = -amassj * alpha * R2 * K.K1;
            const d2 vrij = -dv0 * R0 - dv1 * R1 - dv2 * R2;
            const d2 rsum = rhoi + rhoj;
            const d2 TermMon = div64(d2(P.alfamon * celt * h), rsum, inv64(rsum));
            t[0] = amassj * TermMon * vrij * R0 * K.K2;
            t[1] = amassj * TermMon * vrij * R1 * K.K2;
            t[2] = amassj * TermMon * vrij * R2 * K.K2;
            const d2 rtil = nui * rhoi + nuj * rhoj + 1.0e-3;
            const double atil = 4.0 * (nui * nuj);
            const d2 visc = div64(amassj * atil, rtil, inv64(rtil));
            const d2 fac = {morris ? visc.x : 0.0, morris ? visc.y : 0.0};
            t[3] = t[6] = fac * (-dv0 * K.K2 * rij);
            t[4] = t[7] = fac * (-dv1 * K.K2 * rij);
            t[5] = t[8] = fac * (-dv2 * K.K2 * rij);
        });
    const double* td = s;
    const double* tv = s + 3;
    const double* rvs = s + 6;
    for (int d = 0; d < 3; ++d) tp[d] = tp[d] + s[9 + d] + 0.0;
    int lam = 0;
    if (P.kin_visc > 0.0) {
        const double apg = sqrt(tp[0] * tp[0] + tp[1] * tp[1] + tp[2] * tp[2]) + P.GI;
        const double amo = sqrt(rvs[0] * rvs[0] + rvs[1] * rvs[1] + rvs[2] * rvs[2]);
        double w = 0.0;
        if (apg != 0.0) w = amo / apg * 100.0;
        lam = (w > 5.0 || apg == 0.0) ? 1 : 0;
    }
    const int nf = nfw[i];
    for (int k0 = 0; k0 < nf; k0 += G) {  // inter_EqMoto.f90:286-297
        const int k = k0 + g;
        double ap[3] = {0.0, 0.0, 0.0};
        if (k < nf) {
            const int id = fwl[(size_t)k * N + i];
            const double4 a = W.w0[id];
            const double4 b = W.w1[id];
            const double wm = W.w2[id].w;
            const double R[3] = {xi.x - a.x, xi.y - a.y, xi.z - a.z};
            K64 K;  // kernel_fw(1) = W, kernel_fw(2) = K1
            kvals64(P, R[0] * R[0] + R[1] * R[1] + R[2] * R[2], true, false, true, K);
            const double wd = wdens[id];
            const double A = pi / (rhoi * rhoi) + wpres[id] / (wd * wd);
            const double nw[3] = {b.x, b.y, b.z};
            for (int d = 0; d < 3; ++d) {
                ap[d] = -wd * a.w * K.W * A * nw[d];
                ap[d] = ap[d] - wm * A * R[d] * K.K1;
            }
        }
        add_lanes<G>(tp, ap);  // past the end: zeros
    }
    if (g != 0) return;
    lam_out[i] = lam;
    const double gm = gam[i];
    double a[3];
    for (int d = 0; d < 3; ++d) a[d] = (tp[d] + td[d] + tv[d]) / gm + P.grav[d];
    acc_out[i] = make_double4(a[0], a[1], a[2], 0.0);
    const double dt = scal[SC_DT];
    vel_out[i] = make_double4(vi.x + dt * a[0], vi.y + dt * a[1], vi.z + dt * a[2], vi.w);
}

// Gradients_to_MUSCL.f90:47-91 for the particles with wall neighbours:
// drho = sum r (rho_j - rho_i) PartKernel(1) m_j/rho_j and dvel(r, :) the
// same of var(r); drho[3 i + d], dvel[9 i + 3 r + d].  As k_momentum_dbsph: 2,000
// particles 49 -> 18 us, 70,000 66 -> 39.
template <int G>
__global__ __launch_bounds__(256) void k_dbsph_muscl(DPC* Pp, DWall W, const double4* __restrict__ xm,
                                                     const double4* __restrict__ vel,
                                                     const double2* __restrict__ rp,
                                                     const uint32_t* __restrict__ nbr,
                                                     const int* __restrict__ nnb, const int* __restrict__ nfw,
                                                     const int* __restrict__ fwl, const double* __restrict__ sig,
                                                     const double* __restrict__ wdens,
                                                     double* __restrict__ drho, double* __restrict__ dvel,
                                                     const int* iscal) {
    DPC& P = *Pp;
    const int i = (xcd_block(gridDim.x) * 256 + (int)threadIdx.x) / G, g = threadIdx.x % G;
    if (i >= iscal[IS_N] || nfw[i] <= 0) return;
    const double4 xi = xm[i];
    const double4 vi = vel[i];
    const double rhoi = rp[i].x;
    double s[12];  // drho, dvel
    for (int c = 0; c < 12; ++c) s[c] = 0.0;
    pair_sums64<G, 12>(nbr, (size_t)P.cap, i, nnb[i], g, false, 0u, s, [](uint32_t) { return Nb{}; },
        [&](int j) {
            const double4 x = xm[j], v = vel[j];
            return Nb{x.x, x.y, x.z, v.x, v.y, v.z, rp[j].x, 0.0, 0.0, x.w};
        },
        [&](d2 (&t)[12], const Nb& a, const Nb& b, bool, bool) {
            const d2 R[3] = {xi.x - d2{a.x, b.x}, xi.y - d2{a.y, b.y}, xi.z - d2{a.z, b.z}};
            const K64x2 K = kvals64x2(P, R[0] * R[0] + R[1] * R[1] + R[2] * R[2], true, false, false);
            const d2 rhoj = {a.rho, b.rho};
            const d2 vol = div64(d2{a.m, b.m}, rhoj, inv64(rhoj));
            const d2 dv[3] = {d2{a.u, b.u} - vi.x, d2{a.v, b.v} - vi.y, d2{a.w, b.w} - vi.z};
            for (int d = 0; d < 3; ++d) t[d] = R[d] * (rhoj - rhoi) * K.K1 * vol;
            for (int r = 0; r < 3; ++r)
                for (int d = 0; d < 3; ++d) t[3 + 3 * r + d] = R[d] * dv[r] * K.K1 * vol;
        });
    if (P.muscl_bnd) {  // Gradients_to_MUSCL_boundary.f90:44-86 (one medium)
        const double sg = sig[i];
        const int nf = nfw[i];
        const double v[3] = {vi.x, vi.y, vi.z};
        for (int k0 = 0; k0 < nf; k0 += G) {
            const int k = k0 + g;
            double ta[12], tb[12];  // past the end: zeros
            for (int c = 0; c < 12; ++c) ta[c] = tb[c] = 0.0;
            if (k < nf) {
                const int id = fwl[(size_t)k * P.cap + i];
                const double4 a = W.w0[id];
                const double4 b = W.w1[id];
                const double4 wv = W.w2[id];
                const double wd = wdens[id];
                const double R[3] = {xi.x - a.x, xi.y - a.y, xi.z - a.z};
                K64 K;  // kernel_fw(1) = W, kernel_fw(2) = K1
                kvals64(P, R[0] * R[0] + R[1] * R[1] + R[2] * R[2], true, false, true, K);
                const double nw[3] = {b.x, b.y, b.z};
                const double vw[3] = {wv.x, wv.y, wv.z};
                const double dr = wd - rhoi;
                const double Ww = a.w * K.W / sg;
                for (int d = 0; d < 3; ++d) ta[d] = dr * nw[d] * Ww;
                for (int r = 0; r < 3; ++r)
                    for (int d = 0; d < 3; ++d) ta[3 + 3 * r + d] = (vw[r] - v[r]) * nw[d] * Ww;
                const double vol = wv.w / wd / sg;
                for (int d = 0; d < 3; ++d) tb[d] = R[d] * dr * K.K1 * vol;
                for (int r = 0; r < 3; ++r)
                    for (int d = 0; d < 3; ++d) tb[3 + 3 * r + d] = R[d] * (vw[r] - v[r]) * K.K1 * vol;
            }
            add_lanes<G>(s, ta, tb);
        }
    }
    if (g != 0) return;
    for (int d = 0; d < 3; ++d) drho[3 * (size_t)i + d] = s[d];
    for (int d = 0; d < 9; ++d) dvel[9 * (size_t)i + d] = s[3 + d];
}

// DBSPH_kinematics.f90:52-107 and Euler.f90:152-159, one thread per sorted
// wall slot: with kinematics records (t, v, omega), the mesh's velocity and
// angular velocity at the step's time (the first record at or after it,
// linearly interpolated from the one before; zero past the last) give each
// element omega x (x - centre) + v; then every element moves by dt vel.
// The elements keep their cells: OrdGrid1.f90:108 bins them on the first
// step only.
__global__ __launch_bounds__(256) void k_dbsph_kinematics(DPC* Pp, const double* __restrict__ kin,
                                                          const int* __restrict__ wids, double4* w0,
                                                          double4* w2, double4* wpos, const double* scal) {
    DPC& P = *Pp;
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= P.nw) return;
    const int id = wids[s];
    const double t = scal[SC_TIME], dt = scal[SC_DT];
    double4 a = w0[id];
    double4 g = w2[id];
    if (P.nkin > 0) {
        double va[3] = {0.0, 0.0, 0.0}, om[3] = {0.0, 0.0, 0.0};
        for (int j = 0; j < P.nkin; ++j) {
            const double* r = &kin[7 * j];
            if (r[0] >= t) {
                if (r[0] == t) {
                    for (int d = 0; d < 3; ++d) {
                        va[d] = r[1 + d];
                        om[d] = r[4 + d];
                    }
                } else {
                    const double* q = &kin[7 * (j - 1)];
                    for (int d = 0; d < 3; ++d) {
                        va[d] = q[1 + d] + (r[1 + d] - q[1 + d]) / (r[0] - q[0]) * (t - q[0]);
                        om[d] = q[4 + d] + (r[4 + d] - q[4 + d]) / (r[0] - q[0]) * (t - q[0]);
                    }
                }
                break;
            }
        }
        const double rel[3] = {a.x - P.kin_c[0], a.y - P.kin_c[1], a.z - P.kin_c[2]};
        g.x = (om[1] * rel[2] - om[2] * rel[1]) + va[0];
        g.y = (om[2] * rel[0] - om[0] * rel[2]) + va[1];
        g.z = (om[0] * rel[1] - om[1] * rel[0]) + va[2];
        w2[id] = g;
    }
    a.x = a.x + dt * g.x;
    a.y = a.y + dt * g.y;
    a.z = a.z + dt * g.z;
    w0[id] = a;
    wpos[s] = make_double4(a.x, a.y, a.z, (double)id);
}

// BC_wall_elements.f90:71-158, one wavefront per wall element: the fluid
// particles within 2h (the ones whose fluid-wall list holds the element),
// each giving the MUSCL left state at the element, rho* = rho_L + (u_L - u_R)
// rho_L / c_L (at least 10) and p* = EoS(rho*) (at least -99 kPa), averaged
// with the Shepard weights m/rho W in ascending pg index (the reference's
// serial scatter order); no neighbours: rho0 and 0; negative pressures set
// to 0 unless allowed.  The lanes share the candidates of the 27 cells and
// the contributions; each contribution goes to its rank by pg index in LDS,
// and one lane sums them in that order.
constexpr int DB_WPB = 4;  // wall elements (wavefronts) per 256-thread block
__global__ __launch_bounds__(256) void k_dbsph_walls(DPC* Pp, DWall W, const double4* __restrict__ xm,
                                                     const double4* __restrict__ vel,
                                                     const double2* __restrict__ rp,
                                                     const int* __restrict__ start,
                                                     const double* __restrict__ drho,
                                                     const double* __restrict__ dvel,
                                                     double* __restrict__ wdens, double* __restrict__ wpres,
                                                     int* iscal) {
    DPC& P = *Pp;
    __shared__ int s_m[DB_WPB];
    __shared__ int s_pre[DB_WPB][28];  // candidates of the cells before cell t
    __shared__ int s_c0[DB_WPB][27];   // first sorted slot of cell t
    __shared__ int s_id[DB_WPB][SPH_WF];
    __shared__ double s_c[DB_WPB][3][SPH_WF];   // Ww, rho* Ww, p* Ww in arrival order
    __shared__ double s_r[DB_WPB][3][SPH_WF];   // the same by rank
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int w = blockIdx.x * DB_WPB + wv;
    const bool active = w < P.nw;
    if (lane == 0) s_m[wv] = 0;
    if (active && lane < 27) {  // the 27 cells around the element's cell
        int ci, cj, ck;
        d_cell_indices(P, W.wcell[w], ci, cj, ck);
        const int c = d_cell_number(P, ci + (lane / 3) % 3 - 1, cj + lane / 9 - 1, ck + lane % 3 - 1);
        const int s0 = c ? start[c - 1] : 0;
        s_c0[wv][lane] = s0;
        s_pre[wv][lane + 1] = c ? start[c] - s0 : 0;
    }
    __syncthreads();
    if (active && lane == 0) {
        s_pre[wv][0] = 0;
        for (int t = 1; t <= 27; ++t) s_pre[wv][t] += s_pre[wv][t - 1];
    }
    __syncthreads();
    if (active) {
        const double4 a = W.w0[w];
        const double4 b = W.w1[w];
        const double4 wg = W.w2[w];
        const double uR = wg.x * b.x + wg.y * b.y + wg.z * b.z;
        const int total = s_pre[wv][27];
        // the cells' candidates as one range: candidate k lies in the cell t
        // with s_pre[t] <= k < s_pre[t + 1]
        for (int k0 = lane; k0 < total; k0 += 64) {
            int lo = 0, hi = 27;  // s_pre[lo] <= k0 < s_pre[hi]
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (s_pre[wv][mid] <= k0) lo = mid; else hi = mid;
            }
            const int s = s_c0[wv][lo] + (k0 - s_pre[wv][lo]);
            const double4 xj = xm[s];
            const double R[3] = {xj.x - a.x, xj.y - a.y, xj.z - a.z};
            const double rij = R[0] * R[0] + R[1] * R[1] + R[2] * R[2];
            if (rij > P.square_doubleh) continue;
            const int k = atomicAdd(&s_m[wv], 1);
            if (k >= SPH_WF) continue;
            const double4 vj = vel[s];
            const double rhoj = rp[s].x;
            const double* g = &drho[3 * (size_t)s];
            const double* V = &dvel[9 * (size_t)s];
            const double rhoL = rhoj - (g[0] * R[0] + g[1] * R[1] + g[2] * R[2]);
            const double v[3] = {vj.x, vj.y, vj.z};
            double uC[3];
            for (int r = 0; r < 3; ++r)
                uC[r] = v[r] - (V[3 * r] * R[0] + V[3 * r + 1] * R[1] + V[3 * r + 2] * R[2]);
            const double uL = uC[0] * b.x + uC[1] * b.y + uC[2] * b.z;
            const double cL = sqrt(P.eps / rhoL);
            double rhostar = rhoL + (uL - uR) * rhoL / cL;
            if (rhostar < 10.0) rhostar = 10.0;
            double pstar = P.eps / P.den0 * (rhostar - P.den0) + P.prif;
            if (pstar < -99.0e3) pstar = -99.0e3;
            K64 K;
            kvals64(P, rij, false, false, true, K);
            const double Ww = xj.w / rhoj * K.W;
            s_id[wv][k] = (int)vj.w;
            s_c[wv][0][k] = Ww;
            s_c[wv][1][k] = rhostar * Ww;
            s_c[wv][2][k] = pstar * Ww;
        }
    }
    __syncthreads();
    const int m = s_m[wv] < SPH_WF ? s_m[wv] : SPH_WF;
    if (active) {
        if (lane == 0 && s_m[wv] > SPH_WF) atomicAdd(&iscal[IS_DB_OVERFLOW], 1);
        for (int k = lane; k < m; k += 64) {  // rank by pg index (ids are distinct)
            const int id = s_id[wv][k];
            int r = 0;
            for (int q = 0; q < m; ++q) r += s_id[wv][q] < id;
            s_r[wv][0][r] = s_c[wv][0][k];
            s_r[wv][1][r] = s_c[wv][1][k];
            s_r[wv][2][r] = s_c[wv][2][k];
        }
    }
    __syncthreads();
    if (active && lane == 0) {
        if (m == 0) {
            wdens[w] = P.den0;
            wpres[w] = 0.0;
        } else {
            double den = 0.0, dsum = 0.0, psum = 0.0;
            for (int r = 0; r < m; ++r) {
                den = den + s_r[wv][0][r];
                dsum = dsum + s_r[wv][1][r];
                psum = psum + s_r[wv][2][r];
            }
            double p = psum / den;
            if (!P.neg_wall_p && p < 0.0) p = 0.0;
            wdens[w] = dsum / den;
            wpres[w] = p;
        }
    }
}

}  // namespace sph
