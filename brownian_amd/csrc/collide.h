// The per-substep work of one colloid's collisions, of a replica's serial
// replay and of a colloid's update, as device functions of the per-substep
// kernels; reflect_event and transfer are k_groups' too.
#pragma once
#include "bw_device.h"

namespace bw {

// --------------------------------------------------------------- collisions
// One event: back half-step, stochastic reflection with the colloid's rigid
// body velocity, forward half-step (cpp/fluid_colloid_collision.cpp:36-43).
// (bx,by,bz) is the offset in the binned cell (ix,iy,iz), updated in place.
__device__ inline void reflect_event(const Phys &ph, int L, int ix, int iy, int iz, double &bx, double &by,
                                     double &bz, double &vx, double &vy, double &vz, const double *pc,
                                     const double *vcol, const double *wcol, const ReflDraw &dr, double *rs,
                                     bool fp32) {
    const double Ld = (double)L, dt = ph.dt;
    bx = bx - vx * dt * 0.5;
    by = by - vy * dt * 0.5;
    bz = bz - vz * dt * 0.5;
    double ax = (double)ix + bx, ay = (double)iy + by, az = (double)iz + bz;
    double rsx = img1(ax - pc[0], Ld), rsy = img1(ay - pc[1], Ld), rsz = img1(az - pc[2], Ld);
    double ux, uy, uz;
    stochastic_reflection(ph, Ld, ax, ay, az, rsx, rsy, rsz, dr, ux, uy, uz);
    double nx = ux + vcol[0] + (wcol[1] * rsz - wcol[2] * rsy);
    double ny = uy + vcol[1] + (wcol[2] * rsx - wcol[0] * rsz);
    double nz = uz + vcol[2] + (wcol[0] * rsy - wcol[1] * rsx);
    if (fp32) {  // what the velocity store keeps
        nx = (double)(float)nx; ny = (double)(float)ny; nz = (double)(float)nz;
    }
    rs[0] = rsx; rs[1] = rsy; rs[2] = rsz;
    vx = nx; vy = ny; vz = nz;
    bx = bx + vx * dt * 0.5;
    by = by + vy * dt * 0.5;
    bz = bz + vz * dt * 0.5;
}

// momentum and angular-momentum transfer of one event: dump - vel and
// rs x (dump - vel) (cpp/fluid_colloid_collision.cpp:40-42)
__device__ __forceinline__ void transfer(const double *dump, double vx, double vy, double vz, const double *rs,
                                         double *c) {
    double ex = dump[0] - vx, ey = dump[1] - vy, ez = dump[2] - vz;
    c[0] = ex; c[1] = ey; c[2] = ez;
    c[3] = rs[1] * ez - rs[2] * ey;
    c[4] = rs[2] * ex - rs[0] * ez;
    c[5] = rs[0] * ey - rs[1] * ex;
}

// One wave per colloid g: its pair list for this substep, then the particles
// inside g and no other colloid, ranked in the reference's neigh_fl order
// (stencil position, then id) and reflected; the momentum/torque sums are taken
// in that order.  A particle a reflection moved into a later colloid continues
// the reference's colloid loop serially (k_serial).  The pair partners j > g
// (position and cell) are staged in LDS while the pair list is built, so the
// continuation test of every event reads no global memory.
struct PairColl {
    double px, py, pz;
    int cx, cy, cz;
};

struct CollideLds {  // of one wave
    double c[EV_CAP][6];
    PairColl nb[MD_CAP];
    int ne, nnb;
};
template <class Real>
__device__ __forceinline__ void collide_wave(const Phys &ph, const Dev &d, const Fluid<Real> &f, int substep, int r,
                                             int g, CollideLds &s) {
    const bool fp32 = sizeof(Real) == 4;
    const int lane = threadIdx.x & 63;
    // Loads that do not need the replica record go first, at an in-range
    // index (a workgroup's last colloids may lie past its replica).  Entries
    // of the candidate list and of the event bucket past their counts are
    // stale but valid indices, so the candidates' positions and the events'
    // particles are requested with the counts and discarded when unused.
    const int gs = min(g, ph.n_colloid_total - 1);
    const int mdc_n = d.mdc_cnt[gs], ne_s = d.ev_cnt[gs];
    const int js = d.mdc_list[gs * MDC_CAP + lane], slot_s = d.ev_slot[gs * EV_CAP + lane];
    double pg[3], pj[3], vg[3], wg[3];
    int cg[3], cj[3];
    for (int k = 0; k < 3; k++) {
        pg[k] = d.cpos[3 * gs + k];
        pj[k] = d.cpos[3 * js + k];
        vg[k] = d.cvel[3 * gs + k];
        wg[k] = d.comega[3 * gs + k];
        cg[k] = d.ccell[3 * gs + k];
        cj[k] = d.ccell[3 * js + k];
    }
    const int pid_s = f.pid[slot_s], cell_s = f.cell[slot_s];
    const Real pox_s = f.ox[slot_s], poy_s = f.oy[slot_s], poz_s = f.oz[slot_s];
    const Real pvx_s = f.vx[slot_s], pvy_s = f.vy[slot_s], pvz_s = f.vz[slot_s];
    const Rep R = d.rep[r];
    const int L = R.L;
    const double Ld = (double)L;
    const bool valid = g < R.first_colloid + R.nc;
    const long long step = *d.step;
    const bool full = d.md_stale[r] != 0;
    const int ncand = valid ? (full ? R.nc : mdc_n) : 0;
    int ne = 0;
    if (valid) {
        ne = ne_s;
        if (lane == 0) {
            d.ev_cnt[g] = 0;
            if (ne > EV_CAP) {
                int k = atomicAdd(&d.ovf_cnt[r], 1);
                if (k < OVF_CAP) d.ovf_list[r * OVF_CAP + k] = g;
                else atomicOr(d.status, BW_FLAG_EVENT_OVERFLOW);
            } else if (ne > 0 && ph.draws == BW_DRAWS_INJECTED) {
                atomicAdd(&d.ev_total[r], ne);
            }
        }
        if (ne > EV_CAP) ne = 0;  // full bucket: all its events are replayed serially
    }
    int slot = -1, pid = 0, ix = 0, iy = 0, iz = 0;
    long long key = 0x7fffffffffffffffll;
    Real pox = 0, poy = 0, poz = 0, pvx = 0, pvy = 0, pvz = 0;
    if (lane < ne) {
        slot = slot_s;
        pid = pid_s;
        unpack_cell(cell_s, ix, iy, iz);
        pox = pox_s; poy = poy_s; poz = poz_s;
        pvx = pvx_s; pvy = pvy_s; pvz = pvz_s;
    }
    if (valid) {  // pair list of g (cpp/neighbour_list.cpp:27-39), partners j > g into LDS
        const unsigned long long below = (1ull << lane) - 1ull;
        int nmd = 0, nnb = 0;
        for (int base = 0; base < ncand; base += 64) {
            const int m = base + lane;
            int j = -1;
            bool p = false;
            const bool pre = base == 0 && !full;  // this lane's candidate is js, loaded above
            if (m < ncand) {
                j = pre ? js : (full ? R.first_colloid + m : d.mdc_list[g * MDC_CAP + m]);
                p = j != g && (pre ? md_pair_at(ph, Ld, g, j, pg, pj) : md_pair(ph, d, Ld, g, j));
            }
            const unsigned long long b = __ballot(p);
            const int rank = __popcll(b & below);
            if (p && nmd + rank < MD_CAP) {
                const int e = g * MD_CAP + nmd + rank;
                d.md_list[e] = j;
                // the pair's force addend, summed in list order by k_colloid_update
                double pjv[3], t[3];
                for (int k = 0; k < 3; k++) pjv[k] = pre ? pj[k] : d.cpos[3 * j + k];
                force_addend(ph, Ld, g, j, pg, pjv, t);
                for (int k = 0; k < 3; k++) d.md_f[3 * e + k] = t[k];
            }
            nmd += __popcll(b);
            const bool q = p && j > g && !(ph.surrogate && d.cmode[j]);
            const unsigned long long bq = __ballot(q);
            const int rq = __popcll(bq & below);
            if (q && nnb + rq < MD_CAP) {
                PairColl &e = s.nb[nnb + rq];
                if (pre) {
                    e.px = pj[0]; e.py = pj[1]; e.pz = pj[2];
                    e.cx = cj[0]; e.cy = cj[1]; e.cz = cj[2];
                } else {
                    e.px = d.cpos[3 * j]; e.py = d.cpos[3 * j + 1]; e.pz = d.cpos[3 * j + 2];
                    e.cx = d.ccell[3 * j]; e.cy = d.ccell[3 * j + 1]; e.cz = d.ccell[3 * j + 2];
                }
            }
            nnb += __popcll(bq);
        }
        if (lane == 0) {
            if (nmd > MD_CAP) { atomicOr(d.status, BW_FLAG_LIST_OVERFLOW); nmd = MD_CAP; }
            d.md_cnt[g] = nmd;
            s.nnb = min(nnb, MD_CAP);
        }
    }
    wave_sync();  // the wave's pair partners and list visible to its lanes (LDS is per wave)
    if (lane < ne) {
        int dx = pdiff(ix, cg[0], L), dy = pdiff(iy, cg[1], L), dz = pdiff(iz, cg[2], L);
        key = ((long long)stencil_index(dx, dy, dz) << 32) | (unsigned)pid;
    }
    int rank = 0;
    for (int m = 0; m < ne; m++) {
        long long km = lane_value(key, m);
        rank += (km < key) ? 1 : 0;
    }
    if (lane < ne) {
        double bx = pox, by = poy, bz = poz;
        double vx = pvx, vy = pvy, vz = pvz;
        ReflDraw dr;
        double cont[6] = {0, 0, 0, 0, 0, 0};
        const double dump[3] = {vx, vy, vz};
        if (draw_reflection(d, ph, R, step, substep, g, pid, dr)) {
            double rs[3];
            reflect_event(ph, L, ix, iy, iz, bx, by, bz, vx, vy, vz, pg, vg, wg, dr, rs, fp32);
            transfer(dump, vx, vy, vz, rs, cont);
            f.ox[slot] = (Real)bx; f.oy[slot] = (Real)by; f.oz[slot] = (Real)bz;
            f.vx[slot] = (Real)vx; f.vy[slot] = (Real)vy; f.vz[slot] = (Real)vz;
            // The reference goes on to test this particle, now moved, against
            // every later colloid (cpp/fluid_colloid_collision.cpp:30-35).  A
            // later colloid that now contains it is a pair partner of g; if
            // there is one, the rest of the colloid loop is replayed serially.
            const double ax = (double)ix + bx, ay = (double)iy + by, az = (double)iz + bz;
            const int nnb = s.nnb;
#pragma unroll 2
            for (int m = 0; m < nnb; m++) {
                const PairColl &e = s.nb[m];
                if (!in_stencil(ix, iy, iz, e.cx, e.cy, e.cz, L)) continue;
                double rx = img1(e.px - ax, Ld), ry = img1(e.py - ay, Ld), rz = img1(e.pz - az, Ld);
                if ((rx * rx + ry * ry) + rz * rz <= ph.lim_coll) {
                    int c = atomicAdd(&d.cont_cnt[r], 1);
                    if (c < CONT_CAP) {
                        int q = r * CONT_CAP + c;
                        d.cont_slot[q] = slot;
                        d.cont_from[q] = g + 1;
                        for (int kk = 0; kk < 3; kk++) d.cont_dump[3 * q + kk] = dump[kk];
                    } else {
                        atomicOr(d.status, BW_FLAG_CHAIN_OVERFLOW);
                    }
                    break;
                }
            }
        } else {
            atomicOr(d.status, BW_FLAG_DRAW_MISSING);
        }
        for (int k = 0; k < 6; k++) s.c[rank][k] = cont[k];
    }
    if (lane == 0) s.ne = ne;
    wave_sync();
    if (lane == 0 && valid) {
        double a[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll 2
        for (int e = 0; e < s.ne; e++)
            for (int k = 0; k < 6; k++) a[k] = a[k] + s.c[e][k];
        for (int k = 0; k < 3; k++) {
            d.cdv[3 * g + k] = a[k];
            d.cdw[3 * g + k] = a[3 + k];
        }
    }
}

// By one workgroup, after every colloid's collide_wave: the serial list -- particles
// inside several colloids and the events of overflowed buckets (tested from
// the replica's first colloid on, dump = current velocity), and the
// continuations (from the colloid after the reflecting one, dump = velocity
// before that reflection) -- replayed in ascending particle id, each particle
// through the colloids whose stencil holds its binned cell in ascending order
// (cpp/fluid_colloid_collision.cpp:29-49).  Then the injected-draw totals are
// checked and the replica's counters cleared.
struct SerialLds {
    int chain[SERIAL_CAP], src[SERIAL_CAP];
    int nser, cand_n, serial_events, inj_tot;
    int cand[TCL_CAP];
    int wt[COLLIDE_THREADS / 64];
};
template <class Real>
__device__ __forceinline__ void serial_replay(const Phys &ph, const Dev &d, const Fluid<Real> &f, int substep, int r,
                                              SerialLds &sh) {
    const bool fp32 = sizeof(Real) == 4;
    const Rep R = d.rep[r];
    const int L = R.L;
    const double Ld = (double)L;
    const int gend = R.first_colloid + R.nc;
    const long long step = *d.step;
    const int nchain = d.chain_cnt[r], ncont = d.cont_cnt[r], novf = min(d.ovf_cnt[r], OVF_CAP);
    if (threadIdx.x == 0) {
        sh.serial_events = 0;
        sh.inj_tot = 0;
        sh.nser = 0;
    }
    __syncthreads();
    if (nchain > 0 || ncont > 0 || novf > 0) {
        if (threadIdx.x == 0) {
            int n = 0;
            int nch = min(nchain, CHAIN_CAP);
            if (nchain > CHAIN_CAP) atomicOr(d.status, BW_FLAG_CHAIN_OVERFLOW);
            for (int i = 0; i < nch && n < SERIAL_CAP; i++, n++) { sh.chain[n] = d.chain_slot[r * CHAIN_CAP + i]; sh.src[n] = -1; }
            int nco = min(ncont, CONT_CAP);
            if (ncont > CONT_CAP) atomicOr(d.status, BW_FLAG_CHAIN_OVERFLOW);
            for (int i = 0; i < nco && n < SERIAL_CAP; i++, n++) { sh.chain[n] = d.cont_slot[r * CONT_CAP + i]; sh.src[n] = r * CONT_CAP + i; }
            for (int i = 0; i < novf; i++) {
                int gg = d.ovf_list[r * OVF_CAP + i];
                for (int e = 0; e < EV_CAP && n < SERIAL_CAP; e++, n++) { sh.chain[n] = d.ev_slot[gg * EV_CAP + e]; sh.src[n] = -1; }
            }
            if (n >= SERIAL_CAP) atomicOr(d.status, BW_FLAG_EVENT_OVERFLOW);
            for (int i = 1; i < n; i++) {
                int s = sh.chain[i], q = sh.src[i], p = f.pid[s], j = i - 1;
                while (j >= 0 && f.pid[sh.chain[j]] > p) {
                    sh.chain[j + 1] = sh.chain[j];
                    sh.src[j + 1] = sh.src[j];
                    j--;
                }
                sh.chain[j + 1] = s;
                sh.src[j + 1] = q;
            }
            sh.nser = n;
        }
        __syncthreads();
        const int nser = sh.nser;
        for (int i = 0; i < nser; i++) {
            const int s = sh.chain[i], q = sh.src[i];
            int cx, cy, cz;
            unpack_cell(f.cell[s], cx, cy, cz);
            // colloids whose stencil holds the particle's binned cell, ascending
            const int from = q >= 0 ? d.cont_from[q] : R.first_colloid;
            if (threadIdx.x == 0) sh.cand_n = 0;
            __syncthreads();
            for (int base = from; base < gend; base += blockDim.x) {
                int gg = base + threadIdx.x;
                bool p = gg < gend && !(ph.surrogate && d.cmode[gg]) &&
                         in_stencil(cx, cy, cz, d.ccell[3 * gg], d.ccell[3 * gg + 1], d.ccell[3 * gg + 2], L);
                int tot;
                int idx = block_compact(p, sh.wt, tot);
                if (p && sh.cand_n + idx < TCL_CAP) sh.cand[sh.cand_n + idx] = gg;
                __syncthreads();
                if (threadIdx.x == 0) {
                    // more candidate colloids than the list holds: the replay
                    // would miss collisions, so the capacity error is raised
                    if (sh.cand_n + tot > TCL_CAP) atomicOr(d.status, BW_FLAG_LIST_OVERFLOW);
                    sh.cand_n = min(sh.cand_n + tot, TCL_CAP);
                }
                __syncthreads();
            }
            if (threadIdx.x == 0) {
                const int p = f.pid[s];
                double bx = f.ox[s], by = f.oy[s], bz = f.oz[s];
                double vx = f.vx[s], vy = f.vy[s], vz = f.vz[s];
                double dump[3] = {vx, vy, vz};
                if (q >= 0)
                    for (int kk = 0; kk < 3; kk++) dump[kk] = d.cont_dump[3 * q + kk];
                for (int m = 0; m < sh.cand_n; m++) {
                    const int gg = sh.cand[m];
                    const double *pc = d.cpos + 3 * gg;
                    double ax = (double)cx + bx, ay = (double)cy + by, az = (double)cz + bz;
                    double rx = img1(pc[0] - ax, Ld), ry = img1(pc[1] - ay, Ld), rz = img1(pc[2] - az, Ld);
                    if ((rx * rx + ry * ry) + rz * rz > ph.lim_coll) continue;
                    ReflDraw dr;
                    if (!draw_reflection(d, ph, R, step, substep, gg, p, dr)) {
                        atomicOr(d.status, BW_FLAG_DRAW_MISSING);
                        continue;
                    }
                    double rs[3], c6[6];
                    reflect_event(ph, L, cx, cy, cz, bx, by, bz, vx, vy, vz, pc, d.cvel + 3 * gg, d.comega + 3 * gg,
                                  dr, rs, fp32);
                    transfer(dump, vx, vy, vz, rs, c6);
                    for (int kk = 0; kk < 3; kk++) {
                        d.cdv[3 * gg + kk] += c6[kk];
                        d.cdw[3 * gg + kk] += c6[3 + kk];
                    }
                    sh.serial_events++;
                }
                f.ox[s] = (Real)bx; f.oy[s] = (Real)by; f.oz[s] = (Real)bz;
                f.vx[s] = (Real)vx; f.vy[s] = (Real)vy; f.vz[s] = (Real)vz;
            }
            __syncthreads();
        }
    }
    if (ph.draws == BW_DRAWS_INJECTED) {
        // every GPU event found its (colloid, particle) tuple; equal totals
        // then mean equal sets
        int my_inj = 0;
        for (int i = threadIdx.x; i < R.nc; i += blockDim.x) {
            int base = substep * ph.n_colloid_total + R.first_colloid + i;
            my_inj += d.inj_off[base + 1] - d.inj_off[base];
        }
        atomicAdd(&sh.inj_tot, my_inj);
        __syncthreads();
        if (threadIdx.x == 0 && sh.inj_tot != d.ev_total[r] + sh.serial_events)
            atomicOr(d.status, BW_FLAG_DRAW_MISMATCH);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        d.chain_cnt[r] = 0;
        d.cont_cnt[r] = 0;
        d.ovf_cnt[r] = 0;
        d.ev_total[r] = 0;
    }
}

// One wave per colloid: collision impulse, orientation, WCA force (the pair
// addends k_collide stored with this substep's pair list, summed in list
// order by lane 0), velocity, [run() kick], old force, position into the
// other buffer.  Follows collide_wave of the same
// substep.
struct UpdateLds {  // of one wave
    double f[MD_CAP][3];
};
__device__ __forceinline__ void colloid_update_wave(const Phys &ph, const Dev &d, unsigned flags, int r, int g,
                                                    UpdateLds &s) {
    const int lane = threadIdx.x & 63;
    // Loads that do not need the replica record go first, at an in-range
    // index (a workgroup's last colloids may lie past its replica); the first
    // 64 force addends are requested before their count arrives.
    const int gs = min(g, ph.n_colloid_total - 1);
    ColIn in;  // lane 0: the colloid's own state, in flight with the force terms
    if (lane == 0) colloid_load(ph, d, gs, flags, in);
    int nmd_s = 0;
    double tl[3] = {0, 0, 0};
    if (flags & PH_FORCE) {
        nmd_s = d.md_cnt[gs];
        for (int k = 0; k < 3; k++) tl[k] = d.md_f[3 * (gs * MD_CAP + lane) + k];
    }
    // lanes 0-5: sin (lanes 0-2) or cos (lanes 3-5) of the activity rotation
    // angle about axis lane % 3, from the angular velocity after the impulse,
    // formed as colloid_update forms them (a surrogate-driven colloid's torque
    // may be the mirrored fluid's); lane 0 gathers them below
    const bool driven = (flags & PH_APPLY) && ph.surrogate && d.cmode[gs];
    double torque[3] = {0, 0, 0};
    if (driven)
        for (int k = 0; k < 3; k++) torque[k] = __shfl(lane == 0 ? in.sv[3 + k] : 0.0, 0);
    double tv = 0.0;
    if ((flags & PH_ACTIVITY) && lane < 6) {
        const int k = lane % 3;
        double wk = d.comega[3 * gs + k];
        if (flags & PH_APPLY) {
            const double iw = driven ? (k == 0 ? torque[0] : k == 1 ? torque[1] : torque[2]) : d.cdw[3 * gs + k];
            wk = wk + iw * ph.mass_fl / ph.I_colloid;
        }
        const double b = wk * ph.dt;
        tv = lane < 3 ? sin(b) : cos(b);
    }
    const Rep R = d.rep[r];
    const bool valid = g < R.first_colloid + R.nc;
    int nmd = 0;
    if (valid && (flags & PH_FORCE)) {
        nmd = nmd_s;
        for (int m = lane; m < nmd; m += 64)
            for (int k = 0; k < 3; k++) s.f[m][k] = m < 64 ? tl[k] : d.md_f[3 * (g * MD_CAP + m) + k];
    }
    double trig[6];
    for (int k = 0; k < 6; k++) trig[k] = __shfl(tv, k);
    wave_sync();  // s is the wave's own
    if (valid && lane == 0) {
        double fn[3] = {0, 0, 0};
        if (flags & PH_FORCE) {
            double f0 = 0, f1 = 0, f2 = 0;
#pragma unroll 4
            for (int m = 0; m < nmd; m++) {  // cpp/update.cpp:28 in list order
                f0 = f0 + s.f[m][0];
                f1 = f1 + s.f[m][1];
                f2 = f2 + s.f[m][2];
            }
            fn[0] = f0; fn[1] = f1; fn[2] = f2;
        }
        colloid_update(ph, d, R.L, r, g, flags, fn, in, (flags & PH_ACTIVITY) ? trig : nullptr);
    }
}

}  // namespace bw
