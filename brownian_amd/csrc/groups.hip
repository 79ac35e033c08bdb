// The substeps of a fused MPCD step by groups of colloids (gfx950).
//
// After the rotation pass, colloids that can act on each other within the
// step -- closer than the force cutoff or the reach of a reflected particle,
// plus their displacement bounds, or within reach of one particle -- form a
// group, and k_classify has put every particle that may reach a colloid into
// that colloid's bucket.  Groups are then independent for the whole step:
// k_groups runs all n_sub substeps of a group in one wave or workgroup
// (streaming, stochastic reflection in the reference's event order, serial
// replay, WCA forces, Verlet, activity), with the colloids in LDS, in place of
// four launches per substep over all of them.  A step that has a group of more
// colloids or events than these lists hold, or a reflected particle so fast that
// it may come to another group, is stopped (stop_step) and taken again kernel by
// kernel.  Those launches are bound by latency: 28 us a substep with 8 colloids
// (20^3), 35 with 300 (64^3), 54 with 2400 (128^3), of which the kernels' first
// loads are most.  20 substeps by groups, with the classification and the lists,
// take 0.14, 0.17 and 0.31 ms in place of 0.56, 0.69 and 1.06 (FP32; FP64 at 20^3).
#include "bw_device.h"
#include "collide.h"

namespace bw {

// marks of a working copy's packed cell: at the present substep already; in
// the window's LDS list
constexpr int CURRENT = (int)(1u << 31);
constexpr int IN_WINDOW = -1;

// What a group of NW waves holds: a wave takes a lone colloid, a workgroup of
// four waves 2 to GROUP_MAX (or every group, up to GROUP_WIDE colloids in all).
template <int NW>
struct GroupCaps {
    static constexpr int MAX = NW == 1 ? GROUP_SMALL : GROUP_MAX;  // colloids
    static constexpr int SEL = NW == 1 ? 128 : 384;                // particles that may meet one in the window
    static constexpr int EV = NW == 1 ? 40 : 128;                  // reflection events per substep
    static constexpr int SER = NW == 1 ? 1 : 16;                   // serially replayed particles, of each kind
};

// Working state of one group.  Colloid positions, their cells and FP32 offsets
// in them are double-buffered over the substeps.
template <class Real, int NW>
struct GroupLds {
    static constexpr int MAX = GroupCaps<NW>::MAX, SEL = GroupCaps<NW>::SEL, EV = GroupCaps<NW>::EV,
                         SER = GroupCaps<NW>::SER;
    double pos[2][MAX][3], vel[MAX][3], om[MAX][3], ra[MAX][3], f[MAX][3], of[MAX][3], disp[MAX][3], imp[MAX][6],
        dvw[MAX][6], v0[MAX];
    double pos0[MAX][3];  // at the step's start
    double posw[MAX][3];  // at the window's start
    double pf[MAX * (MAX - 1) / 2 + 1][3];  // pair forces
    double ev[EV][6];     // the events' momentum and torque transfers
    double cont_dump[SER][3];
    long long key[EV];    // stencil position, particle id: the reference's order
    float4 rel[2][MAX];   // FP32 position from the group's origin, displacement bound within the window
    int cell[2][MAX][3], cell0[MAX][3];
    int hot[MAX + 1];     // the buckets' ranges in the group's list of particles
    int g[MAX], sur[MAX], nev[MAX];
    unsigned pair[MAX];   // colloids within the force cutoff
    // the window's particles, then (from SEL) those that had an event in the
    // substep that opened it: bucket entry, id, packed cell, colloids in reach
    int q[SEL + EV], pid[SEL + EV], pc[SEL + EV];
    unsigned reach[SEL + EV];
    Real o[3][SEL + EV], v[3][SEL + EV];
    int ev_i[EV], ev_m[EV];
    unsigned char ord[MAX][EV];
    int chain_i[SER], cont_i[SER], cont_from[SER];
    // counters, by the substep's parity: [0] events, [1] particles inside
    // several colloids, [2] continuations, [3] selected for the window, [4]
    // selected with an event, [5] a colloid left its bound, [6] a fast
    // reflected particle
    int cnt[2][7];
};

// ---- k_groups' rare paths, kept out of line: inlined, they take it from 155
// to 224 VGPRs.  They read the kernel's arguments where the launch put them (a
// reference to by-value arguments would copy all of them to scratch memory).
template <class Real>
struct GroupArgs {
    Phys ph;
    Dev d;
    Fluid<Real> f;
    HotPart<Real> *h;
    int final;
};
template <class Real>
__device__ __forceinline__ const GroupArgs<Real> *group_args() {  // the kernel's only argument
    return (const GroupArgs<Real> *)__builtin_amdgcn_kernarg_segment_ptr();
}
// A particle at (x, y, z) after substep l, with speed v, reflected by the group
// of members m[0..C) of replica r: may it come to an explicitly colliding
// colloid of another group in the rest of the step?  From the colloids'
// positions at the step's start and their displacement bound.
template <class Real>
__device__ __noinline__ bool group_reaches_other(const GroupArgs<Real> *a, int r, double x, double y, double z, double v, int l,
                                                 const int *m, int C) {
    const Phys &ph = a->ph;
    const Dev &d = a->d;
    const Rep R = d.rep[r];
    const double reach = sqrt(ph.lim_coll) + v * ph.dt * (ph.n_sub - 1 - l) + ph.margin, L = (double)R.L;
    for (int g = R.first_colloid; g < R.first_colloid + R.nc; g++) {
        bool member = false;
        for (int c = 0; c < C; c++) member = member || m[c] == g;
        if (member || (ph.surrogate && d.cmode[g])) continue;
        const double ax = img1(d.cpos[3 * g] - x, L), ay = img1(d.cpos[3 * g + 1] - y, L), az = img1(d.cpos[3 * g + 2] - z, L);
        if ((ax * ax + ay * ay) + az * az <= reach * reach) return true;
    }
    return false;
}
// the same for the reflected particle at LDS place i, if it is fast
template <class Real, int NW>
__device__ __noinline__ bool fast_event(const GroupArgs<Real> *a, int r, int l, int C, int i, const GroupLds<Real, NW> *s) {
    const double vx = s->v[0][i], vy = s->v[1][i], vz = s->v[2][i], v = sqrt((vx * vx + vy * vy) + vz * vz);
    int ix, iy, iz;
    unpack_cell(s->pc[i], ix, iy, iz);
    return v * a->ph.ndt > a->ph.group_reach &&
           group_reaches_other<Real>(a, r, (double)ix + (double)s->o[0][i], (double)iy + (double)s->o[1][i],
                                     (double)iz + (double)s->o[2][i], v, l, s->g, C);
}
// the surrogate-driven colloid c's impulse and torque of a substep (as
// colloid_load forms them), in place of its events'
template <class Real, int NW>
__device__ __noinline__ void surrogate_impulse(const GroupArgs<Real> *a, int c, GroupLds<Real, NW> *s) {
    const Dev &d = a->d;
    const int g = s->g[c];
    const ShellPay pay = shell_pay(a->ph, d, g, s->ra[c]);
    const unsigned long long *q = d.sacc + (size_t)SUR_ACC * g;
    for (int k = 0; k < 3; k++) {
        s->dvw[c][k] = pay.lin ? d.csur[6 * g + k] : -unfixq(q[k]) / a->ph.n_sub;
        s->dvw[c][3 + k] = pay.ang ? d.csur[6 * g + 3 + k] : -unfixq(q[3 + k]) / a->ph.n_sub;
    }
}
template <class Real>
__device__ __noinline__ void injected_reflection(const GroupArgs<Real> *a, int r, int substep, int g, int pid, double *out) {
    ReflDraw dr;
    const bool found = draw_reflection(a->d, a->ph, a->d.rep[r], 0, substep, g, pid, dr);
    for (int k = 0; k < 6; k++) out[k] = found ? dr.v[k] : NAN;
}
// The serial replay of a substep, by one lane: n_chain particles inside several
// colloids (tested from the first colloid on) and n_cont continuations, in
// ascending id, each through the colloids whose stencil holds its binned cell
// (cpp/fluid_colloid_collision.cpp:29-49).  Returns its reflections, or'ed with
// REPLAY_MISSING (an injected draw) and REPLAY_ESCAPED (group_reaches_other).
constexpr int REPLAY_MISSING = 1 << 30, REPLAY_ESCAPED = 1 << 29;
template <class Real, int NW>
__device__ __noinline__ int replay(const GroupArgs<Real> *a, int r, int l, int par, int C, int n_chain, int n_cont,
                                   unsigned all, GroupLds<Real, NW> *sp) {
    const Phys &ph = a->ph;
    const Dev &d = a->d;
    GroupLds<Real, NW> &s = *sp;
    const Rep R = d.rep[r];
    const long long step = *d.step;
    const int L = R.L;
    const double Ld = (double)L;
    int last_pid = -1, n = 0, flags = 0;
    for (int it = 0; it < n_chain + n_cont; it++) {
        int best = -1, best_pid = 0x7fffffff;  // the next id
        for (int j = 0; j < n_chain + n_cont; j++) {
            const int p = s.pid[j < n_chain ? s.chain_i[j] : s.cont_i[j - n_chain]];
            if (p > last_pid && p < best_pid) { best = j; best_pid = p; }
        }
        if (best < 0) break;
        last_pid = best_pid;
        const int i = best < n_chain ? s.chain_i[best] : s.cont_i[best - n_chain];
        int cx, cy, cz;
        unpack_cell(s.pc[i], cx, cy, cz);
        double bx = s.o[0][i], by = s.o[1][i], bz = s.o[2][i];
        double vx = s.v[0][i], vy = s.v[1][i], vz = s.v[2][i];
        double dump[3] = {vx, vy, vz};
        if (best >= n_chain)
            for (int k = 0; k < 3; k++) dump[k] = s.cont_dump[best - n_chain][k];
        for (int m = best < n_chain ? 0 : s.cont_from[best - n_chain]; m < C; m++) {
            if (s.sur[m] || !in_stencil(cx, cy, cz, s.cell[par][m][0], s.cell[par][m][1], s.cell[par][m][2], L)) continue;
            const double *pc = s.pos[par][m];
            const double ax = (double)cx + bx, ay = (double)cy + by, az = (double)cz + bz;
            const double rx = img1(pc[0] - ax, Ld), ry = img1(pc[1] - ay, Ld), rz = img1(pc[2] - az, Ld);
            if ((rx * rx + ry * ry) + rz * rz > ph.lim_coll) continue;
            ReflDraw dr;
            if (!draw_reflection(d, ph, R, step, l, s.g[m], best_pid, dr)) {
                flags |= REPLAY_MISSING;
                continue;
            }
            double rs[3], c6[6];
            reflect_event(ph, L, cx, cy, cz, bx, by, bz, vx, vy, vz, pc, s.vel[m], s.om[m], dr, rs, sizeof(Real) == 4);
            transfer(dump, vx, vy, vz, rs, c6);
            for (int k = 0; k < 6; k++) s.dvw[m][k] += c6[k];
            const double v = sqrt((vx * vx + vy * vy) + vz * vz);
            if (v * ph.ndt > ph.group_reach &&
                group_reaches_other<Real>(a, r, (double)cx + bx, (double)cy + by, (double)cz + bz, v, l, s.g, C))
                flags |= REPLAY_ESCAPED;
            s.reach[i] = all;
            n++;
        }
        s.o[0][i] = (Real)bx; s.o[1][i] = (Real)by; s.o[2][i] = (Real)bz;
        s.v[0][i] = (Real)vx; s.v[1][i] = (Real)vy; s.v[2][i] = (Real)vz;
    }
    return n | flags;
}

// Values of the other lanes of a lane's quad (lanes 4i .. 4i+3, all active; axes
// on the first three): lane K's, and those of the next and the previous axis
// (cyclically; lane 3 as lane 2).  Lane permutes of the ALU: a shuffle by way of
// the LDS unit is a wait of some 100 cycles in the chain.
template <int CTRL>
__device__ __forceinline__ double quad_perm(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int K>
__device__ __forceinline__ double quad(double x) { return quad_perm<0x55 * K>(x); }
__device__ __forceinline__ double quad_next(double x) { return quad_perm<1 | 2 << 2>(x); }
__device__ __forceinline__ double quad_prev(double x) { return quad_perm<2 | 1 << 4 | 1 << 6>(x); }

// The stochastic reflection of a particle by a colloid, an axis per lane of a
// quad (k = 0..2; lane 3 only draws): reflect_event's and draw_reflection's
// operations, the draws and the two logarithms side by side on the quad's
// lanes.  o, v: the particle's offset in its cell and velocity along the
// lane's axis, updated; rs: the surface vector; inj: the injected draw (read
// when draws are).  False: it is missing (nothing changed).
template <class Real>
__device__ __forceinline__ bool reflect_quad(const Phys &ph, const Rep &R, const double *inj, long long step, int substep,
                                             int g, int pid, int i_k, double &o, double &v, double pc, double vcol, double wcol,
                                             int l0, int k, double &rs) {
    const double Ld = (double)R.L, dt = ph.dt;
    double u_e, t_k, x1, x2;
    if (ph.draws == BW_DRAWS_INJECTED) {
        if (inj[0] != inj[0]) return false;
        u_e = inj[0];
        t_k = inj[1 + min(k, 2)];
        x1 = 2.0 * inj[4] - 1;
        x2 = 2.0 * inj[5] - 1;
    } else {
        const uint32_t c0 = KIND_REFL | ((uint32_t)substep << 8), jl = (uint32_t)(g - R.first_colloid);
        uint4 a = philox(make_uint4(c0 | ((uint32_t)k << 16), (uint32_t)step, (uint32_t)pid, jl), rep_key(R));
        double ua = u01(a.x, a.y), ub = u01(a.z, a.w);
        u_e = quad<0>(ua);
        const double tx = quad<0>(ub), ty = quad<1>(ua), tz = quad<1>(ub);
        t_k = k == 0 ? tx : k == 1 ? ty : tz;
        // the polar pair: the first accepted try, four tries per round (the
        // first round's lanes 0 and 1 hold the other draws)
        for (uint32_t t = 0;; t += 4) {
            x1 = 2.0 * ua - 1;
            x2 = 2.0 * ub - 1;
            const double z = x1 * x1 + x2 * x2;
            const bool ok = (t > 0 || k >= 2) && z <= 1 && z > 0;
            const unsigned hit = (unsigned)(__ballot(ok) >> l0) & 15u;
            if (hit) {
                const int w = __ffs(hit) - 1;
                x1 = __shfl(x1, l0 + w);
                x2 = __shfl(x2, l0 + w);
                break;
            }
            if (t + 4 >= 65535u) break;
            a = philox(make_uint4(c0 | ((t + 4u + (uint32_t)k) << 16), (uint32_t)step, (uint32_t)pid, jl), rep_key(R));
            ua = u01(a.x, a.y);
            ub = u01(a.z, a.w);
        }
    }
    o = o - v * dt * 0.5;
    const double a_k = (double)i_k + o;
    rs = img1(a_k - pc, Ld);
    // stochastic_reflection: the normal speed's logarithm on lane 0 (and 2,
    // 3), the tangential one's on lane 1
    const double m_beta = ph.mass_fl / ph.kbt;
    const double re = (1 - u_e) * (1 - u_e);
    const double z = x1 * x1 + x2 * x2;
    const double lg = log(k == 1 ? z : re);
    const double sq = sqrt((k == 1 ? -2.0 * lg : -lg) / (k == 1 ? z : m_beta));
    const double val = quad<0>(sq), zt = quad<1>(sq);
    double r0 = quad<0>(rs), r1 = quad<1>(rs), r2 = quad<2>(rs);
    const double nrm = sqrt((r0 * r0 + r1 * r1) + r2 * r2);
    const double un = rs / nrm * val;
    const double tk = img1(t_k * Ld - a_k, Ld);
    double ut = quad_next(un) * quad_prev(tk) - quad_prev(un) * quad_next(tk);
    const double q0 = quad<0>(ut), q1 = quad<1>(ut), q2 = quad<2>(ut);
    ut = ut / sqrt((q0 * q0 + q1 * q1) + q2 * q2);
    const double v1 = x1 * zt * ph.vscale_thermal;
    const double u = ut * v1 + un;
    double nv = u + vcol + (quad_next(wcol) * quad_prev(rs) - quad_prev(wcol) * quad_next(rs));
    if (sizeof(Real) == 4) nv = (double)(float)nv;  // what the velocity store keeps
    v = nv;
    o = o + v * dt * 0.5;
    return true;
}

// The substeps of one group of C colloids (s.g, ascending) by NW waves.
// Latency-bound: a group's substeps are one chain of small dependent phases
// (stream and detect; reflect; sum, force and update), so its colloids and the
// particles that matter stay in LDS, small groups in one wave, whose phases
// need no barrier, and the axes of a reflection or a colloid lie on
// neighbouring lanes.
//
// The particles of the buckets are looked at in windows of substeps: at a
// window's start all of them are brought to the present substep, and those that
// may come to a colloid's surface within the window -- travel plus the
// colloid's displacement bound for the window -- are copied to LDS and streamed
// per substep; the others are streamed when the next window opens.  A colloid
// that leaves its bound opens the next window at once, as does a full LDS list
// (events excepted: these have room of their own).  The window is as long as
// keeps the selected particles at about one per lane (6 per colloid and substep
// at 10 particles per cell and 20 substeps).
//
// False: beyond the LDS lists' capacities.
template <class Real, int NW>
__device__ __forceinline__ bool group_step(const Phys &ph, const Dev &d, const Fluid<Real> &f, HotPart<Real> *h, int final,
                                           int n_col, int r, GroupLds<Real, NW> &s) {
    using G = GroupLds<Real, NW>;
    const int C = G::MAX == 1 ? 1 : n_col;
    constexpr int TH = 64 * NW;
    const int tid = NW == 1 ? threadIdx.x & 63 : threadIdx.x, lane = threadIdx.x & 63;
    auto sync = [&]() {
        if constexpr (NW == 1) wave_sync();
        else __syncthreads();
    };
    const Rep R = ld_const(d.rep + r);
    const int L = R.L;
    const double Ld = (double)L;
    const long long step = ld_const(d.step);
    const unsigned long long below = (1ull << lane) - 1ull;
    // places for the lanes with p in a list counted by cnt[k]
    int *cnt = s.cnt[0];
    auto place = [&](bool p, int k) {
        const unsigned long long b = __ballot(p);
        int base = 0;
        if (b) {
            if (lane == 0) base = atomicAdd(cnt + k, __popcll(b));
            base = __builtin_amdgcn_readfirstlane(base);
        }
        return base + __popcll(b & below);
    };
    bool marg = false, md_far = false, tl_far = false, missing = false, escaped = false, drift = false;
    int par = 0, n_events = 0, n_sel = 0, n_se = 0;
    int opened = 0;            // the window's first substep
    const Real dt = (Real)ph.dt;
    // FP32 positions are taken from the first colloid's cell
    const int o0 = d.ccell[3 * s.g[0]], o1 = d.ccell[3 * s.g[0] + 1], o2 = d.ccell[3 * s.g[0] + 2];
    const double origin[3] = {(double)o0, (double)o1, (double)o2};
    const float Lf = (float)L, iLf = 1.0f / Lf;
    for (int i = tid; i < C * 3; i += TH) {
        const int c = i / 3, k = i - 3 * c, g = s.g[c];
        const double p = d.cpos[3 * g + k];
        const int cc = d.ccell[3 * g + k];
        s.pos[0][c][k] = p;
        (&s.rel[0][c].x)[k] = (float)img1(p - origin[k], Ld);
        s.pos0[c][k] = p;
        s.cell[0][c][k] = cc;
        s.cell0[c][k] = cc;
        s.vel[c][k] = d.cvel[3 * g + k];
        s.om[c][k] = d.comega[3 * g + k];
        s.ra[c][k] = d.cra[3 * g + k];
        s.f[c][k] = d.cf[3 * g + k];
        s.of[c][k] = d.coldf[3 * g + k];
        s.disp[c][k] = d.cdisp[3 * g + k];
        s.imp[c][k] = d.cimp[6 * g + k];
        s.imp[c][3 + k] = d.cimp[6 * g + 3 + k];
        if (k == 0) {
            s.v0[c] = d.cv0[g];
            s.sur[c] = ph.surrogate && d.cmode[g];
        }
    }
    if (tid < 14) s.cnt[0][tid] = 0;
    int n_hot = 0;
    for (int c = 0; c < C; c++) {
        const int n = d.hot_cnt[s.g[c]];
        if (tid == 0) s.hot[c] = n_hot;
        n_hot += n;
    }
    if (tid == 0) s.hot[C] = n_hot;
    h += d.grp_hot[s.g[0]];  // the group's working copies
    int *slots = d.grp_slot + d.grp_hot[s.g[0]];
    sync();
    // A particle's position from the origin lies in [-L/2, L/2 + 1), so its
    // distance to a colloid at b is taken right without the wrap modulo L as
    // long as |b| plus that distance stays below L/2 - 1 along every axis:
    // distances up to `room` (the group's own extent: fast particles link
    // colloids farther apart than link2)
    float extent = 0.0f;
    for (int c = 0; c < C; c++) {
        const float4 b = s.rel[0][c];
        extent = fmaxf(extent, fmaxf(fabsf(b.x), fmaxf(fabsf(b.y), fabsf(b.z))));
    }
    const float room = __int_as_float(__builtin_amdgcn_readfirstlane(  // the same in every lane
        __float_as_int(0.5f * Lf - 1.0f - (extent + (float)ph.margin + 1e-2f))));
    unsigned all = 0;  // the explicitly colliding colloids
    for (int c = 0; c < C; c++)
        if (!s.sur[c]) all |= 1u << c;
    bool open = true;  // the next substep opens a window
    int window_end = 0;
    const float rr = sqrtf((float)ph.lim_coll);
    for (int l = 0; l < ph.n_sub; l++) {
        cnt = s.cnt[l & 1];
        if (l == window_end) open = true;
        // the colloids of mask m that hold a particle of cell (ix,iy,iz)
        // (cpp/fluid_colloid_collision.cpp:32-35); reach: those it comes to
        // within wr of, plus (a window's start) the colloid's bound
        auto detect = [&](unsigned m, int ix, int iy, int iz, Real ox, Real oy, Real oz, float wr, int &n_in, int &m_in,
                          bool &inside, unsigned &reach) {
            n_in = 0;
            m_in = 0;
            inside = false;
            reach = 0;
            const float px = (float)pdiff(ix, o0, L) + (float)ox, py = (float)pdiff(iy, o1, L) + (float)oy,
                        pz = (float)pdiff(iz, o2, L) + (float)oz;
            // 2e-3 covers the FP32 roundings; the exact test follows
            const float rd = rr + 2e-3f, r0 = rd + wr;
            for (; m; m &= m - 1) {
                const int c = __ffs(m) - 1;
                const float4 b = s.rel[par][c];
                float ax = px - b.x, ay = py - b.y, az = pz - b.z;
                const float rs = open ? r0 + b.w : rd;
                if (!(rs <= room)) {
                    ax -= Lf * rintf(ax * iLf); ay -= Lf * rintf(ay * iLf); az -= Lf * rintf(az * iLf);
                }
                const float q2 = (ax * ax + ay * ay) + az * az;
                if (q2 > rs * rs) continue;
                reach |= 1u << c;
                if (q2 > rd * rd) continue;
                const double x = (double)ix + (double)ox, y = (double)iy + (double)oy, z = (double)iz + (double)oz;
                const double rx = img1(s.pos[par][c][0] - x, Ld), ry = img1(s.pos[par][c][1] - y, Ld),
                             rz = img1(s.pos[par][c][2] - z, Ld);
                if ((rx * rx + ry * ry) + rz * rz <= ph.lim_coll) {
                    inside = true;
                    if (in_stencil(ix, iy, iz, s.cell[par][c][0], s.cell[par][c][1], s.cell[par][c][2], L)) {
                        n_in++;
                        m_in = c;
                    }
                }
            }
        };
        // a wave's events (particles at LDS places i, negative: none left)
        auto record = [&](bool on, int i, int ix, int iy, int iz, int n_in, int m_in, int pid) {
            const int e = place(on && n_in == 1, 0);
            if (on && n_in == 1 && e < G::EV) {
                s.ev_i[e] = i;
                s.ev_m[e] = m_in;
                const int dx = pdiff(ix, s.cell[par][m_in][0], L), dy = pdiff(iy, s.cell[par][m_in][1], L),
                          dz = pdiff(iz, s.cell[par][m_in][2], L);
                s.key[e] = ((long long)stencil_index(dx, dy, dz) << 32) | (unsigned)pid;
            }
            if (__ballot(on && n_in > 1)) {
                const int ch = place(on && n_in > 1, 1);
                if (on && n_in > 1 && ch < G::SER) s.chain_i[ch] = i;
            }
        };
        if (open) {
            // ---- a new window: every particle of the buckets to this substep
            const int w = min(max(ph.window * NW / C, NW == 1 ? 1 : ph.window_min), ph.n_sub - l);
            const float wdt = (float)(w * ph.dt);
            for (int c = tid; c < C; c += TH) {
                const double *v = s.vel[c], *a = s.f[c];
                const float vn = sqrtf((float)((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]));
                const float fn = sqrtf((float)((a[0] * a[0] + a[1] * a[1]) + a[2] * a[2]));
                s.rel[par][c].w = vn * wdt + fn / (float)ph.mass_colloid * (wdt * wdt) + (float)ph.tight0 * (wdt / (float)ph.ndt);
                for (int k = 0; k < 3; k++) s.posw[c][k] = s.pos[par][c][k];
            }
            // the last window's particles back to their working copies
            const int n_all = n_sel + n_se;
            for (int j = tid; j < n_all; j += TH) {
                const int i = j < n_sel ? j : G::SEL + j - n_sel;
                h[s.q[i]] = HotPart<Real>{s.o[0][i], s.o[1][i], s.o[2][i], s.pc[i] | CURRENT,
                                          s.v[0][i], s.v[1][i], s.v[2][i], s.pid[i]};
            }
            sync();
            const int late = l - opened - 1;  // substeps the others are behind (l > 0)
            // rounds of TH particles, each round's loads sent before the last
            // round's particles are worked on
            auto fetch = [&](int q) {
                HotPart<Real> v{};
                if (q < n_hot) {
                    if (l == 0) {  // from the buckets
                        int c = 0;
                        while (q >= s.hot[c + 1]) c++;
                        const int slot = d.hot_ent[s.g[c] * d.hot_cap + q - s.hot[c]];
                        slots[q] = slot;
                        v = HotPart<Real>{f.ox[slot], f.oy[slot], f.oz[slot], f.cell[slot] | CURRENT,
                                          f.vx[slot], f.vy[slot], f.vz[slot], f.pid[slot]};
                    } else {
                        v = h[q];
                    }
                }
                return v;
            };
            HotPart<Real> next = fetch(tid);
            {
                for (int q0 = 0; q0 < n_hot; q0 += TH) {
                    const HotPart<Real> now = next;
                    next = fetch(q0 + TH + tid);
                    const int q = q0 + tid, pid = now.pid;
                    const bool on = q < n_hot;
                    int pc = now.cell;
                    Real ox = now.ox, oy = now.oy, oz = now.oz;
                    const Real vx = now.vx, vy = now.vy, vz = now.vz;
                    int ix, iy, iz;
                    unpack_cell(pc, ix, iy, iz);
                    int phantom = pc & PHANTOM;
                    int n_in = 0, m_in = 0;
                    bool inside = false;
                    unsigned reach = 0;
                    if (on) {
                        fly_flat((pc & CURRENT) ? 1 : 1 + late, dt, L, vx, vy, vz, ix, iy, iz, ox, oy, oz);
                        const float wx = (float)vx, wy = (float)vy, wz = (float)vz;
                        const float travel = sqrtf((wx * wx + wy * wy) + wz * wz) * wdt;
                        detect(all, ix, iy, iz, ox, oy, oz, travel, n_in, m_in, inside, reach);
                        if (phantom) {  // no events until it is inside no colloid
                            if (!inside) phantom = 0;
                            n_in = 0;
                        }
                    }
                    const bool sel = reach != 0, ev = n_in > 0;
                    const int is = place(sel && !ev, 3);
                    int i = sel && !ev && is < G::SEL ? is : -1;
                    if (__ballot(ev)) {
                        const int ie = place(ev, 4);
                        if (ev) i = ie < G::EV ? G::SEL + ie : -1;
                    }
                    pc = pack_cell(ix, iy, iz) | phantom;
                    if (i >= 0) {
                        s.q[i] = q;
                        s.pid[i] = pid;
                        s.pc[i] = pc;
                        s.reach[i] = reach;
                        s.o[0][i] = ox; s.o[1][i] = oy; s.o[2][i] = oz;
                        s.v[0][i] = vx; s.v[1][i] = vy; s.v[2][i] = vz;
                        h[q].cell = IN_WINDOW;
                    } else if (on) {
                        h[q] = HotPart<Real>{ox, oy, oz, pc, vx, vy, vz, pid};
                    }
                    if (__ballot(ev)) record(ev, i, ix, iy, iz, n_in, m_in, pid);
                }
            }
            sync();
            const int want = cnt[3], ne = cnt[4];
            if (ne > G::EV) return false;
            n_sel = min(want, G::SEL);
            n_se = ne;
            opened = l;
            open = want > G::SEL;  // some found no room: look again at the next substep
            window_end = l + w;
        } else {
            // ---- streaming and detection of the window's particles
            // (cpp/update.cpp:56-60)
            const int n_all = n_sel + n_se;
            for (int j0 = tid - lane; j0 < n_all; j0 += TH) {
                const int j = j0 + lane;
                const bool on = j < n_all;
                const int i = !on ? 0 : j < n_sel ? j : G::SEL + j - n_sel;
                int n_in = 0, m_in = 0, ix = 0, iy = 0, iz = 0;
                if (on) {
                    const int pc = s.pc[i];
                    int phantom = pc & PHANTOM;
                    unpack_cell(pc, ix, iy, iz);
                    Real ox = s.o[0][i], oy = s.o[1][i], oz = s.o[2][i];
                    fly_flat(1, dt, L, s.v[0][i], s.v[1][i], s.v[2][i], ix, iy, iz, ox, oy, oz);
                    bool inside;
                    unsigned near;
                    detect(s.reach[i], ix, iy, iz, ox, oy, oz, 0.0f, n_in, m_in, inside, near);
                    if (phantom) {
                        if (!inside) phantom = 0;
                        n_in = 0;
                    }
                    s.pc[i] = pack_cell(ix, iy, iz) | phantom;
                    s.o[0][i] = ox; s.o[1][i] = oy; s.o[2][i] = oz;
                }
                if (__ballot(n_in > 0)) record(n_in > 0, i, ix, iy, iz, n_in, m_in, s.pid[i]);
            }
        }
        for (int c = tid; c < C; c += TH) {
            s.nev[c] = 0;
            s.pair[c] = 0;
        }
        sync();
        if (tid < 7) s.cnt[1 - (l & 1)][tid] = 0;  // the next substep's
        const int n_ev = cnt[0], n_chain = cnt[1];
        if (n_ev > G::EV || n_chain > G::SER) return false;
        // ---- pair forces at this substep's positions (cpp/update.cpp:14-28),
        // from the last lane down (the reflections start at the first)
        for (int i = TH - 1 - tid; i < C * (C - 1) / 2; i += TH) {
            int a = 0, b = i;  // the i-th pair a < b
            while (b >= C - 1 - a) { b -= C - 1 - a; a++; }
            b += a + 1;
            double fx, fy, fz;
            if (pair_force(ph, Ld, s.pos[par][a], s.pos[par][b], fx, fy, fz)) {
                s.pf[i][0] = fx; s.pf[i][1] = fy; s.pf[i][2] = fz;
                atomicOr(&s.pair[a], 1u << b);
                atomicOr(&s.pair[b], 1u << a);
            }
        }
        if (ph.draws == BW_DRAWS_INJECTED) {
            for (int e = tid; e < n_ev; e += TH)
                injected_reflection<Real>(group_args<Real>(), r, l, s.g[s.ev_m[e]], s.pid[s.ev_i[e]], s.ev[e]);
            sync();
        }
        // ---- reflections, four lanes per event; the sums are taken below in
        // the reference's order (stencil position, then id)
        for (int e0 = (tid - lane) >> 2; e0 < n_ev; e0 += TH / 4) {
            const int e = e0 + (lane >> 2), l0 = lane & 60, k = lane & 3, kk = min(k, 2);
            if (e < n_ev) {  // whole quads
                const int i = s.ev_i[e], m = s.ev_m[e], pid = s.pid[i];
                const long long key = s.key[e];
                int rank = 0;
                for (int o = 0; o < n_ev; o++) rank += s.ev_m[o] == m && s.key[o] < key ? 1 : 0;
                int ix, iy, iz;
                unpack_cell(s.pc[i], ix, iy, iz);
                double o = s.o[kk][i], v = s.v[kk][i], rs, c_lin = 0, c_ang = 0;
                const double dump = v;
                const bool hit = reflect_quad<Real>(ph, R, s.ev[e], step, l, s.g[m], pid, kk == 0 ? ix : kk == 1 ? iy : iz, o, v,
                                                    s.pos[par][m][kk], s.vel[m][kk], s.om[m][kk], l0, k, rs);
                if (hit) {
                    // cpp/fluid_colloid_collision.cpp:40-42
                    c_lin = dump - v;
                    c_ang = quad_next(rs) * quad_prev(c_lin) - quad_prev(rs) * quad_next(c_lin);
                    const double bx = quad<0>(o), by = quad<1>(o), bz = quad<2>(o);
                    const double vx = quad<0>(v), vy = quad<1>(v), vz = quad<2>(v);
                    const double ax = (double)ix + bx, ay = (double)iy + by, az = (double)iz + bz;
                    // a later colloid that now contains it: the rest of the
                    // colloid loop is replayed serially
                    int ct = -1;
                    for (int j = m + 1; j < C && ct < 0; j++) {
                        if (s.sur[j] || !in_stencil(ix, iy, iz, s.cell[par][j][0], s.cell[par][j][1], s.cell[par][j][2], L))
                            continue;
                        const double rx = img1(s.pos[par][j][0] - ax, Ld), ry = img1(s.pos[par][j][1] - ay, Ld),
                                     rz = img1(s.pos[par][j][2] - az, Ld);
                        if ((rx * rx + ry * ry) + rz * rz <= ph.lim_coll) {
                            if (k == 0) ct = atomicAdd(cnt + 2, 1);
                            ct = __shfl(ct, l0);
                        }
                    }
                    if (ct >= 0 && ct < G::SER) {
                        s.cont_i[ct] = i;
                        s.cont_from[ct] = m + 1;
                        if (k < 3) s.cont_dump[ct][k] = dump;
                    }
                    if (k < 3) {
                        s.o[k][i] = (Real)o;
                        s.v[k][i] = (Real)v;
                    } else {
                        s.reach[i] = all;  // its new velocity may bring it to any of them
                        // groups keep a clearance of group_reach, which
                        // thermal reflections do not use up
                        if (sqrt((vx * vx + vy * vy) + vz * vz) * ph.ndt > ph.group_reach) cnt[6] = 1;
                    }
                } else {
                    missing = true;
                }
                if (k < 3) {
                    s.ev[e][k] = c_lin;
                    s.ev[e][3 + k] = c_ang;
                } else {
                    s.ord[m][rank] = (unsigned char)e;
                    atomicAdd(&s.nev[m], 1);
                }
            }
        }
        n_events += n_ev;
        sync();
        const int n_cont = cnt[2];
        if (n_cont > G::SER) return false;
        // more events of a colloid than the per-substep kernels' bucket holds:
        // those are replayed serially there, by id (fluid inside a colloid)
        if (G::EV > EV_CAP && n_ev > EV_CAP)
            for (int c = 0; c < C; c++)
                if (s.nev[c] > EV_CAP) return false;
        if (cnt[6])
            for (int e = tid; e < n_ev; e += TH)
                if (fast_event<Real, NW>(group_args<Real>(), r, l, C, s.ev_i[e], &s)) escaped = true;
        // ---- per colloid and axis (four lanes per colloid): the events'
        // momentum and torque sums
        for (int i = tid; i < 4 * C; i += TH) {
            const int c = i >> 2, k = i & 3;
            if (k == 3) continue;
            double a = 0, t = 0;
            const int n = s.nev[c];
            for (int e = 0; e < n; e++) {
                const int o = s.ord[c][e];
                a = a + s.ev[o][k];
                t = t + s.ev[o][3 + k];
            }
            s.dvw[c][k] = a;
            s.dvw[c][3 + k] = t;
        }
        if (n_chain | n_cont) {
            sync();
            if (tid == 0) {
                const int n = replay<Real, NW>(group_args<Real>(), r, l, par, C, n_chain, n_cont, all, &s);
                if (n & REPLAY_MISSING) missing = true;
                if (n & REPLAY_ESCAPED) escaped = true;
                n_events += n & (REPLAY_ESCAPED - 1);  // this lane's count is the group's
            }
            sync();
        }
        if (all != (2u << (C - 1)) - 1u) {
            sync();
            for (int c = tid; c < C; c += TH)
                if (s.sur[c]) surrogate_impulse<Real, NW>(group_args<Real>(), c, &s);
            sync();
        }
        // ---- impulse, activity, force, velocity, [kick], position:
        // colloid_update's operations, an axis per lane
        const bool last = l == ph.n_sub - 1, move = !last || !final;
        for (int i0 = tid - lane; i0 < 4 * C; i0 += TH) {  // whole waves
            const int i = i0 + lane;
            const bool on = (i >> 2) < C && (i & 3) < 3;
            const int c = min(i >> 2, C - 1), k = min(i & 3, 2), l0 = lane & 60;
            const double iv = s.dvw[c][k], iw = s.dvw[c][3 + k];
            // (a surrogate-driven colloid has no events: adds +0)
            const double imp0 = s.imp[c][k] + (s.sur[c] ? 0.0 : iv), imp1 = s.imp[c][3 + k] + (s.sur[c] ? 0.0 : iw);
            double v = s.vel[c][k], w = s.om[c][k];
            v = v + iv * ph.mass_fl / ph.mass_colloid;
            w = w + iw * ph.mass_fl / ph.I_colloid;
            // cpp/update.cpp:34-46
            const double bk = w * ph.dt;
            const double sn = sin(bk), cs = cos(bk);
            const double sbx = quad<0>(sn), sby = quad<1>(sn), sbz = quad<2>(sn);
            const double cbx = quad<0>(cs), cby = quad<1>(cs), cbz = quad<2>(cs);
            double mx, my, mz;
            if (k == 0) { mx = cby * cbz; my = -cby * sbz; mz = sby; }
            else if (k == 1) { mx = sbx * sby * cbz + cbx * sbz; my = -sbx * sby * sbz + cbx * cbz; mz = -sbx * cby; }
            else { mx = -cbx * sby * cbz + sbx * sbz; my = cbx * sby * sbz + sbx * cbz; mz = cbx * cby; }
            const double ra = (mx * s.ra[c][0] + my * s.ra[c][1]) + mz * s.ra[c][2];
            // cpp/update.cpp:28: the partners in ascending order
            double fk = 0;
            for (unsigned m = s.pair[c]; m; m &= m - 1) {
                const int j = __ffs(m) - 1, a = min(c, j), b = max(c, j);
                const double t = s.pf[a * (2 * C - a - 1) / 2 + b - a - 1][k];
                fk = j < c ? fk - t : fk + t;
            }
            double of = s.of[c][k];
            v = v + (of + fk) * (ph.dt / (ph.mass_colloid * 2));
            double p = s.pos[par][c][k];
            int cc = s.cell[par][c][k];
            double disp = s.disp[c][k];
            if (last && !final) {
                v = v + ra * s.v0[c];
                if (on) {
                    const int g = s.g[c];
                    d.cpos_run[3 * g + k] = p;
                    d.ccell_run[3 * g + k] = cc;
                }
            }
            if (move) {
                of = fk;
                const double dt2 = ph.dt * ph.dt, ddt = 0.5 * dt2 / ph.mass_colloid;
                const double dx = v * ph.dt + fk * ddt;
                p = p + dx;
                disp = disp + dx;
                p = mod1(p, Ld);
                cc = coord_cell(p, L);
                const int dm = pdiff(cc, s.cell0[c][k], L);
                if (on && (dm > 1 || dm < -1)) tl_far = true;
                const double md = img1(p - s.pos0[c][k], Ld);
                const double m0 = quad<0>(md), m1 = quad<1>(md), m2 = quad<2>(md);
                const double d2 = (m0 * m0 + m1 * m1) + m2 * m2;
                const double wd = img1(p - s.posw[c][k], Ld);
                const double w0 = quad<0>(wd), w1 = quad<1>(wd), w2 = quad<2>(wd);
                const double e2 = (w0 * w0 + w1 * w1) + w2 * w2;
                if (on && d2 > 0.25 * MD_SKIN * MD_SKIN) md_far = true;
                if (on && !last && d2 > ph.margin * ph.margin) marg = true;
                const double mw = (double)s.rel[par][c].w;
                if (on && !(e2 <= mw * mw)) cnt[5] = 1;
            }
            if (on) {
                s.imp[c][k] = imp0;
                s.imp[c][3 + k] = imp1;
                s.vel[c][k] = v;
                s.om[c][k] = w;
                s.f[c][k] = fk;
                s.of[c][k] = of;
                s.disp[c][k] = disp;
                s.pos[par ^ 1][c][k] = p;
                s.cell[par ^ 1][c][k] = cc;
                (&s.rel[par ^ 1][c].x)[k] = (float)img1(p - (k == 0 ? origin[0] : k == 1 ? origin[1] : origin[2]), Ld);
                if (k == 0) s.rel[par ^ 1][c].w = s.rel[par][c].w;
            }
            wave_sync();  // every lane of the colloid has read the old orientation
            if (on) s.ra[c][k] = ra;
        }
        par ^= 1;
        sync();
        if (cnt[5]) open = true;
    }
    // ---- the group's results
    for (int i = tid; i < C * 3; i += TH) {
        const int c = i / 3, k = i - 3 * c, g = s.g[c];
        d.cpos_nxt[3 * g + k] = s.pos[par][c][k];
        d.ccell_nxt[3 * g + k] = s.cell[par][c][k];
        d.cvel[3 * g + k] = s.vel[c][k];
        d.comega[3 * g + k] = s.om[c][k];
        d.cra[3 * g + k] = s.ra[c][k];
        d.cf[3 * g + k] = s.f[c][k];
        d.coldf[3 * g + k] = s.of[c][k];
        d.cdisp[3 * g + k] = s.disp[c][k];
        d.cimp[6 * g + k] = s.imp[c][k];
        d.cimp[6 * g + 3 + k] = s.imp[c][3 + k];
        if (k == 0 && !final) {
            d.ccnt[g] = 0;
            d.sshell[g] = 0;
            for (int j = 0; j < SUR_ACC; j++) d.sacc[(size_t)SUR_ACC * g + j] = 0;
        }
    }
    const int late = ph.n_sub - opened - 1;
    for (int q = tid; q < n_hot; q += TH) {
        const int slot = slots[q];
        const HotPart<Real> now = h[q];
        const int pc = now.cell;
        if (pc == IN_WINDOW) continue;
        int ix, iy, iz;
        unpack_cell(pc, ix, iy, iz);
        Real ox = now.ox, oy = now.oy, oz = now.oz;
        const Real vx = now.vx, vy = now.vy, vz = now.vz;
        fly_flat(late, dt, L, vx, vy, vz, ix, iy, iz, ox, oy, oz);
        f.cell[slot] = pack_cell(ix, iy, iz) | (pc & PHANTOM);
        f.ox[slot] = ox; f.oy[slot] = oy; f.oz[slot] = oz;
        f.vx[slot] = vx; f.vy[slot] = vy; f.vz[slot] = vz;
        if (outside_tile_reach(R, ph.cap, slot, ix, iy, iz)) drift = true;
    }
    const int n_all = n_sel + n_se;
    for (int j = tid; j < n_all; j += TH) {
        const int i = j < n_sel ? j : G::SEL + j - n_sel, slot = slots[s.q[i]], pc = s.pc[i];
        f.cell[slot] = pc;
        f.ox[slot] = s.o[0][i]; f.oy[slot] = s.o[1][i]; f.oz[slot] = s.o[2][i];
        f.vx[slot] = s.v[0][i]; f.vy[slot] = s.v[1][i]; f.vz[slot] = s.v[2][i];
        int ix, iy, iz;
        unpack_cell(pc, ix, iy, iz);
        if (outside_tile_reach(R, ph.cap, slot, ix, iy, iz)) drift = true;
    }
    if (escaped) stop_step(d);  // (that group is on its way, or done)
    unsigned st = 0;
    if (drift) st |= BW_FLAG_DRIFT;
    if (marg) st |= BW_FLAG_MARGIN;
    if (missing) st |= BW_FLAG_DRAW_MISSING;
    if (st) atomicOr(d.status, st);
    if (md_far) atomicOr(&d.md_stale[r], 1);
    if (tl_far) atomicOr(&d.tcl_stale[r], 1);
    if (tid == 0 && ph.draws == BW_DRAWS_INJECTED) atomicAdd(&d.ev_total[r], n_events);
    return true;
}

// The groups' lists, by one workgroup: every colloid's root, the sizes, then
// per group its members (in any order) and its place among the large groups or
// the small ones.  A group of more than GROUP_MAX colloids or with a full bucket
// ends the step here.
__global__ __launch_bounds__(1024) void k_group_lists(Phys ph, Dev d) {
    // roots, sizes, numbers of particles, places: in LDS while they fit
    __shared__ int s_arr[4][GROUP_LDS_COLLOIDS];
    __shared__ int s_mem, s_hot, s_big, s_small, s_over;
    const int nc = ph.n_colloid_total;
    const bool lds = nc <= GROUP_LDS_COLLOIDS;
    int *root = lds ? s_arr[0] : d.grp_root, *size = lds ? s_arr[1] : d.grp_root + nc,
        *off = lds ? s_arr[2] : d.grp_root + 2 * (size_t)nc, *hot = lds ? s_arr[3] : d.grp_root + 3 * (size_t)nc;
    if (threadIdx.x == 0) { s_mem = 0; s_hot = 0; s_big = 0; s_small = 0; s_over = 0; }
    for (int g = threadIdx.x; g < nc; g += 1024) {
        size[g] = 0;
        hot[g] = 0;
    }
    // global arrays: the stores and the atomics of one phase before the loads
    // of the next
    auto sync = [&]() {
        if (!lds) __threadfence();
        __syncthreads();
    };
    sync();
    for (int g = threadIdx.x; g < nc; g += 1024) {
        const int n = d.hot_cnt[g];
        const int p = d.uf_linked[g] ? group_find(d, g) : g;
        root[g] = p;
        atomicAdd(&size[p], 1);
        atomicAdd(&hot[p], n);
        if (n > d.hot_cap) s_over = 1;
    }
    sync();
    for (int g = threadIdx.x; g < nc; g += 1024) {
        if (root[g] != g) continue;
        const int C = size[g];
        if (C > GROUP_MAX) s_over = 1;
        const int o = atomicAdd(&s_mem, C);
        d.grp_hot[g] = atomicAdd(&s_hot, hot[g]);
        if (C > GROUP_SMALL || nc <= GROUP_WIDE) d.grp_big[atomicAdd(&s_big, 1)] = make_int2(o, C);
        else d.grp_small[atomicAdd(&s_small, 1)] = make_int2(o, C);
        off[g] = o;
    }
    sync();
    if (stopped(ph, d)) return;
    if (s_over) {
        if (threadIdx.x == 0) stop_step(d);
        return;
    }
    for (int g = threadIdx.x; g < nc; g += 1024) d.grp_mem[atomicAdd(&off[root[g]], 1)] = g;
    if (threadIdx.x == 0) {
        d.grp_cnt[0] = s_big;
        d.grp_cnt[1] = s_small;
    }
}

// One workgroup per large group, then one wave per small one; WIDE: a workgroup
// for every group (up to GROUP_WIDE colloids).  Two workgroups per CU are all
// that a WIDE launch has (212 VGPRs, none spilled; 252 and some in FP64); the
// other takes three in FP32 (168, some spilled), which 2400 groups need to run
// at once.  final: the last substep ends with update_velocity_colloid (no kick,
// no position update).
template <class Real, bool WIDE>
__global__ __launch_bounds__(256, WIDE || sizeof(Real) == 8 ? 2 : 3) void k_groups(GroupArgs<Real> a) {
    const Phys &ph = a.ph;
    const Dev &d = a.d;
    const Fluid<Real> &f = a.f;
    HotPart<Real> *h = a.h;
    const int final = a.final;
    __shared__ union {
        GroupLds<Real, 4> big;
        GroupLds<Real, 1> small[WIDE ? 1 : 4];
    } s;
    const int n_big = ld_const(d.grp_cnt), n_small = WIDE ? 0 : ld_const(d.grp_cnt + 1);
    if (stopped(ph, d)) return;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    // members in ascending order into g[0..C)
    auto members = [&](int2 grp, int *g) {
        const int v = lane < grp.y ? d.grp_mem[grp.x + lane] : 0x7fffffff;
        int rank = 0;
        for (int j = 0; j < grp.y; j++) rank += lane_value(v, j) < v ? 1 : 0;
        if (lane < grp.y) g[rank] = v;
    };
    if ((int)blockIdx.x < n_big) {
        const int2 grp = ld_const(d.grp_big + blockIdx.x);
        if (w == 0) members(grp, s.big.g);
        __syncthreads();
        const int r = __builtin_amdgcn_readfirstlane(d.crep[s.big.g[0]]);
        if (!group_step<Real, 4>(ph, d, f, h, final, grp.y, r, s.big)) stop_step(d);
    } else if constexpr (!WIDE) {
        const int i = ((int)blockIdx.x - n_big) * 4 + w;
        if (i >= n_small) return;
        const int2 grp = ld_const(d.grp_small + i);
        members(grp, s.small[w].g);
        wave_sync();
        const int r = __builtin_amdgcn_readfirstlane(d.crep[s.small[w].g[0]]);
        if (!group_step<Real, 1>(ph, d, f, h, final, grp.y, r, s.small[w])) stop_step(d);
    }
}

// With injected draws, after k_groups: every event found its tuple; equal
// totals over the step then mean equal sets
__global__ __launch_bounds__(256) void k_check_draws(Phys ph, Dev d) {
    __shared__ int s_tot;
    if (stopped(ph, d)) return;
    const Rep R = d.rep[blockIdx.x];
    if (threadIdx.x == 0) s_tot = 0;
    __syncthreads();
    int mine = 0;
    for (int i = threadIdx.x; i < ph.n_sub * R.nc; i += 256) {
        const int b = (i / R.nc) * ph.n_colloid_total + R.first_colloid + i % R.nc;
        mine += d.inj_off[b + 1] - d.inj_off[b];
    }
    atomicAdd(&s_tot, mine);
    __syncthreads();
    if (threadIdx.x == 0) {
        if (s_tot != d.ev_total[blockIdx.x]) atomicOr(d.status, BW_FLAG_DRAW_MISMATCH);
        d.ev_total[blockIdx.x] = 0;
    }
}

// The pair list at the colloids' present positions (cpp/neighbour_list.cpp:27-39),
// a wave per colloid: what the per-substep path leaves after its last substep
__global__ __launch_bounds__(256) void k_pair_lists(Phys ph, Dev d, const int2 *wgt) {
    if (stopped(ph, d)) return;
    const int lane = threadIdx.x & 63;
    const int2 wt = wgt[blockIdx.x];
    const int r = wt.x, g = wt.y + (threadIdx.x >> 6);
    const Rep R = d.rep[r];
    if (g >= R.first_colloid + R.nc) return;
    const bool full = d.md_stale[r] != 0;
    const int n = full ? R.nc : d.mdc_cnt[g];
    int w = 0;
    for (int base = 0; base < n; base += 64) {
        const int m = base + lane;
        int j = -1;
        bool p = false;
        if (m < n) {
            j = full ? R.first_colloid + m : d.mdc_list[g * MDC_CAP + m];
            p = j != g && md_pair(ph, d, (double)R.L, g, j);
        }
        const unsigned long long b = __ballot(p);
        const int rank = __popcll(b & ((1ull << lane) - 1ull));
        if (p && w + rank < MD_CAP) d.md_list[g * MD_CAP + w + rank] = j;
        w += __popcll(b);
    }
    if (lane == 0) {
        if (w > MD_CAP) { atomicOr(d.status, BW_FLAG_LIST_OVERFLOW); w = MD_CAP; }
        d.md_cnt[g] = w;
    }
}

template <class Real>
void launch_groups(const Phys &ph, const Dev &d, const Fluid<Real> &f, HotPart<Real> *h, bool final, hipStream_t st) {
    hipLaunchKernelGGL(k_group_lists, dim3(1), dim3(1024), 0, st, ph, d);
    // at most n/2 large groups, or n/4 workgroups of small ones (WIDE: n groups)
    const GroupArgs<Real> a{ph, d, f, h, (int)final};
    if (ph.n_colloid_total <= GROUP_WIDE) hipLaunchKernelGGL((k_groups<Real, true>), dim3(ph.n_colloid_total), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_groups<Real, false>), dim3(ph.n_colloid_total / 2 + 1), dim3(256), 0, st, a);
    if (ph.draws == BW_DRAWS_INJECTED) hipLaunchKernelGGL(k_check_draws, dim3(ph.n_rep), dim3(256), 0, st, ph, d);
}
template void launch_groups<float>(const Phys &, const Dev &, const Fluid<float> &, HotPart<float> *, bool, hipStream_t);
template void launch_groups<double>(const Phys &, const Dev &, const Fluid<double> &, HotPart<double> *, bool,
                                    hipStream_t);
void launch_pair_lists(const Phys &ph, const Dev &d, const int2 *wgt, int nwg, hipStream_t st) {
    hipLaunchKernelGGL(k_pair_lists, dim3(nwg), dim3(256), 0, st, ph, d, wgt);
}

}  // namespace bw
