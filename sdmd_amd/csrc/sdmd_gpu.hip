// sdmd_gpu.hip - MI355X (gfx950) event engine for the sDMD hot path.
//
// Plain FP64 path: bit-exact with the reference event loop.  One workgroup
// owns one system and runs SingleThreadRun (SGThread.c:67-156) on the
// device:
//   event        wave 0 takes the CBT root (AssignJob, SGThread.c:237-259)
//                and executes it (DoEvent, Events.c:25-114)
//   sweep        x += v*dt, t -= dt of every atom (UpdateData/TimeForward,
//                ToolFunctions.c:23-36): the event's atoms at once, the
//                others when they are read, or every few pops (same steps,
//                same bits)
//   predict      the renewed atoms (Predict, SGThread.c:158-211), two side
//                by side: the 27 neighbour cells' atoms in the reference's
//                order into LDS, every lane evaluates a candidate (shell
//                lookup + contact-time quadratic), and one wave runs an
//                ordered min-with-first-index selection that reproduces
//                JobAssign's strict '<' and CheckDuplication's inheritance
//                (TimePrediction.c:1101-1158)
//   tree         wave 0 updates the complete binary tree (CBT.c:56-83)
// A pop is a chain of dependent loads, LDS exchanges and FP64 sequences on
// one CU; what bounds it is the length of that chain.
// Arithmetic follows the reference's operation order; the file is compiled
// with -ffp-contract=off, so every product and sum rounds separately as on
// the x86-64 reference build, and double sqrt/div are correctly rounded.


#include <cstddef>
#include <mutex>

#include "sdmd_dev.h"
#include "sdmd_remd.h"

namespace sdmd {

// ---------------------------------------------------------------- shared state
constexpr int PWIN = 768;          // candidates of one pass (a predicted atom has 60 to 400)
constexpr int LOGK = 32;           // pops between two sweeps at most
constexpr int PCON = 16;           // constraint partners staged per predicted atom
constexpr int PCONSTEP = 8;        // steps per staged constraint
constexpr int NGATHER = 46;        // words of Atom loaded through Sys.gbase

// The atom being predicted, staged once per Predict.  The first NGATHER
// words are loaded by one wavefront, one word per lane, through the gather
// table of Sys (filled by atom_gather_table in the same order).
struct Atom {
    double x, y, z, vx, vy, vz;
    long long counter;
    double t, pot;                 // current event record (JobAssign target)
    long long pc;
    int cx, cy, cz, type, hbbond, hbnb, protein, aanum, nbstat, nbnum;
    int nbp[SDMD_NBSLOTS];
    int partner, evtype, sub, hbitype;
    int ro, ro1, bo, bo1, co, co1; // cmap_off, bond_off, con_off at i and i + 1
    int leaf;
    // not gathered
    int i, role, nb, spanok, rowlo, over, ncand, cnt_eval, hbscan;
    int exclude, below;            // CheckDuplication against atoms < below other than exclude (-1: against none)
    double wt;                     // its wall time (+inf: none offered)
    double zn;                     // its thermostat draw
    double pot0;                   // the record before the prediction (a repeated selection restarts from it)
    long long pc0;
    int sub0, nbnum0;
};
static_assert(offsetof(Atom, leaf) == 4 * (NGATHER - 1), "gathered words come first");

// one atom's candidates in program order, and its bonds, constraints and
// connection row
struct Cand {
    int j[PWIN];
    unsigned char cell[PWIN], fl[PWIN], hfl[PWIN];
    signed char sub[PWIN];
    double t[PWIN], pot[PWIN], ht[PWIN], hpot[PWIN];
    int cellcnt[27], celloff[28];
    double shift[27][3];           // periodic image of neighbour cell c (PBCShift)
    double pcc[3];                 // cell-crossing time along each axis
    int bj[MAXBOND];
    double bt[MAXBOND], bjt[MAXBOND];
    signed char bsub[MAXBOND];
    unsigned char bfl[MAXBOND];
    double con_dmin[PCON], con_dmax[PCON];
    int con_step0[PCON], con_nstep[PCON];
    double con_d[PCON][PCONSTEP], con_e[PCON][PCONSTEP];
    // connection row by offset from its first column: bits 0-1 BOND and
    // CONSTRAINT, bits 2-6 the constraint's slot + 1 (0: not staged)
    unsigned char conn[128];
};

struct Smem {
    Atom A[2];
    Cand c[2];
    // loop scalars
    int target, partner, stale, renew[4], err, root, flush;
    double dt;
    long long zpos;
    // pops whose time step the atoms have not taken yet (see sweep)
    int nlog;
    double log[LOGK];
};

// The collision table (RightPair resolved per type pair) and the step pool
// of the tables, in LDS: a candidate's shell is found without leaving the CU
struct PairTab {
    double dmin[NT * NT], dmax[NT * NT];
    int step0[NT * NT], nstep[NT * NT];
    double d[LPOOL], e[LPOOL];
};

// ---------------------------------------------------------------- lazy sweep
// UpdateData + TimeForward (ToolFunctions.c:23-36) advance every atom by
// every pop's dt: x += v dt, t -= dt, each step rounded.  The result of an
// atom depends only on its own steps, so they are taken when the atom is
// next read, or by a sweep of all atoms every few pops: sm.log holds the dt
// of the last sm.nlog pops and S.lag[i] how many of them atom i has taken.
// The same operations in the same order give the same bits; the sweep's
// memory traffic is paid once per LOGK pops (a sweep per pop cost 33 us of a
// 73 us pop at 26 080 atoms).
template <class SYS>
__device__ __forceinline__ int lag_of(SYS &S, int n, int j) { return n ? (int)G(S.lag)[j] : 0; }

__device__ __forceinline__ void steps_pos(const double *log, int l, int n, double &x, double &y, double &z, double vx,
                                          double vy, double vz) {
    for (; l < n; l++) {
        const double dt = log[l];
        x = x + vx * dt;
        y = y + vy * dt;
        z = z + vz * dt;
    }
}
template <class SYS>
__device__ __forceinline__ double evt_now(SYS &S, const Smem &sm, int j) {
    double t = G(S.evt)[j];
    const int n = sm.nlog;
    for (int l = lag_of(S, n, j); l < n; l++) t = t - sm.log[l];
    return t;
}
template <class SYS>
__device__ __forceinline__ void pos_now(SYS &S, const Smem &sm, int j, double *p) {
    const int n = sm.nlog, l = lag_of(S, n, j);
    double x = G(S.x)[j], y = G(S.y)[j], z = G(S.z)[j];
    if (l < n) steps_pos(sm.log, l, n, x, y, z, G(S.vx)[j], G(S.vy)[j], G(S.vz)[j]);
    p[0] = x; p[1] = y; p[2] = z;
}

struct PosLazy {      // the stored positions with the steps an atom has not taken yet
    const Sys &S;
    const Smem &sm;
    __device__ void pos(int j, double *p) const { pos_now(S, sm, j, p); }
    __device__ int first(int cell) const { return G(S.celllist)[S.N + cell]; }
    __device__ int next(int, int j) const { return G(S.celllist)[j]; }
};

// pair kinematics of the staged atom and j's current state
__device__ __forceinline__ void calc_params_now(SV &S, const Smem &sm, const Atom &A, int j, Kin &k) {
    double p[3];
    pos_now(S, sm, j, p);
    calc_params_at(S, A.x, A.y, A.z, A.vx, A.vy, A.vz, A.cx, A.cy, A.cz, j, p[0], p[1], p[2], G(S.vx)[j], G(S.vy)[j],
                   G(S.vz)[j], k);
}

// UpdateData + TimeForward over all atoms: each takes the steps it still lacks
template <int B>
__device__ __forceinline__ void sweep(SV &S, Smem &sm) {
    const int n = sm.nlog, N = S.N;
    for (int i = threadIdx.x + 1; i <= N; i += B) {
        int l = G(S.lag)[i];
        const double vx = G(S.vx)[i], vy = G(S.vy)[i], vz = G(S.vz)[i];
        double x = G(S.x)[i], y = G(S.y)[i], z = G(S.z)[i], t = G(S.evt)[i];
        for (; l < n; l++) {
            const double dt = sm.log[l];
            x = x + vx * dt;
            y = y + vy * dt;
            z = z + vz * dt;
            t = t - dt;
        }
        G(S.x)[i] = x; G(S.y)[i] = y; G(S.z)[i] = z; G(S.evt)[i] = t;
        G(S.lag)[i] = 0;
    }
    __syncthreads();
    if (threadIdx.x == 0) sm.nlog = 0;
    __syncthreads();
}

__device__ __forceinline__ int in_nb_list(const Atom &A, int j, int *err) {   // FindElemInList(neighborPartner, j, -1, -1, 0)
    for (int k = 1; k < SDMD_NBSLOTS; k++) {
        if (A.nbp[k] == 0) return 0;
        if (A.nbp[k] == j) return k;
    }
    if (A.nbnum == 0) return 0;
    if (A.nbnum == j) return 5;
    if (A.nbstat == 0) return 0;
    if (A.nbstat == j) return 6;
    *err = ERR_NBLIST;
    return 0;
}

// ---------------------------------------------------------------- wave helpers
// Ordered selection over n entries in program order, run by one full wave.
// Entry k offers its computed time ct[k] (+inf when it would not reach
// JobAssign or fails `t > 0`); flagged entries (bit 0) first offer j's
// current event (CheckDuplication; jt(k) its time) when strictly earlier
// than the running minimum.  Returns the winning entry and whether it was
// inherited.
template <class JT>
__device__ __forceinline__ void wave_select(int n, const double *ct, const unsigned char *fl, const JT &jt, double &m,
                                            int &win, int &inh) {
    const int lane = threadIdx.x & 63;
    for (int base = 0; base < n; base += 64) {
        const int k = base + lane;
        const bool in = k < n;
        const double tk = in ? ct[k] : __builtin_inf();
        unsigned long long mask = __ballot(in && (fl[in ? k : 0] & 1));
        const int end = min(base + 64, n);
        int start = base;
        while (true) {
            const int d = mask ? base + __ffsll((long long)mask) - 1 : end;
            const double t = (k >= start && k < d) ? tk : __builtin_inf();
            const int src = wave_first_min(t);
            const double tm = lane_get(t, src);
            if (tm < m) { m = tm; win = base + src; inh = 0; }
            if (d >= end) break;
            const double tj = jt(d), td = lane_get(tk, d - base);
            if (m > tj) { m = tj; win = d; inh = 1; }
            else if (td < m) { m = td; win = d; inh = 0; }
            start = d + 1;
            mask &= mask - 1;
        }
    }
}

// JobAssign / CheckDuplication result applied to the staged record (lane 0)
__device__ __forceinline__ void take_computed(Atom &A, SV &S, double t, double pot, int sub, int type, int j) {
    A.pot = pot; A.sub = sub; A.t = t; A.evtype = type;
    if (j) { A.partner = j; A.pc = G(S.evc)[j]; }
    else A.partner = INVALID;
}

__device__ __forceinline__ void take_inherited(Atom &A, SV &S, const Smem &sm, int j, int type) {
    A.partner = j; A.pot = G(S.evpot)[j]; A.sub = G(S.evsub)[j]; A.t = evt_now(S, sm, j); A.evtype = type;
    A.pc = G(S.evc)[j];
}

// CheckDuplication's condition; A.exclude is an atom whose record is being
// written by another wavefront (it held none when A's prediction began)
__device__ __forceinline__ bool dup_open(const Atom &A, int j) { return A.exclude >= 0 && j != A.exclude && j < A.below; }
__device__ __forceinline__ bool dupable(SV &S, const Atom &A, int j, int type) {
    return dup_open(A, j) && G(S.evp)[j] == A.i && G(S.evtype)[j] == type && G(S.evpc)[j] == A.counter;
}

// ---------------------------------------------------------------- candidate evaluation
// one BondTime entry, TimePrediction.c:219-293
__device__ __forceinline__ void eval_bond(SV &S, const Smem &sm, const Atom &A, Cand &C, int q) {
    const int e = A.bo + q;
    const int j = G(S.bond_j)[e];
    const double lo = G(S.bond_dmin)[e], hi = G(S.bond_dmax)[e];
    C.bj[q] = j;
    const bool dup = dupable(S, A, j, SDMD_BOND);
    C.bfl[q] = dup ? 1 : 0;
    C.bjt[q] = dup ? evt_now(S, sm, j) : 0;
    Kin k;
    calc_params_now(S, sm, A, j, k);
    double t;
    int sub;
    if (k.rr - hi > ZERO && k.b >= 0) {
        sub = SDMD_WELLBOUNC;
        t = 1e-16 * A.i * j;
    } else if (!(k.rr - hi > ZERO) && lo - k.rr > ZERO && k.b < 0) {
        sub = SDMD_CORECOLLI;
        t = 1e-16 * A.i * j;
    } else {
        int s;
        double d2;
        if (k.b < 0 && calc_disc(k, lo) > 0) { s = -1; d2 = lo; sub = SDMD_CORECOLLI; }
        else { s = 1; d2 = hi; sub = SDMD_WELLBOUNC; }
        t = calc_time(k, s, d2);
        if (t < 0) t = INFINIT;
    }
    C.bt[q] = (t > 0) ? t : __builtin_inf();
    C.bsub[q] = (signed char)sub;
}

// FindPair's shell search (shell_lookup) for a collision or constraint pair
// on radii d(k) and energies e(k): strictly increasing, non-zero, nstep <= 16
template <class D, class E>
__device__ __forceinline__ int shell_fast(double dmin, double dmax, int nstep, const D &d, const E &e, double direction,
                                          double d2, double &flo, double &fhi, double &lopot, double &hipot, int *err) {
    const double dir = (direction < 0) ? 1 : -1;
    const double tol = dir * ZERO;
    flo = fhi = INFINIT;
    lopot = hipot = 0;
    if (dmin == 0) { *err = ERR_TABLE; return -1; }
    if (d2 < dmin - ZERO) return -1;
    int ks = 0;
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 4) {
        if (k0 < nstep) {
            double r[4];
#pragma unroll
            for (int u = 0; u < 4; u++) r[u] = d(k0 + u < nstep ? k0 + u : nstep - 1);
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (k0 + u < nstep) ks += (d2 >= r[u] + tol) ? 1 : 0;
        }
    }
    flo = dmin;
    if (ks > 0) {
        flo = d(ks - 1);
        lopot = e(ks - 1);
    }
    if (ks < nstep) {
        fhi = d(ks);
        hipot = -1 * e(ks);
        return ks == 0 ? 0 : -1;
    }
    if (dmax > 0) {
        if (d2 < dmax + ZERO) {
            fhi = dmax; hipot = 0;
            return (nstep == 0 && dir == 1) ? 0 : 1;
        }
        flo = INFINIT; fhi = INFINIT; lopot = 0; hipot = 0;
        return -1;
    }
    fhi = INFINIT; hipot = INFINIT;
    return 1;
}

// candidate k of the staged atom: CollisionTime (TimePrediction.c:79-179)
// and, for a free H-bond atom, HBTime's scan (TimePrediction.c:414-478).
// Every field of j that either may need is loaded at once (one round trip);
// shells come from LDS.
template <bool TAB>
__device__ __forceinline__ void eval_candidate(SV &S, const Smem &sm, const PairTab *T, const Atom &A, Cand &C,
                                               int kidx, double calib, int *err) {
    const int j = C.j[kidx], i = A.i;
    double tout = __builtin_inf(), pot = 0, ht = __builtin_inf(), hpot = 0;
    int sub = SDMD_INVALID_INTER;
    unsigned char fl = 0, hfl = 0;
    if (j != i) {
        const int n = sm.nlog;
        const int l = lag_of(S, n, j);
        const int evp = G(S.evp)[j], evtype = G(S.evtype)[j], tj = G(S.type)[j];
        const long long evpc = G(S.evpc)[j];
        double x = G(S.x)[j], y = G(S.y)[j], z = G(S.z)[j];
        const double vx = G(S.vx)[j], vy = G(S.vy)[j], vz = G(S.vz)[j];
        const bool hb = A.role == 'A' || A.role == 'D' || A.role == 'S';
        int rj = 0, hj = 0, aj = 0, pj = 0;
        if (hb) { rj = G(S.role)[j]; hj = G(S.hbbond)[j]; aj = G(S.aanum)[j]; pj = G(S.protein)[j]; }
        steps_pos(sm.log, l, n, x, y, z, vx, vy, vz);
        const bool mine = dup_open(A, j) && evp == i && evpc == A.counter;
        if (mine && evtype == SDMD_COLI) fl = 1;
        // PBCShift + CalculateParameters
        const double *sh = C.shift[C.cell[kidx]];
        Kin k;
        k.r1 = A.x - (x + sh[0]);
        k.r2 = A.y - (y + sh[1]);
        k.r3 = A.z - (z + sh[2]);
        const double v1 = A.vx - vx, v2 = A.vy - vy, v3 = A.vz - vz;
        k.rr = k.r1 * k.r1 + k.r2 * k.r2 + k.r3 * k.r3;
        k.b = k.r1 * v1 + k.r2 * v2 + k.r3 * v3;
        k.v2 = v1 * v1 + v2 * v2 + v3 * v3;
        int cb = 0;
        if (A.spanok) {
            const unsigned off = (unsigned)(j - A.rowlo);
            if (off < 128u) cb = C.conn[off];
        } else {
            cb = cmap_get(S, i, j) & (SDMD_BOND_CONNECT | SDMD_CONSTRAINT_CONNECT);
        }
        if (!((cb & SDMD_BOND_CONNECT) || A.hbbond == j || in_nb_list(A, j, err)) && k.rr <= calib) {
            double lo, hi, lopot, hipot;
            int cs;
            const int con = cb & SDMD_CONSTRAINT_CONNECT, slot = (cb >> 2) - 1;
            bool skip = false;
            if (con && slot >= 0 && S.steps_sorted) {
                const double *d = C.con_d[slot], *e = C.con_e[slot];
                cs = shell_fast(C.con_dmin[slot], C.con_dmax[slot], C.con_nstep[slot], [&](int q) { return d[q]; },
                                [&](int q) { return e[q]; }, k.b, k.rr, lo, hi, lopot, hipot, err);
            } else {
                const int t12 = A.type * NT + tj;
                if (TAB && !con && S.ltab) {
                    const double *d = T->d + T->step0[t12], *e = T->e + T->step0[t12];
                    cs = shell_fast(T->dmin[t12], T->dmax[t12], T->nstep[t12], [&](int q) { return d[q]; },
                                    [&](int q) { return e[q]; }, k.b, k.rr, lo, hi, lopot, hipot, err);
                } else {
                    FP f;
                    cs = find_pair(S, i, j, con ? K_CONSTRAINT : K_COLLISION, k.b, k.rr, f, 0, 0, err);
                    lo = f.lo; hi = f.hi; lopot = f.lopot; hipot = f.hipot;
                }
                if (!con && lopot == 0 && hipot == 0) skip = true;
            }
            if (!skip) {
                int s;
                double d2;
                if (k.b < 0 && calc_disc(k, lo) > 0) {
                    s = -1; d2 = lo; pot = lopot;
                    sub = (cs == 0) ? SDMD_CORECOLLI : SDMD_TBDCAPTR;
                } else {
                    s = 1; d2 = hi; pot = hipot;
                    if (con) sub = (cs == 1) ? SDMD_WELLBOUNC : SDMD_TBDESCAP;
                    else if (cs == 1) skip = true;
                    else sub = SDMD_TBDESCAP;
                }
                if (!skip) {
                    const double t = calc_time(k, s, d2);
                    tout = (t > 0) ? t : __builtin_inf();
                    fl |= 2;   // reached the quadratic
                }
            }
        }
        if (hb) {
            const int ri = A.role;
            const bool pairok = (ri == 'A' && rj == 'D') || (ri == 'D' && rj == 'A') || (ri == 'S' && tj == 2) ||
                                (rj == 'S' && A.type == 2) || (ri == 'S' && rj == 'S');
            int sep = A.aanum - aj;
            if (sep < 0) sep = -sep;
            if (pairok && hj == 0 && ((A.protein == pj && sep >= 4) || A.protein != pj)) {
                hfl = 4 | ((mine && evtype == SDMD_HB) ? 1 : 0);    // bit 2: an H-bond candidate
                if (A.hbscan && k.rr <= calib && check_pair_match(S, i, j, err) >= 0) {
                    FP f;
                    const int cs = find_pair(S, i, j, K_HB, k.b, k.rr, f, 0, 0, err);
                    if (k.b < 0 && cs == 1 && calc_disc(k, f.lo) > 0) {
                        hpot = f.lopot;
                        double t = calc_time(k, -1, f.lo);
                        if (t < 0) t = INFINIT;
                        ht = (t > 0) ? t : __builtin_inf();
                        hfl |= 2;
                    }
                }
            }
        }
    }
    C.t[kidx] = tout;
    C.pot[kidx] = pot;
    C.sub[kidx] = (signed char)sub;
    C.fl[kidx] = fl;
    C.ht[kidx] = ht;
    C.hpot[kidx] = hpot;
    C.hfl[kidx] = hfl;
}

// ---------------------------------------------------------------- lane-0 pieces
__device__ void job_assign_atom(Atom &A, SV &S, double t, double pot, int sub, int type, int j) {
    if (t > 0 && A.t > t) take_computed(A, S, t, pot, sub, type, j);
}

__device__ double next_normal(Sys &S, Smem &sm) {
    if (sm.zpos >= S.nz) { sm.err = ERR_NORMALS; return 1.0; }
    return G(S.zn)[sm.zpos++];
}

// PBCandCrossCellTime along axis n, TimePrediction.c:598-632 (INFINIT: none)
__device__ __forceinline__ double pcc_axis(SV &S, double pos, double v, int ci, int n) {
    double t = -1;
    const double lo = ci * S.cellsize[n + 1], hi = (ci + 1) * S.cellsize[n + 1];
    if (v > 0) t = (hi - pos + ZERO) / v;
    else if (v < 0) t = (lo - pos - ZERO) / v;
    return (t > 0 && INFINIT > t) ? t : INFINIT;
}

// HBTime for a bonded HB atom, TimePrediction.c:330-383
__device__ void hb_time_bonded(SV &S, const Smem &sm, Atom &A, int *err) {
    const int j = A.hbbond;
    if (dupable(S, A, j, SDMD_HB) && A.t > evt_now(S, sm, j)) { take_inherited(A, S, sm, j, SDMD_HB); return; }
    Kin k;
    calc_params_now(S, sm, A, j, k);
    FP f;
    int cs = find_pair(S, A.i, j, K_HB, k.b, k.rr, f, 0, 0, err);
    int s, sub;
    double d2, pot;
    if (k.b < 0 && calc_disc(k, f.lo) > 0) {
        s = -1; d2 = f.lo; pot = f.lopot;
        sub = (cs == 0) ? SDMD_CORECOLLI : SDMD_TBDCAPTR;
    } else {
        s = 1; d2 = f.hi; pot = f.hipot;
        sub = (cs == 1) ? SDMD_TBDHBBRIK : SDMD_TBDESCAP;
    }
    double t = calc_time(k, s, d2);
    if (t < 0) t = INFINIT;
    job_assign_atom(A, S, t, pot, sub, SDMD_HB, j);
}

// HBNeighborTime, TimePrediction.c:486-579
__device__ void hb_neighbor_time(SV &S, const Smem &sm, Atom &A, int *err) {
    int flag = 0;
    for (int n = 1; n <= A.nbstat; n++) {
        const int j = A.nbp[n];
        if (flag == 0) A.nbnum = n;
        if (dupable(S, A, j, SDMD_HBNE) && A.t > evt_now(S, sm, j)) {
            take_inherited(A, S, sm, j, SDMD_HBNE);
            A.nbnum = n;
            flag = 1;
            continue;
        }
        Kin k;
        calc_params_now(S, sm, A, j, k);
        int host, nb, partner;
        const bool ads = (A.role == 'A' || A.role == 'D' || A.role == 'S');
        if (ads && A.hbbond && G(S.hbnb)[A.hbbond] == j) { host = A.i; nb = j; partner = A.hbbond; }
        else { host = j; nb = A.i; partner = G(S.hbbond)[j]; }
        FP f;
        int cs = find_pair(S, nb, host, K_NEIGHBOR, k.b, k.rr, f, partner, 0, err);
        int s, sub;
        double d2, pot;
        if (k.b < 0 && calc_disc(k, f.lo) > 0) {
            s = -1; d2 = f.lo; pot = f.lopot;
            sub = (cs == 0) ? SDMD_CORECOLLI : SDMD_TBDCAPTR;
        } else {
            s = 1; d2 = f.hi; pot = f.hipot;
            sub = (cs == 1) ? SDMD_WELLBOUNC : SDMD_TBDESCAP;
        }
        double t = calc_time(k, s, d2);
        if (t < 0) t = INFINIT;
        if (t > 0 && A.t > t) {
            take_computed(A, S, t, pot, sub, SDMD_HBNE, j);
            A.nbnum = n;
            flag = 1;
        }
    }
}

// ---------------------------------------------------------------- Predict
// Stage atom i (one wave): the gathered words, one per lane.
__device__ __forceinline__ void stage_atom(const Sys &S, Atom &A, int i, int exclude, int below) {
    const int lane = threadIdx.x & 63;
    if (lane < NGATHER) ((int *)&A)[lane] = G(S.gbase[lane])[(size_t)i * S.gstride[lane]];
    if (lane == NGATHER) {
        const int role = G(S.role)[i];
        A.i = i;
        A.role = role;
        A.exclude = exclude;
        A.below = below;
        A.cnt_eval = 0;
        A.wt = __builtin_inf();
    }
}

// Second level (the waves of a team; rank r of nw): bonds, connection row,
// constraint shells and cell-crossing times on one wave each where the team
// has several, and the candidates of the 27 cells (DMD.c:117-121 order, each
// in list order: the cell arrays hold a list back to front) on all of them.
template <bool CELLS>
__device__ __forceinline__ void stage_neighbours(SV &S, const Smem &sm, Atom &A, Cand &C, int r, int nw, int *err) {
    const int lane = threadIdx.x & 63;
    // occupancy of the 27 cells, by every wave for itself
    const int cl = min(lane, 26);
    int n1 = A.cx + c_OX[cl], n2 = A.cy + c_OY[cl], n3 = A.cz + c_OZ[cl];
    if (n1 < 0) n1 = S.cellnum[1] - 1; else if (n1 >= S.cellnum[1]) n1 = 0;
    if (n2 < 0) n2 = S.cellnum[2] - 1; else if (n2 >= S.cellnum[2]) n2 = 0;
    if (n3 < 0) n3 = S.cellnum[3] - 1; else if (n3 >= S.cellnum[3]) n3 = 0;
    const int cell = n3 * S.cellnum[1] * S.cellnum[2] + n2 * S.cellnum[1] + n1 + 1;
    int cnt = G(S.ccnt)[cell];
    if (lane >= 27) cnt = 0;
    if (r == 0) {
        // connection row and constraints
        const int nrow = A.ro1 - A.ro, ncon = A.co1 - A.co;
        if (lane < 32) ((int *)C.conn)[lane] = 0;
        int rj = 0, rb = 0, rc = 0;
        if (lane < nrow) { rj = G(S.cmap_j)[A.ro + lane]; rb = G(S.cmap_bits)[A.ro + lane]; rc = G(S.cmap_con)[A.ro + lane]; }
        double dmin = 0, dmax = 0;
        int step0 = 0, nstep = 0;
        if (lane < ncon && lane < PCON) {
            const sdmd_pair *p = &S.con[A.co + lane];
            dmin = G(p)->dmin; dmax = G(p)->dmax; step0 = G(p)->step0; nstep = G(p)->nstep;
            C.con_dmin[lane] = dmin; C.con_dmax[lane] = dmax; C.con_nstep[lane] = nstep;
        }
        const int lo = lane_get(rj, 0), hi = nrow > 0 ? lane_get(rj, min(nrow, 64) - 1) : lo;
        const bool spanok = nrow <= 64 && hi - lo < 128;
        const int slot = rc - A.co;                       // rc < 0: no constraint
        const int ns = __shfl(nstep, slot & 15, 64);
        if (lane < nrow && spanok) {
            const bool staged = rc >= 0 && slot >= 0 && slot < PCON && ns <= PCONSTEP;
            C.conn[rj - lo] = (unsigned char)((rb & (SDMD_BOND_CONNECT | SDMD_CONSTRAINT_CONNECT)) | (staged ? (slot + 1) << 2 : 0));
        }
        if (lane == 0) { A.spanok = spanok; A.rowlo = lo; }
#pragma unroll
        for (int u = 0; u < PCON * PCONSTEP / 64; u++) {
            const int q = (lane + 64 * u) / PCONSTEP, k = lane % PCONSTEP;
            const int s0 = __shfl(step0, q, 64), sn = __shfl(nstep, q, 64);
            if (q < ncon && k < sn) { C.con_d[q][k] = G(S.sd)[s0 + k]; C.con_e[q][k] = G(S.se)[s0 + k]; }
        }
    }
    if (r == nw - 1) {
        const int nb = A.bo1 - A.bo;
        if (lane < min(nb, MAXBOND)) eval_bond(S, sm, A, C, lane);
        else if (lane >= 32 && lane < 35) {
            const int n = lane - 32;
            C.pcc[n] = pcc_axis(S, n == 0 ? A.x : n == 1 ? A.y : A.z, n == 0 ? A.vx : n == 1 ? A.vy : A.vz,
                                n == 0 ? A.cx : n == 1 ? A.cy : A.cz, n);
        }
        if (lane == 0) A.nb = nb;
        if (nb > MAXBOND) *err = ERR_CELLCAP;
    }
    const int incl = scan32_incl(cnt);
    const int off = incl - cnt;
    const bool over = __ballot(cnt > CELL_CAP) != 0, broken = __ballot(cnt > S.N) != 0;
    const int ntot = lane_get(incl, 26);
    if (r == 0) {
        if (lane < 27) {
            C.cellcnt[lane] = cnt;
            C.celloff[lane] = off;
            // PBCShift, ToolFunctions.c:801-817, for the cell's atoms
            const int ci[3] = {A.cx, A.cy, A.cz}, cj[3] = {n1, n2, n3};
            for (int n = 0; n < 3; n++) {
                double s = 0;
                if (ci[n] != cj[n]) {
                    if (ci[n] == 0 && cj[n] == S.cellnum[n + 1] - 1) s = -1 * S.box[n + 1];
                    else if (ci[n] == S.cellnum[n + 1] - 1 && cj[n] == 0) s = S.box[n + 1];
                }
                C.shift[lane][n] = s;
            }
            if (broken) *err = ERR_LINKLIST;
        }
        if (lane == 27) C.celloff[27] = incl;             // lanes 27.. repeat the total
        if (lane == 0) {
            A.over = over && !broken;
            A.ncand = broken ? 0 : ntot;             // a broken list: no scan (the error ends the run)
        }
    }
    if (CELLS && !over && ntot <= PWIN) {
        // four cells at a time, 16 atoms of each per load
        int v[7];
#pragma unroll
        for (int u = 0; u < 7; u++) {
            const int c = (u * nw + r) * 4 + (lane >> 4), q = lane & 15;
            const int cc = __shfl(cnt, min(c, 31), 64), id = __shfl(cell, min(c, 26), 64);
            v[u] = (c < 27 && q < cc) ? G(S.cmem)[(size_t)id * CELL_CAP + q] : 0;
        }
#pragma unroll
        for (int u = 0; u < 7; u++) {
            const int c = (u * nw + r) * 4 + (lane >> 4);
            const int cc = __shfl(cnt, min(c, 31), 64), o = __shfl(off, min(c, 31), 64), id = __shfl(cell, min(c, 26), 64);
            if (c < 27) {
                int q = lane & 15;
                if (q < cc) { C.j[o + cc - 1 - q] = v[u]; C.cell[o + cc - 1 - q] = (unsigned char)c; }
                for (q += 16; q < cc; q += 16) {
                    C.j[o + cc - 1 - q] = G(S.cmem)[(size_t)id * CELL_CAP + q];
                    C.cell[o + cc - 1 - q] = (unsigned char)c;
                }
            }
        }
    }
}

// The predicted atom's record from the evaluated entries, in the reference's
// order (one wave): bonds and collisions ...
__device__ __forceinline__ void select_bonds(SV &S, const Smem &sm, Atom &A, Cand &C) {
    double m = A.t;
    int win = -1, inh = 0;
    wave_select(min(A.nb, MAXBOND), C.bt, C.bfl, [&](int d) { return C.bjt[d]; }, m, win, inh);
    if ((threadIdx.x & 63) == 0 && win >= 0) {
        if (inh) take_inherited(A, S, sm, C.bj[win], SDMD_BOND);
        else take_computed(A, S, C.bt[win], 0, C.bsub[win], SDMD_BOND, C.bj[win]);
    }
}
__device__ __forceinline__ void select_collisions(SV &S, const Smem &sm, Atom &A, Cand &C, int n) {
    double m = A.t;
    int win = -1, inh = 0;
    wave_select(n, C.t, C.fl, [&](int d) { return evt_now(S, sm, C.j[d]); }, m, win, inh);
    if ((threadIdx.x & 63) == 0 && win >= 0) {
        if (inh) take_inherited(A, S, sm, C.j[win], SDMD_COLI);
        else take_computed(A, S, C.t[win], C.pot[win], C.sub[win], SDMD_COLI, C.j[win]);
    }
}
// ... cell crossing, thermostat, the bonded H-bond partner (lane 0) ...
__device__ __forceinline__ void assign_onebody(SV &S, const Smem &sm, Atom &A, const Cand &C, int *err) {
    double t_ev = INFINIT;
    for (int n = 0; n < 3; n++)
        if (t_ev > C.pcc[n]) t_ev = C.pcc[n];
    job_assign_atom(A, S, t_ev, 0, SDMD_INVALID_INTER, SDMD_PCC, 0);
    if (S.thermostat) {
        const double z = A.zn;
        job_assign_atom(A, S, S.thermoF * ((z < 0) ? (-z) : (z)), 0, SDMD_INVALID_INTER, SDMD_THER, 0);
    }
    // HBTime head, TimePrediction.c:309-330
    if (A.hbitype != SDMD_HBSKIP && A.hbbond > 0) hb_time_bonded(S, sm, A, err);
}
// ... the free H-bond scan ...
__device__ __forceinline__ void select_hbonds(SV &S, const Smem &sm, Atom &A, Cand &C, int n) {
    double m = A.t;
    int win = -1, inh = 0;
    wave_select(n, C.ht, C.hfl, [&](int d) { return evt_now(S, sm, C.j[d]); }, m, win, inh);
    if ((threadIdx.x & 63) == 0 && win >= 0) {
        if (inh) take_inherited(A, S, sm, C.j[win], SDMD_HB);
        else take_computed(A, S, C.ht[win], C.hpot[win], SDMD_TBDHBFORM, SDMD_HB, C.j[win]);
    }
}
// ... H-bond neighbours and the wall, and the record stored (lane 0)
__device__ __forceinline__ void assign_tail(SV &S, const Smem &sm, Atom &A, int *err) {
    hb_neighbor_time(S, sm, A, err);
    if (S.wall) {
        WallEv w;
        if (wall_time(S, A.y, A.z, A.vy, A.vz, A.type, w, err)) {
            A.wt = w.t;
            job_assign_atom(A, S, w.t, w.pot, w.sub, SDMD_WALL, 0);
        }
    }
    const int i = A.i;
    G(S.evt)[i] = A.t; G(S.evpot)[i] = A.pot; G(S.evpc)[i] = A.pc;
    G(S.evp)[i] = A.partner; G(S.evtype)[i] = A.evtype; G(S.evsub)[i] = A.sub;
    G(S.nbnum)[i] = A.nbnum;
    G(S.hbitype)[i] = SDMD_NOEVENT;
}

__device__ __forceinline__ void finish_atom(SV &S, unsigned long long *prof, unsigned long long &pt, const Smem &sm, Atom &A,
                                            Cand &C, int *err) {
    const int lane = threadIdx.x & 63, n = A.ncand;
    select_bonds(S, sm, A, C);
    wave_sync();
    FPROF(prof, PH_BONDSEL, pt);
    select_collisions(S, sm, A, C, n);
    wave_sync();
    if (lane == 0) assign_onebody(S, sm, A, C, err);
    wave_sync();
    FPROF(prof, PH_SELECT, pt);
    if (A.hbscan) select_hbonds(S, sm, A, C, n);
    wave_sync();
    FPROF(prof, PH_HB, pt);
    if (lane == 0) assign_tail(S, sm, A, err);
}

// The free H-bond scan runs unless the last event of the atom was a skipped
// H-bond (HBTime head, TimePrediction.c:309-330)
__device__ __forceinline__ int wants_hbscan(const Atom &A) {
    return A.hbitype != SDMD_HBSKIP && A.hbbond <= 0 && (A.role == 'A' || A.role == 'D' || A.role == 'S');
}

// The lists of cells that hold more atoms than their arrays, walked side by
// side, one lane per cell (the reference's, Events.c:158-200), into `ids`:
// atom | neighbour cell << 27.  Once per prediction: a walk is a chain of
// dependent loads (30 us for a cell of 185 atoms), and a window holds the
// lists of a few cells only.
__device__ __forceinline__ void walk_lists(SV &S, const Atom &A, const Cand &C, unsigned *ids) {
    if (threadIdx.x < 27) {
        const int c = threadIdx.x, end = C.celloff[c + 1];
        int j = G(S.celllist)[S.N + cell_index(S, A.cx, A.cy, A.cz, c)];
        for (int g = C.celloff[c]; j && g < end; g++, j = G(S.celllist)[j]) ids[g] = (unsigned)j | (unsigned)c << 27;
    }
}

// candidates [w0, w0 + n) of the staged atom's ordered list (all threads)
template <int B>
__device__ __forceinline__ void gather_window(SV &S, const Atom &A, Cand &C, const unsigned *ids, int w0, int n) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (!A.over) {
        for (int c = wave; c < 27; c += B / 64) {
            const int cnt = C.cellcnt[c], g = C.celloff[c] + cnt - 1 - lane - w0;
            if (lane < cnt && g >= 0 && g < n) {
                C.j[g] = G(S.cmem)[(size_t)cell_index(S, A.cx, A.cy, A.cz, c) * CELL_CAP + lane];
                C.cell[g] = (unsigned char)c;
            }
        }
    } else if (ids) {
        for (int k = threadIdx.x; k < n; k += B) {
            const unsigned v = ids[w0 + k];
            C.j[k] = (int)(v & 0x7ffffffu);
            C.cell[k] = (unsigned char)(v >> 27);
        }
    } else if (wave == 0 && lane < 27) {
        // more candidates than the other atom's arrays hold: the lists again
        int g = C.celloff[lane] - w0;
        if (g < n && C.celloff[lane + 1] > w0) {
            int j = G(S.celllist)[S.N + cell_index(S, A.cx, A.cy, A.cz, lane)];
            for (; j && g < n; g++, j = G(S.celllist)[j])
                if (g >= 0) { C.j[g] = j; C.cell[g] = (unsigned char)lane; }
        }
    }
    __syncthreads();
}

// The staged atom's prediction over windows of candidates: the running
// minimum (and CheckDuplication against it) carries over, so the result is
// that of one sequential pass.  All threads.
template <int B, bool TAB>
__device__ __forceinline__ void predict_windows(SV &S, unsigned long long *prof, unsigned long long &pt, Smem &sm,
                                                const PairTab *T, Atom &A, Cand &C, double calib, int *err) {
    const int tid = threadIdx.x, wave = tid >> 6;
    const int ntot = A.ncand;
    const int wsz = min(S.win, PWIN);
    // the other atom's candidate arrays hold nothing while windows are used
    Cand &other = &C == &sm.c[0] ? sm.c[1] : sm.c[0];
    static_assert(offsetof(Cand, hpot) == offsetof(Cand, t) + 3 * sizeof(double) * PWIN, "one block of times and energies");
    constexpr int IDS = 4 * PWIN * (int)(sizeof(double) / sizeof(unsigned));
    unsigned *ids = (A.over && ntot <= IDS && S.N < (1 << 27)) ? (unsigned *)other.t : nullptr;
    if (ids) {
        walk_lists(S, A, C, ids);
        __syncthreads();
    }
    FPROF(prof, PH_GATHER, pt);
    if (wave == 0) select_bonds(S, sm, A, C);
    FPROF(prof, PH_BONDSEL, pt);
    for (int pass = 0; pass < 2; pass++) {
        if (pass == 1) {
            FPROF(prof, PH_EVAL, pt);
            if (tid == 0) assign_onebody(S, sm, A, C, err);
            __syncthreads();
            FPROF(prof, PH_SELECT, pt);
            if (!A.hbscan) break;
        }
        for (int w0 = 0; w0 < ntot; w0 += wsz) {
            const int n = min(ntot - w0, wsz);
            gather_window<B>(S, A, C, ids, w0, n);
            int ev = 0;
            for (int k = tid; k < n; k += B) {
                eval_candidate<TAB>(S, sm, T, A, C, k, calib, err);
                ev += ((pass ? C.hfl[k] : C.fl[k]) >> 1) & 1;
            }
            if (ev) atomicAdd(&A.cnt_eval, ev);
            __syncthreads();
            if (wave == 0) {
                if (pass == 0) select_collisions(S, sm, A, C, n);
                else select_hbonds(S, sm, A, C, n);
            }
            __syncthreads();
        }
    }
    __syncthreads();
    FPROF(prof, PH_HB, pt);
    if (tid == 0) assign_tail(S, sm, A, err);
    __syncthreads();
}

// What a bulk prediction's resolution needs to know of an atom besides its
// record: the earliest time any other entry offered (one wave).  -1 where the
// record also depends on H-bond slots.
__device__ __forceinline__ double other_offers(SV &S, const Atom &A, const Cand &C) {
    const int lane = threadIdx.x & 63;
    double m = __builtin_inf();
    if (lane < min(A.nb, MAXBOND) && !(A.evtype == SDMD_BOND && C.bj[lane] == A.partner)) m = C.bt[lane];
    for (int k = lane; k < A.ncand; k += 64) {
        const bool p = C.j[k] == A.partner;
        if (!(p && A.evtype == SDMD_COLI)) m = fmin(m, C.t[k]);
        if (A.hbscan && !(p && A.evtype == SDMD_HB)) m = fmin(m, C.ht[k]);
    }
    if (lane == 0) {
        if (A.evtype != SDMD_PCC)
            for (int n = 0; n < 3; n++) m = fmin(m, C.pcc[n]);
        const double t = S.thermoF * ((A.zn < 0) ? (-A.zn) : (A.zn));
        if (S.thermostat && A.evtype != SDMD_THER && t > 0) m = fmin(m, t);
        if (A.evtype != SDMD_WALL && A.wt > 0) m = fmin(m, A.wt);
    }
    return (A.nbstat > 0 || A.hbbond > 0) ? -1 : wave_min_d(m);
}

// MODE of a prediction: one of the event loop or a single call; the first
// pass of a bulk prediction (no CheckDuplication, the draw by atom number,
// other_offers left in S.bulk_t2); a repeated one of a bulk prediction
// (CheckDuplication against the atoms before it, the same draw, no counting),
// which begins with what the first pass began with: the skipped H-bond event's
// flag above all, which a prediction takes back
enum { M_LOOP, M_BULK, M_AGAIN };

// Predict of up to two atoms whose records were already reset (ResetTarget),
// SGThread.c:158-211.  All threads call this.  Two atoms are predicted side
// by side, each by half of the workgroup's waves: their predictions read
// each other's record only through CheckDuplication, and the second atom's
// selection is repeated when the first one's new event names it (its
// evaluated candidates stay as they are).  Bound by the latency of one
// candidate's evaluation, not by throughput: 205 candidates occupy four
// wavefronts.
template <int B, bool TAB, int MODE = M_LOOP>
__device__ __forceinline__ void predict_atoms(Sys &M, SV &S, unsigned long long *prof, Smem &sm, const PairTab *T, int n, int i0, int i1) {
    constexpr int W = B / 64;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int nw = (W > 1 && n == 2) ? W / 2 : W;      // waves per team
    const int team = wave / nw, r = wave % nw;
    unsigned long long pt = prof ? wall_clock64() : 0;
    double calib = S.cutoffr * SDMD_EXTEND_RATIO;
    calib *= calib;
    int err = 0;
    for (int s = 0; s < n; s++)
        if ((s == team || (nw == W && team == 0)) && r == 0) {
            Atom &A = sm.A[s];
            const int i = s ? i1 : i0;
            stage_atom(M, A, i, MODE == M_BULK ? -1 : n == 2 ? (s ? i0 : i1) : 0, MODE == M_AGAIN ? i : INT_MAX);
            const long long zp = sm.zpos + (MODE == M_LOOP ? s : i - 1);
            if (lane == 0 && S.thermostat) A.zn = zp < S.nz ? G(S.zn)[zp] : 1.0;
        }
    __syncthreads();
    FPROF(prof, PH_STAGE, pt);
    for (int s = 0; s < n; s++)
        if (s == team || (nw == W && team == 0)) {
            Atom &A = sm.A[s];
            if (r == 0 && lane == 0) {
                if (MODE == M_BULK) {
                    G(S.bulk_pot)[A.i] = A.pot; G(S.bulk_pc)[A.i] = A.pc; G(S.bulk_sub)[A.i] = A.sub;
                    G(S.bulk_nbnum)[A.i] = A.nbnum; G(S.bulk_hbit)[A.i] = A.hbitype;
                }
                if (MODE == M_AGAIN) {
                    A.pot = G(S.bulk_pot)[A.i]; A.pc = G(S.bulk_pc)[A.i]; A.sub = G(S.bulk_sub)[A.i];
                    A.nbnum = G(S.bulk_nbnum)[A.i]; A.hbitype = G(S.bulk_hbit)[A.i];
                }
                A.hbscan = wants_hbscan(A);
                A.pot0 = A.pot; A.pc0 = A.pc; A.sub0 = A.sub; A.nbnum0 = A.nbnum;
            }
            stage_neighbours<true>(S, sm, A, sm.c[s], r, nw, &err);
        }
    if (err) atomicCAS(&sm.err, 0, err);
    __syncthreads();
    FPROF(prof, PH_GATHER, pt);
    const int wsz = min(S.win, PWIN);
    bool whole = true;
    for (int s = 0; s < n; s++) whole = whole && !sm.A[s].over && sm.A[s].ncand <= wsz;
    err = 0;
    if (whole) {
        for (int s = 0; s < n; s++)
            if (s == team || (nw == W && team == 0)) {
                Atom &A = sm.A[s];
                Cand &C = sm.c[s];
                int ev = 0;
                for (int k = r * 64 + lane; k < A.ncand; k += nw * 64) {
                    eval_candidate<TAB>(S, sm, T, A, C, k, calib, &err);
                    ev += ((C.fl[k] >> 1) & 1) + ((C.hfl[k] >> 1) & 1);
                }
                if (ev) atomicAdd(&A.cnt_eval, ev);
            }
        if (err) atomicCAS(&sm.err, 0, err);
        __syncthreads();
        FPROF(prof, PH_EVAL, pt);
        err = 0;
        for (int s = 0; s < n; s++)
            if ((s == team || (nw == W && team == 0)) && r == 0) {
                finish_atom(S, prof, pt, sm, sm.A[s], sm.c[s], &err);
                if (MODE == M_BULK) {
                    wave_sync();
                    const double t2 = other_offers(S, sm.A[s], sm.c[s]);
                    if (lane == 0) G(S.bulk_t2)[sm.A[s].i] = t2;
                }
            }
        __syncthreads();
        if (MODE == M_LOOP && n == 2) {
            const Atom &P = sm.A[0];
            Atom &A = sm.A[1];
            if (P.partner == i1) {                     // uniform: the record in LDS is final
                if (wave == 0) {
                    // CheckDuplication against the first atom's new record
                    Cand &C = sm.c[1];
                    const bool same = P.pc == A.counter;
                    if (same && P.evtype == SDMD_BOND && lane < min(A.nb, MAXBOND) && C.bj[lane] == i0) {
                        C.bfl[lane] = 1;
                        C.bjt[lane] = P.t;
                    }
                    if (same && (P.evtype == SDMD_COLI || P.evtype == SDMD_HB))
                        for (int k = lane; k < A.ncand; k += 64)
                            if (C.j[k] == i0) {
                                if (P.evtype == SDMD_COLI) C.fl[k] |= 1;
                                else C.hfl[k] |= (C.hfl[k] >> 2) & 1;
                            }
                    if (lane == 0) {
                        A.t = INFINIT; A.evtype = SDMD_INVD; A.partner = INVALID;
                        A.pot = A.pot0; A.pc = A.pc0; A.sub = A.sub0; A.nbnum = A.nbnum0;
                        A.exclude = 0;
                    }
                    wave_sync();
                    finish_atom(S, prof, pt, sm, A, C, &err);
                }
                __syncthreads();
            }
        }
    } else {
        for (int s = 0; s < n; s++) {
            Atom &A = sm.A[s];
            Cand &C = sm.c[s];
            if (MODE == M_LOOP && s == 1) {
                // the second atom's bonds again, now against the first
                // atom's new record
                if (threadIdx.x == 0) A.exclude = 0;
                __syncthreads();
                if (threadIdx.x < min(A.nb, MAXBOND)) eval_bond(S, sm, A, C, threadIdx.x);
                __syncthreads();
            }
            predict_windows<B, TAB>(S, prof, pt, sm, T, A, C, calib, &err);
            if (MODE == M_BULK && threadIdx.x == 0) G(S.bulk_t2)[A.i] = -1;
        }
    }
    if (err) atomicCAS(&sm.err, 0, err);
    if (threadIdx.x == 0 && S.thermostat && MODE == M_LOOP)   // one draw per predicted atom, in order
        for (int s = 0; s < n; s++) {
            if (sm.zpos < S.nz) sm.zpos++;
            else sm.err = ERR_NORMALS;
        }
    if (threadIdx.x == 0 && MODE != M_AGAIN)
        // statistics: candidates scanned, quadratic evaluations
        for (int s = 0; s < n; s++) {
            const Atom &A = sm.A[s];
            M.candidates += A.ncand > 0 ? A.ncand - 1 : 0;
            M.pair_evals += A.cnt_eval + min(A.nb, MAXBOND) + A.nbstat + (A.hbbond > 0 ? 1 : 0);
        }
    __syncthreads();
    FPROF(prof, PH_TAIL, pt);
}

// Predict(renewList) with ResetTarget, SGThread.c:158-211
template <int B, bool TAB>
__device__ void predict_list(Sys &M, SV &S, unsigned long long *prof, Smem &sm, const PairTab *T, const int *renew) {
    if (threadIdx.x == 0) {
        for (int n = 1; renew[n]; n++) {
            const int i = renew[n];
            G(S.evtype)[i] = SDMD_INVD;
            G(S.evt)[i] = INFINIT;
            G(S.evp)[i] = INVALID;
        }
    }
    __syncthreads();
    const bool two = renew[1] && renew[2] && renew[1] != renew[2];
    for (int n = 1; renew[n]; n += two ? 2 : 1)
        predict_atoms<B, TAB>(M, S, prof, sm, T, two ? 2 : 1, renew[n], two ? renew[2] : 0);
}

// ---------------------------------------------------------------- CBT, CBT.c
// the winner of a stretch of a path: its time, atom << 1 | (its level's
// sibling is to the right of all below)
struct PathMin {
    double t;
    int v;
    // this stretch above another one
    __device__ __forceinline__ void after(const PathMin &o) {
        if (!(t < o.t || (t == o.t && (v & 1)))) { t = o.t; v = o.v; }
    }
    // that of the lane a DPP move reads from (none: one that never wins)
    template <int CTRL, int ROWS>
    __device__ __forceinline__ PathMin from() const {
        const unsigned long long w = (unsigned long long)__double_as_longlong(t);
        const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)w, CTRL, ROWS, 0xF, false);
        const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0x7ff00000, (int)(unsigned)(w >> 32), CTRL, ROWS, 0xF, false);
        return {__longlong_as_double((long long)(((unsigned long long)hi << 32) | lo)),
                __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false)};
    }
};
// UpdateCBT (CBT.c:33-39, 56-83) for one or two renewed atoms, by one wave.
// A path's nodes follow from the leaf's index alone, so each lane holds one
// level (lanes 0..31 the first atom's path, 32..63 the second's): the path's
// node, the sibling on the way up and its current event time, read at once
// instead of level by level; the walk itself runs on registers.  Where the
// second path meets nodes the first has just written, it takes their new
// values.
__device__ __forceinline__ void cbt_update(SV &S, Smem &sm, int n, int a0, int l0, double t0, int a1, int l1, double t1) {
    const int lane = threadIdx.x & 63, half = lane >> 5, k = lane & 31;
    const int L = half ? l1 : l0;
    const bool on = half < n && k < 31 - __clz(L);
    const int f = on ? L >> (k + 1) : 1, sib = on ? (L >> k) ^ 1 : 1;
    int of = G(S.node)[f], sv = G(S.node)[sib];
    double st = evt_now(S, sm, on ? sv : a0);
    int nv = of;               // the node's new value and its time
    double nt = 0;
    bool done = false;         // the walk reached this lane's level
    for (int h = 0; h < n; h++) {
        if (h == 1) {
            // nodes of the first path among this path's nodes and siblings
            const int d0 = 31 - __clz(l0);
            const int ms = d0 - (31 - __clz(sib)), mf = d0 - (31 - __clz(f));
            const int qs = (half && ms >= 1 && (l0 >> ms) == sib) ? ms - 1 : -1;
            const int qf = (half && mf >= 1 && (l0 >> mf) == f) ? mf - 1 : -1;
            const int sn = __shfl(nv, max(qs, 0), 64), fn = __shfl(nv, max(qf, 0), 64);
            const double tn = __shfl(nt, max(qs, 0), 64);
            const int ds = __shfl((int)done, max(qs, 0), 64), df = __shfl((int)done, max(qf, 0), 64);
            if (qs >= 0 && ds) { sv = sn; st = tn; }
            if (qf >= 0 && df) { of = fn; nv = fn; }
        }
        const int a = h ? a1 : a0, d = 31 - __clz(h ? l1 : l0);
        const bool here = half == h && on;
        // node = (evt[left] < evt[right]) ? left : right: on equal times the
        // one to the right, so a level's winner is the smallest (time, place)
        // of the atom and the siblings up to there, and the sibling is to the
        // right where the path is the left child
        PathMin e = {here ? st : __builtin_inf(), here ? (sv << 1) | (int)!((L >> k) & 1) : 0};
        if (here && k == 0) e.after({h ? t1 : t0, a << 1});
        e.after(e.from<0x111, 0xF>());                 // row_shr:1, 2, 4, 8
        e.after(e.from<0x112, 0xF>());
        e.after(e.from<0x114, 0xF>());
        e.after(e.from<0x118, 0xF>());
        e.after(e.from<0x142, 0xA>());                 // row_bcast:15
        const int cur = e.v >> 1;
        // the walk ends where a node keeps its value, except on nodes that
        // held the atom itself from the leaf on
        const unsigned changed = (unsigned)(__ballot(here && of != a) >> (32 * h));
        const int first = changed ? __builtin_ctz(changed) : 32;
        const unsigned kept = (unsigned)(__ballot(here && k >= first && cur == of) >> (32 * h));
        const int last = kept ? __builtin_ctz(kept) : d - 1;
        if (here && k <= last) {
            nv = cur; nt = e.t; done = true;
            if (nv != of) G(S.node)[f] = nv;
        }
        if (lane == 32 * h + d - 1) sm.root = nv;      // the top level: node 1
        wave_sync();
    }
}

// CreateCBT (CBT.c:16-30).  Inserting atom a splits leaf a - 1: its atom
// moves to node 2 (a - 1), a takes node 2 (a - 1) + 1.  So the atom of a
// leaf depends on the leaf's number alone (the right child 2c + 1 holds c +
// 1, a left child what its parent held), and since no event time changes
// meanwhile every inner node is the winner of its two children.
template <int B>
__device__ void cbt_create(Sys &S) {
    const int N = S.N, tid = threadIdx.x;
    if (tid == 0) { G(S.node)[0] = 0; G(S.leaf)[0] = 0; S.count = N; }
    for (int m = N + tid; m < 2 * N; m += B) {
        const int c = m >> __builtin_ctz(m);           // up the left edge to a right child (or node 1)
        const int a = c == 1 ? 1 : (c >> 1) + 1;
        G(S.node)[m] = a;
        G(S.leaf)[a] = m;
    }
    __syncthreads();
    for (int hi = N - 1; hi >= 1;) {                   // level by level, the deepest first
        const int lo = 1 << (31 - __clz(hi));
        for (int m = lo + tid; m <= hi; m += B) {
            const int l = G(S.node)[2 * m], r = G(S.node)[2 * m + 1];
            G(S.node)[m] = (G(S.evt)[l] < G(S.evt)[r]) ? l : r;
        }
        __syncthreads();
        hi = lo - 1;
    }
}

// ThermostatEvent, Events.c:396-420 (Andersen, no flow terms)
__device__ void thermostat_event(Sys &S, Smem &sm, int i) {
    double sp[3];
    for (int n = 0; n < 3; n++) {
        do {
            const double variance = S.T / G(S.mass)[i];
            sp[n] = next_normal(S, sm) * sqrt(variance) + 0;
            sp[n] += 0.0 + 0.0 + 0.0 * (S.currenttime - 0.0);
        } while (sp[n] == 0 && sm.err == 0);
    }
    G(S.vx)[i] = sp[0]; G(S.vy)[i] = sp[1]; G(S.vz)[i] = sp[2];
}

// PBCandCrossCellEvent + PBC("part") + LinkList("part"), Events.c:158-272
__device__ void pcc_event(Sys &S, int i, int *err) {
    const int old[3] = {G(S.cx)[i], G(S.cy)[i], G(S.cz)[i]};
    double *c[3] = {S.x, S.y, S.z};
    int *ci[3] = {S.cx, S.cy, S.cz};
    for (int n = 0; n < 3; n++) {
        if (old[n] == 0 || old[n] == S.cellnum[n + 1] - 1) {
            for (int m = 0; m < (S.wall ? 1 : 3); m++) {   // PBC: a cylinder wraps x only
                if (c[m][i] >= S.box[m + 1]) c[m][i] -= S.box[m + 1];
                else if (c[m][i] < 0) c[m][i] += S.box[m + 1];
            }
            break;
        }
    }
    const int N = S.N;
    const int oldc = old[2] * S.cellnum[1] * S.cellnum[2] + old[1] * S.cellnum[1] + old[0] + 1;
    for (int n = 0; n < 3; n++) {
        int v = (int)(c[n][i] / S.cellsize[n + 1]);
        if (v == S.cellnum[n + 1]) v--;
        if (v < 0 || v >= S.cellnum[n + 1]) { *err = ERR_CELL; return; }
        ci[n][i] = v;
    }
    const int newc = G(S.cz)[i] * S.cellnum[1] * S.cellnum[2] + G(S.cy)[i] * S.cellnum[1] + G(S.cx)[i] + 1;
    // out of the old cell: its array holds the list back to front, so the
    // atom before i in the list is the next array entry (or the list's head)
    int *m = S.cmem + (size_t)oldc * CELL_CAP;
    const int cnt = G(S.ccnt)[oldc];
    int nx = oldc + N;
    if (cnt <= CELL_CAP) {
        int q = 0;
        while (q < cnt && G(m)[q] != i) q++;
        if (q >= cnt) { *err = ERR_LINKLIST; return; }
        if (q < cnt - 1) nx = G(m)[q + 1];
        for (; q < cnt - 1; q++) G(m)[q] = G(m)[q + 1];
    } else {
        int guard = 0;
        while (G(S.celllist)[nx] != i) {
            nx = G(S.celllist)[nx];
            if (nx == 0 || ++guard > N) { *err = ERR_LINKLIST; return; }
        }
    }
    G(S.celllist)[nx] = G(S.celllist)[i];
    G(S.ccnt)[oldc] = cnt - 1;
    if (cnt == CELL_CAP + 1) {                          // the list fits its array again
        int j = G(S.celllist)[oldc + N];
        for (int q = CELL_CAP - 1; q >= 0 && j; q--, j = G(S.celllist)[j]) G(m)[q] = j;
    }
    // into the new one, at the head
    const int cn = G(S.ccnt)[newc];
    G(S.celllist)[i] = G(S.celllist)[newc + N];
    G(S.celllist)[newc + N] = i;
    if (cn < CELL_CAP) G(S.cmem)[(size_t)newc * CELL_CAP + cn] = i;
    G(S.ccnt)[newc] = cn + 1;
}

__device__ void do_event(Sys &S, Smem &sm, int t, int p, int *err) {   // DoEvent, Events.c:25-114
    const int ty = G(S.evtype)[t];
    const PosLazy pos{S, sm};
    switch (ty) {
    case SDMD_COLI: case SDMD_BOND: case SDMD_HBNE:
        interaction_event(S, pos, t, p, 0, 0, err);
        break;
    case SDMD_HB: {
        const int nbi = G(S.hbnb)[t], nbj = G(S.hbnb)[p];
        interaction_event(S, pos, t, p, nbi, nbj, err);
        hb_event(S, t, p, nbi, nbj, err);
        break;
    }
    case SDMD_THER: thermostat_event(S, sm, t); break;
    case SDMD_PCC: pcc_event(S, t, err); break;
    case SDMD_WALL: {
        double vx = G(S.vx)[t], vy = G(S.vy)[t], vz = G(S.vz)[t];
        wall_event(S, G(S.y)[t], G(S.z)[t], vx, vy, vz, G(S.mass)[t], G(S.evpot)[t], G(S.evsub)[t], err);
        G(S.vx)[t] = vx; G(S.vy)[t] = vy; G(S.vz)[t] = vz;
        break;
    }
    default: *err = ERR_EVENTTYPE; return;
    }
    if (ty >= 0 && ty < 16) S.per_type[ty]++;
}

// One pop up to its re-predictions (wave 0): AssignJob, UpdateData and
// TimeForward of the event's atoms, HazardCheck, DoEvent, the event counters
// and ResetTarget.  Lane 0 holds the target, lane 1 the partner: their state
// is loaded side by side, and a collision, bond or H-bond-neighbour event
// (InteractionEvent without its H-bond branch, Events.c:770-1025) runs on
// registers.
__device__ __forceinline__ void pop_event(Sys &M, SV &S, unsigned long long *prof, unsigned long long &pt, Smem &sm) {
    const int lane = threadIdx.x & 63;
    const int target = sm.root, n0 = sm.nlog;
    const int p0 = G(S.evp)[target], ty = G(S.evtype)[target], sub = G(S.evsub)[target];
    const double pot0 = G(S.evpot)[target];
    const long long pc = G(S.evpc)[target];
    const int partner = p0 > 0 ? p0 : 0;
    const int a = (lane == 1 && partner) ? partner : target;
    double x = G(S.x)[a], y = G(S.y)[a], z = G(S.z)[a], t = G(S.evt)[a];
    double vx = G(S.vx)[a], vy = G(S.vy)[a], vz = G(S.vz)[a];
    const double mass = G(S.mass)[a];
    const long long counter = G(S.evc)[a];
    const int cx = G(S.cx)[a], cy = G(S.cy)[a], cz = G(S.cz)[a];
    for (int l = lag_of(S, n0, a); l < n0; l++) {
        const double h = sm.log[l];
        x = x + vx * h; y = y + vy * h; z = z + vz * h; t = t - h;
    }
    const double dt = lane_get(t, 0);
    if (S.trace) {
        if (M.trace_n < S.trace_cap) {
            if (lane == 0) {
                sdmd_gpu_pop_rec &r = S.trace[M.trace_n];
                r.target = target; r.partner = p0; r.type = ty; r.sub = sub; r.dt = dt; r.pot = pot0;
            }
        } else {
            if (lane == 0) sm.err = ERR_TRACE;
            return;
        }
    }
    FPROF(prof, PH_POP, pt);
    x = x + vx * dt; y = y + vy * dt; z = z + vz * dt; t = t - dt;
    const bool mine = lane == 0 || (lane == 1 && partner);
    if (mine) {
        G(S.x)[a] = x; G(S.y)[a] = y; G(S.z)[a] = z; G(S.evt)[a] = t;
        G(S.lag)[a] = (unsigned char)(n0 + 1);
    }
    const bool stale = partner && pc < lane_get(counter, 1);       // HazardCheck, SGThread.c:215-235
    const bool pair = partner && (ty == SDMD_COLI || ty == SDMD_BOND || ty == SDMD_HBNE);
    int err = 0;
    if (lane == 0) {
        sm.log[n0] = dt;
        sm.nlog = n0 + 1;
        sm.dt = dt;
        sm.target = target;
        sm.partner = partner;
        sm.stale = stale;
        M.currenttime += dt;
        sm.renew[0] = (partner && !stale) ? 2 : 1;
        sm.renew[1] = target;
        sm.renew[2] = (partner && !stale) ? partner : 0;
        sm.renew[3] = 0;
        if (stale) M.recal++;
        else M.frame++;
        sm.flush = n0 + 1 >= S.logk || (S.hash_every > 0 && (M.pops + 1) % S.hash_every == 0);
    }
    if (!stale && pair) {
        // InteractionEvent, Events.c:798-1024, from the two lanes' state
        const int ci[3] = {lane_get(cx, 0), lane_get(cy, 0), lane_get(cz, 0)};
        const int cj[3] = {lane_get(cx, 1), lane_get(cy, 1), lane_get(cz, 1)};
        double pj[3] = {lane_get(x, 1), lane_get(y, 1), lane_get(z, 1)};
        const double pi[3] = {lane_get(x, 0), lane_get(y, 0), lane_get(z, 0)};
        const double vi[3] = {lane_get(vx, 0), lane_get(vy, 0), lane_get(vz, 0)};
        const double vj[3] = {lane_get(vx, 1), lane_get(vy, 1), lane_get(vz, 1)};
        const double mi = lane_get(mass, 0), mj = lane_get(mass, 1);
        for (int n = 0; n < 3; n++) {
            if (ci[n] != cj[n]) {
                if (ci[n] == 0 && cj[n] == S.cellnum[n + 1] - 1) pj[n] -= S.box[n + 1];
                else if (ci[n] == S.cellnum[n + 1] - 1 && cj[n] == 0) pj[n] += S.box[n + 1];
            }
        }
        const double r1 = pi[0] - pj[0], r2 = pi[1] - pj[1], r3 = pi[2] - pj[2];
        const double v1 = vi[0] - vj[0], v2 = vi[1] - vj[1], v3 = vi[2] - vj[2];
        const double d2 = r1 * r1 + r2 * r2 + r3 * r3;
        const double b = r1 * v1 + r2 * v2 + r3 * v3;
        const double mu = mi * mj / (mi + mj);
        double pot = pot0;
        int s = 0;
        bool ok = true;
        switch (sub) {
        case SDMD_CORECOLLI: s = 1; pot = 0; break;
        case SDMD_WELLBOUNC: s = (b < 0) ? 1 : -1; pot = 0; break;
        case SDMD_WELLCAPTR: s = -1; break;
        case SDMD_WELLESCAP: s = (b < 0) ? -1 : 1; break;
        case SDMD_TBDCAPTR:
            if (b * b - 2 * d2 * pot / mu <= 0) { pot = 0; s = 1; } else s = -1;
            break;
        case SDMD_TBDESCAP:
            if (b * b - 2 * d2 * pot / mu <= 0) { pot = 0; s = (b < 0) ? 1 : -1; }
            else s = (b < 0) ? -1 : 1;
            break;
        default: err = ERR_SUBTYPE; ok = false; break;
        }
        if (ok) {
            const double phi = (-1 * b + s * sqrt((b * b - 2 * d2 * pot / mu))) / ((mi + mj) * d2);
            if (isnan(phi)) {
                err = ERR_PHI_NAN;
            } else {
                const double fi = mj * phi, fj = mi * phi;
                if (lane == 0) { vx = vx + fi * r1; vy = vy + fi * r2; vz = vz + fi * r3; }
                else { vx = vx - fj * r1; vy = vy - fj * r2; vz = vz - fj * r3; }
                if (mine) { G(S.vx)[a] = vx; G(S.vy)[a] = vy; G(S.vz)[a] = vz; }
            }
        }
        if (lane == 0) M.per_type[ty]++;
    } else if (!stale && lane == 0) {
        do_event(M, sm, target, partner, &err);
        if (!err) err = sm.err;                    // a thermostat event's draws used up
    }
    const bool failed = __ballot(err != 0) != 0;
    if (failed && lane == 0 && !sm.err) sm.err = err;
    // SGThread.c:100-104, then ResetTarget of the renewed atoms; a failed
    // event is the last of the run and leaves the records as they are
    if (mine && !stale) G(S.evc)[a] = counter + 1;
    if (!failed && (lane == 0 || (lane == 1 && partner && !stale))) {
        G(S.evtype)[a] = SDMD_INVD;
        G(S.evt)[a] = INFINIT;
        G(S.evp)[a] = INVALID;
    }
}

__device__ unsigned long long fnv(unsigned long long h, const void *p, int n) {
    const unsigned char *c = (const unsigned char *)p;
    for (int i = 0; i < n; i++) { h ^= c[i]; h *= 1099511628211ULL; }
    return h;
}

__device__ unsigned long long state_hash(const Sys &S) {
    unsigned long long h = 1469598103934665603ULL;
    for (int i = 1; i <= S.N; i++) {
        const double p[3] = {G(S.x)[i], G(S.y)[i], G(S.z)[i]}, v[3] = {G(S.vx)[i], G(S.vy)[i], G(S.vz)[i]};
        const long long c = G(S.evc)[i];
        h = fnv(h, p, sizeof p);
        h = fnv(h, v, sizeof v);
        h = fnv(h, &S.evt[i], sizeof(double));
        h = fnv(h, &c, sizeof c);
    }
    return h;
}

// ---------------------------------------------------------------- kernels
// The system struct is copied into LDS for the kernel's lifetime: its
// pointers and constants are then LDS reads instead of dependent global
// loads, and the run scalars it holds are written back at the end.
template <int B>
__device__ __forceinline__ void sys_load(Sys &dst, const Sys *src) {
    const int n = (int)(sizeof(Sys) / sizeof(int));
    for (int k = threadIdx.x; k < n; k += B) ((int *)&dst)[k] = ((const int *)src)[k];
    __syncthreads();
}

template <int B>
__device__ __forceinline__ void sys_store(Sys *dst, const Sys &src) {
    __syncthreads();
    const int n = (int)(sizeof(Sys) / sizeof(int));
    for (int k = threadIdx.x; k < n; k += B) ((int *)dst)[k] = ((const int *)&src)[k];
}

// the collision table and the tables' step pool into LDS
template <int B>
__device__ __forceinline__ void tab_load(PairTab &T, const Sys &S) {
    for (int k = threadIdx.x; k < NT * NT; k += B) {
        const sdmd_pair *p = S.rpair + k;
        T.dmin[k] = G(p)->dmin; T.dmax[k] = G(p)->dmax; T.step0[k] = G(p)->step0; T.nstep[k] = G(p)->nstep;
    }
    if (S.ltab)
        for (int k = threadIdx.x; k < S.ltab; k += B) { T.d[k] = G(S.sd)[k]; T.e[k] = G(S.se)[k]; }
    __syncthreads();
}

#ifndef SDMD_PLAIN_RUN
// ---------------------------------------------------------------- bulk Predict(1..N)
// Prepare predicts the atoms in order (SGThread.c:47-62), and atom i's
// CheckDuplication may take over the record of an earlier atom j whose event
// names i.  Everything else of a prediction is independent of the order, so
// (1) every atom is predicted without CheckDuplication, all over the GPU,
// together with the earliest time any entry but its winner offers (t2);
// (2) each atom's earlier namers j -- those with a pair event naming it -- are
//     linked to it;
// (3) each atom with namers is resolved.  A namer's own event names a later
//     atom, so it has taken over nothing and its record is that of (1).
//     Running minimum of the reference's scan: if a namer j is the atom's
//     own winner (same pair, same type) with e_j its event time, and e_j is
//     earlier than t2 and than every other namer's event, j's record is
//     taken over whatever the order of the entries; if no namer is the
//     winner and every e_j is later than the winner's time, none is;
// (4) the atoms left (ties, H-bond slots, windowed scans) are predicted again
//     in order with CheckDuplication against the atoms before them, and with
//     them any later atom that one of their changed records names.
// One workgroup per system predicting atom after atom took 45 ms for 5 000
// atoms (9 us each).
__global__ __launch_bounds__(256) void k_bulk_reset(Sys *systems) {
    const Sys &S = systems[blockIdx.x];
    if (blockIdx.y == 0 && threadIdx.x == 0) systems[blockIdx.x].bulk_err = 0;
    for (int i = 1 + blockIdx.y * 256 + threadIdx.x; i <= S.N; i += 256 * gridDim.y) {   // ResetTarget for 1..N
        G(S.evtype)[i] = SDMD_INVD;
        G(S.evt)[i] = INFINIT;
        G(S.evp)[i] = INVALID;
        G(S.bulk_head)[i] = 0;
        G(S.bulk_flag)[i] = 0;
    }
}

template <int B>
__global__ __launch_bounds__(B) void k_bulk_predict(Sys *systems, int per) {
    const int first = 1 + blockIdx.y * per;            // this workgroup's atoms: [first, first + per)
    if (first > systems[blockIdx.x].N) return;
    __shared__ Smem sm;
    __shared__ Sys Sl;
    __shared__ PairTab tab;
    Sys &Sg = systems[blockIdx.x];
    SV &V = fixed_view(systems + blockIdx.x);
    sys_load<B>(Sl, &Sg);
    Sys &S = Sl;
    tab_load<B>(tab, S);
    if (threadIdx.x == 0) {
        sm.err = 0; sm.zpos = S.zpos; sm.nlog = 0;
        S.candidates = S.pair_evals = 0;               // this workgroup's counts
    }
    __syncthreads();
    const int last = min(first + per - 1, S.N);
    for (int i = first; i <= last; i += 2)
        predict_atoms<B, true, M_BULK>(S, V, nullptr, sm, &tab, i < last ? 2 : 1, i, i + 1);
    if (threadIdx.x == 0) {
        atomicAdd((unsigned long long *)&Sg.candidates, (unsigned long long)S.candidates);
        atomicAdd((unsigned long long *)&Sg.pair_evals, (unsigned long long)S.pair_evals);
        if (sm.err) atomicCAS(&Sg.bulk_err, 0, sm.err);
    }
}

__global__ __launch_bounds__(256) void k_bulk_link(Sys *systems) {
    const Sys &S = systems[blockIdx.x];
    for (int j = 1 + blockIdx.y * 256 + threadIdx.x; j <= S.N; j += 256 * gridDim.y) {
        const int p = G(S.evp)[j];
        if (p > j && p <= S.N) S.bulk_next[j] = atomicExch(&S.bulk_head[p], j);
    }
}

__global__ __launch_bounds__(256) void k_bulk_resolve(Sys *systems) {
    const Sys &S = systems[blockIdx.x];
    for (int i = 1 + blockIdx.y * 256 + threadIdx.x; i <= S.N; i += 256 * gridDim.y) {
        const int head = G(S.bulk_head)[i];
        if (!head) continue;
        const int p = G(S.evp)[i], type = G(S.evtype)[i];
        const double t = G(S.evt)[i], t2 = G(S.bulk_t2)[i];
        int win = 0;                                   // the namer that is the winner
        double e = __builtin_inf();                    // the earliest event of the other namers
        for (int j = head; j; j = G(S.bulk_next)[j]) {
            if (j == p && G(S.evtype)[j] == type) win = j;
            else e = fmin(e, G(S.evt)[j]);
        }
        if (t2 < 0) {
            G(S.bulk_flag)[i] = 1;
        } else if (!win) {
            if (!(e > t)) G(S.bulk_flag)[i] = 1;
        } else {
            const double ew = G(S.evt)[win];
            if (ew < t2 && ew < e) {                   // CheckDuplication's inheritance
                G(S.evpot)[i] = G(S.evpot)[win];
                G(S.evsub)[i] = G(S.evsub)[win];
                G(S.evt)[i] = ew;
                G(S.evpc)[i] = G(S.evc)[win];
            } else {
                G(S.bulk_flag)[i] = 1;
            }
        }
    }
}

// (4) and the tree, one workgroup per system
template <int B>
__global__ __launch_bounds__(B) void k_bulk_finish(Sys *systems) {
    __shared__ Smem sm;
    __shared__ Sys Sl;
    __shared__ PairTab tab;
    __shared__ int next;
    sys_load<B>(Sl, &systems[blockIdx.x]);
    Sys &S = Sl;
    SV &V = fixed_view(systems + blockIdx.x);
    const int tid = threadIdx.x, N = S.N;
    if (tid == 0) { sm.err = S.bulk_err; sm.zpos = S.zpos; sm.nlog = 0; next = INT_MAX; }
    __syncthreads();
    bool loaded = false;
    int from = 1;
    while (from <= N && sm.err == 0) {
        for (int i = from + tid; i <= N; i += B)       // the first flagged atom from `from` on
            if (G(S.bulk_flag)[i]) { atomicMin(&next, i); break; }
        __syncthreads();
        const int i = next;
        __syncthreads();
        if (i > N) break;
        if (!loaded) { tab_load<B>(tab, S); loaded = true; }
        const int p0 = G(S.evp)[i], ty0 = G(S.evtype)[i];
        const double t0 = G(S.evt)[i];
        __syncthreads();
        if (tid == 0) {
            next = INT_MAX;
            G(S.evtype)[i] = SDMD_INVD;
            G(S.evt)[i] = INFINIT;
            G(S.evp)[i] = INVALID;
        }
        __syncthreads();
        predict_atoms<B, true, M_AGAIN>(S, V, nullptr, sm, &tab, 1, i, 0);
        if (tid == 0) {
            const int p1 = G(S.evp)[i];
            if (p1 != p0 || G(S.evtype)[i] != ty0 || G(S.evt)[i] != t0) {
                if (p0 > i && p0 <= N) G(S.bulk_flag)[p0] = 1;
                if (p1 > i && p1 <= N) G(S.bulk_flag)[p1] = 1;
            }
        }
        from = i + 1;
        __syncthreads();
    }
    const bool ok = sm.err == 0;
    if (ok) cbt_create<B>(S);
    __syncthreads();
    if (tid == 0) {
        if (S.thermostat) {
            S.zpos += N;
            if (S.zpos > S.nz) { S.zpos = S.nz; S.error = S.error ? S.error : ERR_NORMALS; }
        }
        if (sm.err) S.error = sm.err;
    }
    sys_store<B>(&systems[blockIdx.x], Sl);
}

#endif  // SDMD_PLAIN_RUN

// ---------------------------------------------------------------- event loop
// Compiled apart (this file with SDMD_PLAIN_RUN = 0 and = 1, beside the unit
// without it): phase times have kernels of their own, because their marks cost
// a run that takes none 2 %.
struct PlainRun {
    hipStream_t stream;
    Sys *sys;
    int nsys;
    long long npops, budget;
    double t_end, t_out;
};
template <int B, bool PROF> void plain_launch_run(const PlainRun &r);

#ifdef SDMD_PLAIN_RUN
// t_out: stop after the first executed event that leaves the clock at or
// past t_out -- where SingleThreadRun writes its output (SGThread.c:130-139)
template <int B, bool PROF>
__global__ __launch_bounds__(B) void k_run(Sys *systems, long long npops, long long budget, double t_end,
                                           double t_out) {
    __shared__ Smem sm;
    __shared__ Sys Sl;
    __shared__ PairTab tab;
    __shared__ int stop;
    sys_load<B>(Sl, &systems[blockIdx.x]);
    Sys &S = Sl;                           // counters and clock
    SV &V = fixed_view(systems + blockIdx.x);
    unsigned long long *const prof = PROF ? V.prof : nullptr;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const unsigned long long t_start = wall_clock64();
    // npops < 0 asks for -npops executed events instead of pops
    const long long maxpops = npops < 0 ? LLONG_MAX : npops, evgoal = npops < 0 ? -npops : LLONG_MAX;
    const long long frame0 = S.frame;
    if (S.error || maxpops == 0) return;
    tab_load<B>(tab, S);
    if (tid == 0) { sm.err = 0; sm.zpos = S.zpos; stop = 0; sm.nlog = 0; sm.root = G(S.node)[1]; }
    __syncthreads();
    unsigned long long pt = prof ? wall_clock64() : 0;
    for (long long pop = 0;; pop++) {
        if (wave == 0) {
            // device-time budget of a bounded run
            if (pop >= maxpops || (long long)(wall_clock64() - t_start) > budget || S.currenttime > t_end ||
                S.frame - frame0 >= evgoal || stop) {
                if (lane == 0) stop = 1;
            } else {
                pop_event(S, V, prof, pt, sm);
            }
        }
        __syncthreads();
        if (sm.err || stop) break;
        const int flush = sm.flush;        // wave 0 runs ahead into the next pop's event
        FPROF(prof, PH_EVENT, pt);
        predict_atoms<B, true>(S, V, prof, sm, &tab, sm.renew[0], sm.renew[1], sm.renew[2]);
        if (prof) pt = wall_clock64();
        if (flush) sweep<B>(V, sm);
        FPROF(prof, PH_SWEEP, pt);
        if (wave == 0) {
            cbt_update(V, sm, sm.renew[0], sm.renew[1], sm.A[0].leaf, sm.A[0].t, sm.renew[2], sm.A[1].leaf, sm.A[1].t);
            FPROF(prof, PH_TREE, pt);
            if (lane == 0) {
                S.pops++;
                S.last_exec = !sm.stale;
                // an error of a prediction ends the run here, before the next pop
                if (sm.err || (!sm.stale && S.currenttime >= t_out)) stop = 1;
                if (V.trace && S.trace_n < V.trace_cap) {
                    sdmd_gpu_pop_rec &r = S.trace[S.trace_n];
                    r.exec = !sm.stale;
                    r.rand_calls = sm.zpos;
                    int n = 0;
                    for (int k = 1; sm.renew[k] && n < 2; k++, n++) {
                        const int a = sm.renew[k];
                        r.r[n].atom = a; r.r[n].partner = G(S.evp)[a]; r.r[n].type = G(S.evtype)[a];
                        r.r[n].sub = G(S.evsub)[a]; r.r[n].counter = G(S.evc)[a]; r.r[n].pcounter = G(S.evpc)[a];
                        r.r[n].time = G(S.evt)[a]; r.r[n].pot = G(S.evpot)[a];
                    }
                    r.nrenew = n;
                    S.trace_n++;
                }
                if (V.hash_every > 0 && S.pops % V.hash_every == 0 && S.hash_n < S.hash_cap) {
                    G(S.hashes)[2 * S.hash_n] = S.pops;
                    G(S.hashes)[2 * S.hash_n + 1] = (long long)state_hash(S);
                    S.hash_n++;
                }
            }
            wave_sync();
        }
    }
    __syncthreads();
    if (sm.nlog) sweep<B>(V, sm);
    if (tid == 0) {
        S.zpos = sm.zpos;
        if (sm.err) S.error = sm.err;
    }
    sys_store<B>(&systems[blockIdx.x], Sl);
}

template <int B, bool PROF>
void plain_launch_run(const PlainRun &r) {
    hipLaunchKernelGGL((k_run<B, PROF>), dim3(r.nsys), dim3(B), 0, r.stream, r.sys, r.npops, r.budget, r.t_end, r.t_out);
}
template void plain_launch_run<64, SDMD_PLAIN_RUN>(const PlainRun &);
template void plain_launch_run<128, SDMD_PLAIN_RUN>(const PlainRun &);
template void plain_launch_run<256, SDMD_PLAIN_RUN>(const PlainRun &);
template void plain_launch_run<512, SDMD_PLAIN_RUN>(const PlainRun &);
template void plain_launch_run<1024, SDMD_PLAIN_RUN>(const PlainRun &);

}  // namespace sdmd
#else
// cell arrays from the lists, for every cell of every system
__global__ __launch_bounds__(256) void k_cells(const Sys *systems) {
    const Sys &S = systems[blockIdx.x];
    const int N = S.N, ncell = S.cellnum[1] * S.cellnum[2] * S.cellnum[3];
    for (int c = 1 + blockIdx.y * 256 + threadIdx.x; c <= ncell; c += 256 * gridDim.y) {
        int cnt = 0;
        for (int j = G(S.celllist)[N + c]; j && cnt <= N; j = G(S.celllist)[j]) cnt++;
        G(S.ccnt)[c] = cnt;
        if (cnt > CELL_CAP) continue;
        int q = cnt - 1;
        for (int j = G(S.celllist)[N + c]; j && q >= 0; j = G(S.celllist)[j]) G(S.cmem)[(size_t)c * CELL_CAP + q--] = j;
    }
}

// single operations behind the fine-grained entry points
enum { OP_PREDICT, OP_CREATE_TREE, OP_UPDATE_TREE, OP_DO_EVENT, OP_CELL_MOVE };

// CalKinetE + CalPotenE (ToolFunctions.c:626-752) of every system at its
// current time: one wavefront per atom i, one lane per neighbour cell
// (periodic wrap with position shift) walking its list for partners j > i.
// Bound by the lists' dependent loads, so the atoms are spread over the GPU:
// gridDim.y workgroups per system leave their sums in `part`
// (k_energy_reduce).
__global__ __launch_bounds__(64 * EWAVES) void k_energy(Sys *systems, double *part) {
    const Sys &S = systems[blockIdx.x];
    const int N = S.N, tid = threadIdx.x, lane = tid & 63;
    const double cut2 = S.cutoffr * S.cutoffr;
    const int c = min(lane, 26);
    Sum2 ke = {0, 0}, pe = {0, 0};
    int err = 0;
    for (int i = 1 + blockIdx.y * EWAVES + (tid >> 6); i <= N; i += EWAVES * gridDim.y) {
        const double xi = G(S.x)[i], yi = G(S.y)[i], zi = G(S.z)[i];
        const double vi[3] = {G(S.vx)[i], G(S.vy)[i], G(S.vz)[i]};
        if (lane == 0) ke.add(0.5 * G(S.mass)[i] * (vi[0] * vi[0] + vi[1] * vi[1] + vi[2] * vi[2]));
        int cc[3] = {G(S.cx)[i] + c_OX[c], G(S.cy)[i] + c_OY[c], G(S.cz)[i] + c_OZ[c]};
        double sh[3] = {0, 0, 0};
        for (int k = 0; k < 3; k++) {
            if (cc[k] < 0) { cc[k] = S.cellnum[k + 1] - 1; sh[k] = -1 * S.box[k + 1]; }
            else if (cc[k] >= S.cellnum[k + 1]) { cc[k] = 0; sh[k] = S.box[k + 1]; }
        }
        const int cell = cc[2] * S.cellnum[1] * S.cellnum[2] + cc[1] * S.cellnum[1] + cc[0] + 1;
        int guard = 0;
        for (int j = lane < 27 ? G(S.celllist)[N + cell] : 0; j && ++guard <= N; j = G(S.celllist)[j]) {
            if (j <= i) continue;
            const double r1 = xi - (G(S.x)[j] + sh[0]), r2 = yi - (G(S.y)[j] + sh[1]), r3 = zi - (G(S.z)[j] + sh[2]);
            const double rr = r1 * r1 + r2 * r2 + r3 * r3;
            if (rr > cut2) continue;
            const double vj[3] = {G(S.vx)[j], G(S.vy)[j], G(S.vz)[j]};
            pe.add(pair_energy(S, i, j, r1, r2, r3, rr, vi, vj, &err));
        }
    }
    energy_partial(ke, pe, err || S.error, part);
}

struct Renew { int a[4]; };                // a renew list by value (at most two atoms, zero-terminated)

template <int B>
__global__ __launch_bounds__(B) void k_op(Sys *systems, int sys, int op, Renew renew, int a, int b,
                                          sdmd_op_status *status) {
    __shared__ Smem sm;
    __shared__ Sys Sl;
    sys_load<B>(Sl, &systems[sys]);
    Sys &S = Sl;
    SV &V = fixed_view(systems + sys);
    const int tid = threadIdx.x;
    if (tid == 0) { sm.err = 0; sm.zpos = S.zpos; sm.nlog = 0; }
    __syncthreads();
    if (op == OP_CREATE_TREE) cbt_create<B>(S);
    if (op == OP_PREDICT) {
        predict_list<B, false>(S, V, V.prof, sm, nullptr, renew.a);
    } else if (op == OP_UPDATE_TREE) {
        const int n = renew.a[0];
        if (tid < 64 && n > 0) {
            const int a0 = renew.a[1], a1 = n > 1 ? renew.a[2] : a0;
            cbt_update(V, sm, n, a0, G(S.leaf)[a0], G(S.evt)[a0], a1, G(S.leaf)[a1], G(S.evt)[a1]);
        }
    } else if (tid == 0) {
        int err = 0;
        if (op == OP_DO_EVENT) {
            // SingleThreadRun, SGThread.c:100-104
            S.frame++;
            do_event(S, sm, a, b, &err);
            G(S.evc)[a]++;
            if (b > 0) G(S.evc)[b]++;
        } else if (op == OP_CELL_MOVE) pcc_event(S, a, &err);
        if (err) sm.err = err;
    }
    __syncthreads();
    if (tid == 0) {
        S.zpos = sm.zpos;
        if (sm.err) S.error = sm.err;
        status->error = S.error;
    }
    sys_store<B>(&systems[sys], Sl);
}

// UpdateData + TimeForward (ToolFunctions.c:23-36) of one system by dt
__global__ __launch_bounds__(256) void k_advance(Sys *systems, int sys, double dt, sdmd_op_status *status) {
    Sys &S = systems[sys];
    for (int i = 1 + blockIdx.x * 256 + threadIdx.x; i <= S.N; i += 256 * gridDim.x) {
        G(S.x)[i] += G(S.vx)[i] * dt;
        G(S.y)[i] += G(S.vy)[i] * dt;
        G(S.z)[i] += G(S.vz)[i] * dt;
        G(S.evt)[i] -= dt;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        S.currenttime += dt;
        status->error = S.error;
    }
}

// AssignJob's event and HazardCheck's verdict (SGThread.c:215-259); target 0:
// the tree holds no event
__global__ __launch_bounds__(64) void k_pop(const Sys *systems, int sys, sdmd_op_status *status) {
    const Sys &S = systems[sys];
    if (threadIdx.x != 0) return;
    const int root = G(S.node)[1];
    sdmd_gpu_event ev = {};
    if (root >= 1 && root <= S.N) {
        ev.target = root;
        ev.partner = G(S.evp)[root];
        ev.type = G(S.evtype)[root];
        ev.sub = G(S.evsub)[root];
        ev.time = G(S.evt)[root];
        ev.potential = G(S.evpot)[root];
        if (ev.partner > 0 && ev.partner <= S.N) ev.stale = G(S.evpc)[root] < G(S.evc)[ev.partner];
    }
    status->ev = ev;
}

}  // namespace sdmd

using namespace sdmd;

// ==================================================================== host side
// The words of a staged Atom in the order of its first NGATHER members:
// device address of the word for atom 0 and its stride from atom to atom.
static void atom_gather_table(Sys *S) {
    int w = 0;
    auto word = [&](const int *p, int stride) { S->gbase[w] = p; S->gstride[w] = stride; w++; };
    auto wide = [&](const void *p) { word((const int *)p, 2); word((const int *)p + 1, 2); };
    for (const double *p : {S->x, S->y, S->z, S->vx, S->vy, S->vz}) wide(p);
    wide(S->evc); wide(S->evt); wide(S->evpot); wide(S->evpc);
    for (const int *p : {S->cx, S->cy, S->cz, S->type, S->hbbond, S->hbnb, S->protein, S->aanum, S->nbstat, S->nbnum})
        word(p, 1);
    for (int k = 0; k < SDMD_NBSLOTS; k++) word(S->nbp + k, SDMD_NBSLOTS);
    for (const int *p : {S->evp, S->evtype, S->evsub, S->hbitype}) word(p, 1);
    for (const int *p : {S->cmap_off, S->bond_off, S->con_off}) { word(p, 1); word(p + 1, 1); }
    word(S->leaf, 1);
}

static int upload_system(sdmd_gpu_ctx *c, sdmd_arena *ar, int s, const sdmd_system_desc *d, const sdmd_gpu_opts *o) {
    Sys *S = &c->host_sys[s];
    memset(S, 0, sizeof *S);
    const int N = d->natom;
    const size_t N1 = (size_t)N + 1;
    S->N = N;
    S->ncelllist = d->ncelllist;
    for (int k = 0; k < 3; k++) {
        S->cellnum[k + 1] = d->cellnum[k];
        S->cellsize[k + 1] = d->cellsize[k];
        S->box[k + 1] = d->box[k];
    }
    S->cutoffr = d->cutoffr;
    S->T = d->temperature;
    S->thermoF = d->thermo_freq;
    S->thermostat = d->thermostat;
    for (int k = 0; k < 6; k++) S->hbpot[k] = d->hb_pot[k];
    S->wall = d->wall;
    S->wall_type = d->wall_type;
    for (int k = 0; k < 3; k++) S->wallpos[k + 1] = d->wall_pos[k];
    S->currenttime = d->currenttime;
    S->steps_sorted = 1;
    {
        auto check_list = [&](const sdmd_pair &p) {
            for (int k = 0; k < p.nstep; k++) {
                const double v = d->step_d[p.step0 + k];
                if (!(v > 0) || (k > 0 && !(v > d->step_d[p.step0 + k - 1]))) S->steps_sorted = 0;
            }
        };
        for (int k = 0; k < NT * NT; k++) check_list(d->pair[k]);
        for (int k = 0; k < SDMD_NHBCLASS * NT * NT; k++) check_list(d->hbpair[k]);
        for (int k = 0; k < d->con_off[d->natom + 1]; k++) check_list(d->con[k]);
    }
    int rc = 0;
#define UP(field, src, n) arena_add(ar, &S->field, src, n)
#define UPBIG(field, n) if ((rc = dev_upload(c, &S->field, (decltype(+S->field))nullptr, n))) return rc
    // what a run changes, first and in the order sdmd_dyn_scatter copies it back
    UP(x, d->x, N1); UP(y, d->y, N1); UP(z, d->z, N1);
    UP(vx, d->vx, N1); UP(vy, d->vy, N1); UP(vz, d->vz, N1);
    UP(type, d->type, N1); UP(cx, d->cellx, N1); UP(cy, d->celly, N1); UP(cz, d->cellz, N1);
    UP(hbbond, d->hb_bond, N1); UP(hbitype, d->hb_itype, N1);
    UP(nbp, d->nb_partner, N1 * SDMD_NBSLOTS); UP(nbnum, d->nb_partnernum, N1); UP(nbstat, d->nb_status, N1);
    UP(dynj, d->dyn_j, N1 * SDMD_DYNSLOTS); UP(dynb, d->dyn_bits, N1 * SDMD_DYNSLOTS);
    UP(evp, d->ev_partner, N1); UP(evtype, d->ev_type, N1); UP(evsub, d->ev_sub, N1);
    UP(evc, (const long long *)d->ev_counter, N1); UP(evpc, (const long long *)d->ev_pcounter, N1);
    UP(evt, d->ev_time, N1); UP(evpot, d->ev_pot, N1);
    UP(celllist, d->celllist, (size_t)d->ncelllist);
    c->dyn[s].bytes = ar->used;
    UP(mass, d->mass, N1); UP(aatype, d->aatype, N1); UP(protein, d->protein, N1); UP(aanum, d->aanum, N1);
    UP(role, (const signed char *)d->hb_role, N1);
    UP(hbnb, d->hb_neighbor, N1);
    const int nb = d->bond_off[N + 1], nc = d->con_off[N + 1], ncm = d->cmap_off[N + 1];
    UP(bond_off, d->bond_off, N1 + 1); UP(bond_j, d->bond_j, (size_t)nb);
    UP(bond_dmin, d->bond_dmin, (size_t)nb); UP(bond_dmax, d->bond_dmax, (size_t)nb);
    UP(con_off, d->con_off, N1 + 1); UP(con_j, d->con_j, (size_t)nc); UP(con, d->con, (size_t)nc);
    UP(cmap_off, d->cmap_off, N1 + 1); UP(cmap_j, d->cmap_j, (size_t)ncm); UP(cmap_bits, d->cmap_bits, (size_t)ncm);
    UP(pair, d->pair, (size_t)NT * NT);
    UP(hbpair, d->hbpair, (size_t)SDMD_NHBCLASS * NT * NT);
    UP(sd, d->step_d, (size_t)d->nstep_pool + 1); UP(se, d->step_e, (size_t)d->nstep_pool + 1);
    UP(sacc, d->step_acc, (size_t)d->nstep_pool + 1);
    UP(node, (const int *)nullptr, 2 * N1);
    UP(leaf, (const int *)nullptr, N1 + 1);
    S->win = (o && o->window > 0) ? o->window : MAXC;
    {
        // the constraint entry of each connection row entry (the first of
        // its partner, as FindPair finds it)
        int *cc = (int *)malloc(sizeof(int) * (size_t)(ncm > 0 ? ncm : 1));
        if (!cc) return SDMD_ENOMEM;
        for (int a = 1; a <= N; a++)
            for (int k = d->cmap_off[a]; k < d->cmap_off[a + 1]; k++) {
                cc[k] = -1;
                if (!(d->cmap_bits[k] & SDMD_CONSTRAINT_CONNECT)) continue;
                for (int q = d->con_off[a]; q < d->con_off[a + 1]; q++)
                    if (d->con_j[q] == d->cmap_j[k]) { cc[k] = q; break; }
            }
        UP(cmap_con, (const int *)cc, (size_t)ncm);
        free(cc);
    }
    if (!o || o->mode == SDMD_MODE_PLAIN) {
        // the plain engine's derived tables: cell arrays (filled by k_cells),
        // pops each atom has taken, the collision table with RightPair resolved (ToolFunctions.c:278-292)
        const size_t ncell = (size_t)d->cellnum[0] * d->cellnum[1] * d->cellnum[2];
        UP(ccnt, (const int *)nullptr, ncell + 1);
        UPBIG(cmem, (ncell + 1) * CELL_CAP);
        UP(lag, (const unsigned char *)nullptr, N1);
        UP(bulk_t2, (const double *)nullptr, N1);
        UP(bulk_head, (const int *)nullptr, N1); UP(bulk_next, (const int *)nullptr, N1);
        UP(bulk_flag, (const int *)nullptr, N1);
        UP(bulk_pot, (const double *)nullptr, N1); UP(bulk_pc, (const long long *)nullptr, N1);
        UP(bulk_sub, (const int *)nullptr, N1); UP(bulk_nbnum, (const int *)nullptr, N1);
        UP(bulk_hbit, (const int *)nullptr, N1);
        sdmd_pair rp[NT * NT];
        auto back = [](int t) { return t == 3 ? 1 : t == 4 ? 2 : t == 27 ? 26 : t; };
        int pool = 0, most = 0;
        for (int t1 = 0; t1 < NT; t1++)
            for (int t2 = 0; t2 < NT; t2++) {
                const int a = back(t1), b = back(t2);
                const int cand[4] = {t1 * NT + t2, a * NT + t2, t1 * NT + b, a * NT + b};
                sdmd_pair p = {0, 0, 0, 0};
                for (int q = 3; q >= 0; q--)
                    if (d->pair[cand[q]].dmin > 0) p = d->pair[cand[q]];
                rp[t1 * NT + t2] = p;
                pool = p.step0 + p.nstep > pool ? p.step0 + p.nstep : pool;
                most = p.nstep > most ? p.nstep : most;
            }
        UP(rpair, (const sdmd_pair *)rp, (size_t)NT * NT);
        S->ltab = (S->steps_sorted && pool > 0 && pool <= LPOOL && most <= 16) ? pool : 0;
        // a sweep of all atoms every logk pops: rare for large systems (its
        // memory traffic), frequent for small ones (an atom read late takes
        // the steps it lacks one by one, about 20 ns each)
        S->logk = N / 64 < 8 ? 8 : (N / 64 > LOGK ? LOGK : N / 64);
    }
    if (o && o->trace) {
        S->trace_cap = o->trace_capacity > 0 ? o->trace_capacity : 100000;
        UPBIG(trace, (size_t)S->trace_cap);
    }
    if (o && (o->profile & 1)) {
        UP(prof, (const unsigned long long *)nullptr, (size_t)PH_NPH);
    }
    if (o && o->hash_every > 0) {
        S->hash_every = o->hash_every;
        S->hash_cap = (o->trace_capacity > 0 ? o->trace_capacity : 1000000) / o->hash_every + 1;
        UPBIG(hashes, (size_t)S->hash_cap * 2);
    }
#undef UP
#undef UPBIG
    if ((rc = arena_commit(c, ar))) return rc;
    c->dyn[s].dev = (char *)S->x;
    if (!o || o->mode == SDMD_MODE_PLAIN) atom_gather_table(S);
    return SDMD_OK;
}

// One system's block of changing arrays into c->hostbuf (on the context's
// stream, waited for), and from there into the caller's arrays.
int sdmd_dyn_download(sdmd_gpu_ctx *c, int s) {
    if (!c->hostbuf) {
        size_t most = 0;
        for (int k = 0; k < c->nsys; k++) most = c->dyn[k].bytes > most ? c->dyn[k].bytes : most;
        if (hipHostMalloc((void **)&c->hostbuf, most, hipHostMallocDefault) != hipSuccess) {
            c->hostbuf = nullptr;
            return SDMD_EDEVICE;
        }
        c->hostbuf_bytes = most;
    }
    int rc = hip_ok(hipMemcpyAsync(c->hostbuf, c->dyn[s].dev, c->dyn[s].bytes, hipMemcpyDeviceToHost, c->stream));
    return rc ? rc : hip_ok(hipStreamSynchronize(c->stream));
}

void sdmd_dyn_scatter(const sdmd_gpu_ctx *c, int s, sdmd_system_desc *d) {
    const Sys &S = c->host_sys[s];
    const size_t N1 = (size_t)S.N + 1;
    auto get = [&](void *dst, const void *dev, size_t bytes) {
        if (dst) memcpy(dst, c->hostbuf + ((const char *)dev - c->dyn[s].dev), bytes);
    };
#define DOWN(dst, src, n) get(dst, src, sizeof(*(src)) * (n))
    DOWN(d->x, S.x, N1); DOWN(d->y, S.y, N1); DOWN(d->z, S.z, N1);
    DOWN(d->vx, S.vx, N1); DOWN(d->vy, S.vy, N1); DOWN(d->vz, S.vz, N1);
    DOWN(d->type, S.type, N1);
    DOWN(d->cellx, S.cx, N1); DOWN(d->celly, S.cy, N1); DOWN(d->cellz, S.cz, N1);
    DOWN(d->hb_bond, S.hbbond, N1); DOWN(d->hb_itype, S.hbitype, N1);
    DOWN(d->nb_partner, S.nbp, N1 * SDMD_NBSLOTS); DOWN(d->nb_partnernum, S.nbnum, N1); DOWN(d->nb_status, S.nbstat, N1);
    DOWN(d->dyn_j, S.dynj, N1 * SDMD_DYNSLOTS); DOWN(d->dyn_bits, S.dynb, N1 * SDMD_DYNSLOTS);
    DOWN(d->ev_partner, S.evp, N1); DOWN(d->ev_type, S.evtype, N1); DOWN(d->ev_sub, S.evsub, N1);
    DOWN(d->ev_counter, S.evc, N1); DOWN(d->ev_pcounter, S.evpc, N1);
    DOWN(d->ev_time, S.evt, N1); DOWN(d->ev_pot, S.evpot, N1);
    DOWN(d->celllist, S.celllist, (size_t)S.ncelllist);
#undef DOWN
}

static int sync_to_device(sdmd_gpu_ctx *c) {
    return hip_ok(hipMemcpyAsync(c->dev_sys, c->host_sys, sizeof(Sys) * c->nsys, hipMemcpyHostToDevice, c->stream));
}

static int sync_from_device(sdmd_gpu_ctx *c) {
    if (c->mode == SDMD_MODE_FAST) return sdmd_fast_sync(c);
    if (hipMemcpyAsync(c->host_sys, c->dev_sys, sizeof(Sys) * c->nsys, hipMemcpyDeviceToHost, c->stream) != hipSuccess)
        return SDMD_EDEVICE;
    return hip_ok(hipStreamSynchronize(c->stream));
}

static int resolve_scratch(int dev, double **out);

extern "C" int sdmd_gpu_open(const sdmd_system_desc *const *systems, int32_t nsys, const sdmd_gpu_opts *opts,
                             sdmd_gpu_ctx **out) {
    if (!systems || nsys <= 0 || !out) return SDMD_EINVAL;
    int block = (opts && opts->block) ? opts->block : 256;
    if (block != 64 && block != 128 && block != 256 && block != 512 && block != 1024) return SDMD_EINVAL;
    const int mode = opts ? opts->mode : SDMD_MODE_PLAIN;
    if (mode != SDMD_MODE_PLAIN && mode != SDMD_MODE_FAST) return SDMD_EUNSUPPORTED;
    if (mode == SDMD_MODE_FAST && block == 128) return SDMD_EINVAL;
    if (opts && (opts->window < 0 || opts->window > MAXC)) return SDMD_EINVAL;
    for (int s = 0; s < nsys; s++) {
        const sdmd_system_desc *d = systems[s];
        if (!d || d->natom < 2) return SDMD_EINVAL;
        if (d->cellnum[0] < 3 || d->cellnum[1] < 3 || d->cellnum[2] < 3) return SDMD_EINVAL;
        long ncell = (long)d->cellnum[0] * d->cellnum[1] * d->cellnum[2];
        if (d->ncelllist != d->natom + ncell + 1) return SDMD_EINVAL;
    }
    int dev_count = 0;
    if (hipGetDeviceCount(&dev_count) != hipSuccess || dev_count == 0) return SDMD_EDEVICE;
    sdmd_gpu_ctx *c = (sdmd_gpu_ctx *)calloc(1, sizeof *c);
    c->nsys = nsys;
    c->block = block;
    c->mode = mode;
    // an event loop's workgroup fills a CU's LDS (130 KB of tables and
    // candidates): with more systems than CUs a small one leaves the other
    // SIMDs idle while systems wait (400 pops of 512 systems of 59 atoms: 64
    // threads 15.3 ms, 256 threads 10.4 ms)
    int cus = 0, at = 0;
    if (hipGetDevice(&at) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, at) != hipSuccess)
        cus = 0;
    c->run_block = (cus > 0 && nsys > cus && block < 256) ? 256 : block;
    if (hipStreamCreate(&c->stream) != hipSuccess) { free(c); return SDMD_EDEVICE; }
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || resolve_scratch(dev, &c->scratch) != SDMD_OK) {
        HIPV(hipStreamDestroy(c->stream));
        free(c);
        return SDMD_EDEVICE;
    }
    HIPV(hipEventCreate(&c->ev0));
    HIPV(hipEventCreate(&c->ev1));
    c->host_sys = (Sys *)calloc((size_t)nsys, sizeof(Sys));
    c->desc = (const sdmd_system_desc **)calloc((size_t)nsys, sizeof(void *));
    c->dyn = (sdmd_dyn_block *)calloc((size_t)nsys, sizeof(sdmd_dyn_block));
    int rc = (c->host_sys && c->desc && c->dyn) ? SDMD_OK : SDMD_ENOMEM;
    if (rc == SDMD_OK)
        rc = hip_ok(hipHostMalloc((void **)&c->status, sizeof *c->status, hipHostMallocCoherent));
    sdmd_arena ar = {};
    for (int s = 0; s < nsys && rc == SDMD_OK; s++) {
        c->desc[s] = systems[s];
        rc = upload_system(c, &ar, s, systems[s], opts);
    }
    if (rc == SDMD_OK) rc = dev_upload(c, &c->dev_sys, (const Sys *)nullptr, (size_t)nsys);
    if (rc == SDMD_OK) {
        // energy workgroups per system: about 2048 in all (8 per CU), each
        // with an atom per wavefront at least
        int maxn = 1;
        for (int s = 0; s < nsys; s++) maxn = systems[s]->natom > maxn ? systems[s]->natom : maxn;
        const int want = (maxn + EWAVES - 1) / EWAVES, fit = (2048 + nsys - 1) / nsys;
        c->echunks = want < fit ? want : fit;
        rc = dev_upload(c, &c->epart, (const double *)nullptr, (size_t)ENERGY_PART * nsys * c->echunks);
    }
    if (rc == SDMD_OK) rc = sync_to_device(c);
    if (rc == SDMD_OK && mode == SDMD_MODE_PLAIN) {
        hipLaunchKernelGGL(k_cells, dim3(nsys, 64), dim3(256), 0, c->stream, c->dev_sys);
        rc = hip_ok(hipGetLastError());
    }
    if (rc == SDMD_OK) rc = hip_ok(hipStreamSynchronize(c->stream));
    if (rc == SDMD_OK && mode == SDMD_MODE_FAST) rc = sdmd_fast_open(c, opts);
    if (rc != SDMD_OK) { sdmd_gpu_close(c); return rc; }
    *out = c;
    return SDMD_OK;
}

extern "C" int sdmd_gpu_close(sdmd_gpu_ctx *c) {
    if (!c) return SDMD_EINVAL;
    if (c->stream) HIPV(hipStreamSynchronize(c->stream));
    for (int k = 0; k < c->nalloc; k++) HIPV(hipFree(c->allocs[k]));
    if (c->status) HIPV(hipHostFree(c->status));
    if (c->hostbuf) HIPV(hipHostFree(c->hostbuf));
    free(c->allocs);
    if (c->ev0) HIPV(hipEventDestroy(c->ev0));
    if (c->ev1) HIPV(hipEventDestroy(c->ev1));
    if (c->stream) HIPV(hipStreamDestroy(c->stream));
    sdmd_fast_close(c);
    free(c->host_sys);
    free(c->desc);
    free(c->dyn);
    free(c);
    return SDMD_OK;
}

extern "C" int sdmd_gpu_set_normals(sdmd_gpu_ctx *c, int32_t s, const double *z, int64_t n) {
    if (!c || s < 0 || s >= c->nsys || n < 0 || (n > 0 && !z)) return SDMD_EINVAL;
    int rc = sync_from_device(c);
    if (rc) return rc;
    Sys &S = c->host_sys[s];
    double *p = nullptr;
    if ((rc = dev_upload(c, &p, z, (size_t)n))) return rc;
    S.zn = p;
    S.nz = n;
    S.zpos = 0;
    rc = sync_to_device(c);
    return rc ? rc : hip_ok(hipStreamSynchronize(c->stream));
}

// A workgroup of k_bulk_predict fills a CU's LDS and predicts two atoms at a
// time: all CUs get an equal share of the atoms, in pieces of at most 32 (a
// piece costs its set-up, 54 KB of tables, about one pair of atoms), so that
// uneven systems balance.
static void launch_prepare(sdmd_gpu_ctx *c) {
    int maxn = 1;
    long long atoms = 0;
    for (int s = 0; s < c->nsys; s++) {
        maxn = c->host_sys[s].N > maxn ? c->host_sys[s].N : maxn;
        atoms += c->host_sys[s].N;
    }
    int per = 2;
    while (per < 32 && atoms > 256LL * per) per += 2;
    while ((maxn + per - 1) / per > 65535) per *= 2;   // a grid's y dimension ends at 65 536 (2.1 million atoms)
    const dim3 gp(c->nsys, (maxn + per - 1) / per), ga(c->nsys, maxn < 64 * 256 ? (maxn + 255) / 256 : 64);
    hipLaunchKernelGGL(k_bulk_reset, ga, dim3(256), 0, c->stream, c->dev_sys);
    hipLaunchKernelGGL((k_bulk_predict<256>), gp, dim3(256), 0, c->stream, c->dev_sys, per);
    hipLaunchKernelGGL(k_bulk_link, ga, dim3(256), 0, c->stream, c->dev_sys);
    hipLaunchKernelGGL(k_bulk_resolve, ga, dim3(256), 0, c->stream, c->dev_sys);
    hipLaunchKernelGGL((k_bulk_finish<512>), dim3(c->nsys), dim3(512), 0, c->stream, c->dev_sys);
}
template <int B>
static void launch_run(sdmd_gpu_ctx *c, long long n, long long budget, double t_end, double t_out) {
    const PlainRun r = {c->stream, c->dev_sys, c->nsys, n, budget, t_end, t_out};
    if (c->host_sys[0].prof) plain_launch_run<B, true>(r);
    else plain_launch_run<B, false>(r);
}
template <int B>
static void launch_op(sdmd_gpu_ctx *c, int s, int op, Renew renew, int a, int b) {
    hipLaunchKernelGGL((k_op<B>), dim3(1), dim3(B), 0, c->stream, c->dev_sys, s, op, renew, a, b, c->status);
}

#define DISPATCH(block, fn, ...) do { switch (block) { \
    case 64: fn<64>(__VA_ARGS__); break; case 128: fn<128>(__VA_ARGS__); break; \
    case 256: fn<256>(__VA_ARGS__); break; case 512: fn<512>(__VA_ARGS__); break; \
    default: fn<1024>(__VA_ARGS__); break; } } while (0)

static int check_errors(sdmd_gpu_ctx *c) {
    int rc = sync_from_device(c);
    if (rc) return rc;
    for (int s = 0; s < c->nsys; s++)
        if (c->host_sys[s].error) return SDMD_ESTATE;
    return SDMD_OK;
}

extern "C" int sdmd_gpu_prepare(sdmd_gpu_ctx *c) {
    if (!c) return SDMD_EINVAL;
    if (c->mode == SDMD_MODE_FAST) return sdmd_fast_prepare(c);
    HIPV(hipEventRecord(c->ev0, c->stream));
    launch_prepare(c);
    HIPV(hipEventRecord(c->ev1, c->stream));
    if (hipGetLastError() != hipSuccess) return SDMD_EDEVICE;
    if (hipStreamSynchronize(c->stream) != hipSuccess) return SDMD_EDEVICE;
    float ms = 0;
    HIPV(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    return check_errors(c);
}

static int run_bounded(sdmd_gpu_ctx *c, int64_t pops, double max_ms, double t_end, double t_out = INFINITY);

extern "C" int sdmd_gpu_run(sdmd_gpu_ctx *c, int64_t pops) {
    return pops < 0 ? SDMD_EINVAL : run_bounded(c, pops, 0, INFINIT);
}

extern "C" int sdmd_gpu_run_for(sdmd_gpu_ctx *c, int64_t pops, double max_ms) {
    return pops < 0 ? SDMD_EINVAL : run_bounded(c, pops, max_ms, INFINIT);
}

extern "C" int sdmd_gpu_run_until(sdmd_gpu_ctx *c, double t_end, int64_t max_pops) {
    return max_pops < 0 ? SDMD_EINVAL : run_bounded(c, max_pops, 0, t_end);
}

extern "C" int sdmd_gpu_run_to_output(sdmd_gpu_ctx *c, double t_out, double t_end, int64_t max_pops) {
    if (!c || max_pops < 0) return SDMD_EINVAL;
    if (c->mode != SDMD_MODE_PLAIN) return SDMD_EUNSUPPORTED;
    return run_bounded(c, max_pops, 0, t_end, t_out);
}

extern "C" int sdmd_gpu_run_events(sdmd_gpu_ctx *c, int64_t events, double max_ms) {
    if (!c || events <= 0) return SDMD_EINVAL;
    return run_bounded(c, -events, max_ms, INFINIT);
}

// pops >= 0: pops per system; pops < 0: -pops executed events per system
static int run_bounded(sdmd_gpu_ctx *c, int64_t pops, double max_ms, double t_end, double t_out) {
    if (!c) return SDMD_EINVAL;
    if (c->mode == SDMD_MODE_FAST) return sdmd_fast_run(c, pops, max_ms, t_end);
    long long budget = 1LL << 62;
    if (max_ms > 0) {
        int dev = 0, khz = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0)
            return SDMD_EDEVICE;
        budget = (long long)(max_ms * khz);
    }
    HIPV(hipEventRecord(c->ev0, c->stream));
    DISPATCH(c->run_block, launch_run, c, (long long)pops, budget, t_end, t_out);
    HIPV(hipEventRecord(c->ev1, c->stream));
    if (hipGetLastError() != hipSuccess) return SDMD_EDEVICE;
    if (hipStreamSynchronize(c->stream) != hipSuccess) return SDMD_EDEVICE;
    float ms = 0;
    HIPV(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    return check_errors(c);
}

// After a single operation: its launch, its end and, from the pinned status
// word, its error; errors other systems carry from earlier calls are known on
// the host (every run and prepare copies them back).  One wait per call: the
// struct copy and second wait of a run cost as much as the operation.
static int op_result(sdmd_gpu_ctx *c, int s) {
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(c->stream) != hipSuccess) return SDMD_EDEVICE;
    c->host_sys[s].error = c->status->error;
    for (int k = 0; k < c->nsys; k++)
        if (c->host_sys[k].error) return SDMD_ESTATE;
    return SDMD_OK;
}

static int run_op(sdmd_gpu_ctx *c, int s, int op, const int32_t *renew, int a, int b) {
    if (!c || s < 0 || s >= c->nsys) return SDMD_EINVAL;
    if (c->mode != SDMD_MODE_PLAIN) return SDMD_EUNSUPPORTED;
    Renew list = {};
    if (renew) {
        const int n = renew[0];
        if (n < 0 || n > 2) return SDMD_EINVAL;
        for (int k = 0; k <= n; k++) list.a[k] = renew[k];
        for (int k = 1; k <= n; k++)
            if (list.a[k] < 1 || list.a[k] > c->host_sys[s].N) return SDMD_EINVAL;
    }
    DISPATCH(c->block, launch_op, c, s, op, list, a, b);
    return op_result(c, s);
}

extern "C" int sdmd_gpu_predict(sdmd_gpu_ctx *c, int32_t s, const int32_t *renew) {
    if (!renew) return SDMD_EINVAL;
    return run_op(c, s, OP_PREDICT, renew, 0, 0);
}
extern "C" int sdmd_gpu_create_tree(sdmd_gpu_ctx *c, int32_t s) { return run_op(c, s, OP_CREATE_TREE, nullptr, 0, 0); }
extern "C" int sdmd_gpu_update_tree(sdmd_gpu_ctx *c, int32_t s, const int32_t *renew) {
    if (!renew) return SDMD_EINVAL;
    return run_op(c, s, OP_UPDATE_TREE, renew, 0, 0);
}
extern "C" int sdmd_gpu_advance(sdmd_gpu_ctx *c, int32_t s, double dt) {
    if (!c || s < 0 || s >= c->nsys) return SDMD_EINVAL;
    if (c->mode != SDMD_MODE_PLAIN) return SDMD_EUNSUPPORTED;
    const int blocks = (c->host_sys[s].N + 255) / 256;
    hipLaunchKernelGGL(k_advance, dim3(blocks < 1024 ? blocks : 1024), dim3(256), 0, c->stream, c->dev_sys, s, dt, c->status);
    return op_result(c, s);
}
extern "C" int sdmd_gpu_do_event(sdmd_gpu_ctx *c, int32_t s, int32_t t, int32_t p) {
    if (!c || s < 0 || s >= c->nsys || t < 1 || t > c->host_sys[s].N || p < 0 || p > c->host_sys[s].N) return SDMD_EINVAL;
    return run_op(c, s, OP_DO_EVENT, nullptr, t, p);
}
extern "C" int sdmd_gpu_cell_move(sdmd_gpu_ctx *c, int32_t s, int32_t a) {
    if (!c || s < 0 || s >= c->nsys || a < 1 || a > c->host_sys[s].N) return SDMD_EINVAL;
    return run_op(c, s, OP_CELL_MOVE, nullptr, a, 0);
}

extern "C" int sdmd_gpu_pop(sdmd_gpu_ctx *c, int32_t s, sdmd_gpu_event *out) {
    if (!c || s < 0 || s >= c->nsys || !out) return SDMD_EINVAL;
    if (c->mode != SDMD_MODE_PLAIN) return SDMD_EUNSUPPORTED;
    hipLaunchKernelGGL(k_pop, dim3(1), dim3(64), 0, c->stream, c->dev_sys, s, c->status);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(c->stream) != hipSuccess) return SDMD_EDEVICE;
    if (c->status->ev.target == 0) return SDMD_ESTATE;
    *out = c->status->ev;
    return SDMD_OK;
}

extern "C" int sdmd_gpu_download(sdmd_gpu_ctx *c, int32_t s, sdmd_system_desc *d) {
    if (!c || s < 0 || s >= c->nsys || !d) return SDMD_EINVAL;
    if (c->mode == SDMD_MODE_FAST) {
        if (d->natom != c->host_sys[s].N) return SDMD_EINVAL;
        return sdmd_fast_download(c, s, d);
    }
    int rc = sync_from_device(c);
    if (rc) return rc;
    const Sys &S = c->host_sys[s];
    if (d->natom != S.N) return SDMD_EINVAL;
    if ((rc = sdmd_dyn_download(c, s))) return rc;
    sdmd_dyn_scatter(c, s, d);
    d->currenttime = S.currenttime;
    return SDMD_OK;
}

extern "C" int sdmd_gpu_set_tree(sdmd_gpu_ctx *c, int32_t s, const int32_t *node, const int32_t *leaf) {
    if (!c || s < 0 || s >= c->nsys || !node || !leaf) return SDMD_EINVAL;
    if (c->mode != SDMD_MODE_PLAIN) return SDMD_EUNSUPPORTED;
    const int N = c->host_sys[s].N;
    for (int a = 1; a <= N; a++)                       // every atom's leaf holds it
        if (leaf[a] < 1 || leaf[a] >= 2 * N || node[leaf[a]] != a) return SDMD_EINVAL;
    int rc = sync_from_device(c);
    if (rc) return rc;
    Sys &S = c->host_sys[s];
    S.count = N;                                       // every atom inserted (CreateCBT's state)
    if (hipMemcpy(S.node, node, sizeof(int) * 2 * (size_t)N, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(S.leaf, leaf, sizeof(int) * ((size_t)N + 1), hipMemcpyHostToDevice) != hipSuccess)
        return SDMD_EDEVICE;
    rc = sync_to_device(c);
    return rc ? rc : hip_ok(hipStreamSynchronize(c->stream));
}

extern "C" int sdmd_gpu_get_tree(sdmd_gpu_ctx *c, int32_t s, int32_t *node, int32_t *leaf) {
    if (!c || s < 0 || s >= c->nsys) return SDMD_EINVAL;
    if (c->mode != SDMD_MODE_PLAIN) return SDMD_EUNSUPPORTED;
    const Sys &S = c->host_sys[s];
    if (node && hipMemcpy(node, S.node, sizeof(int) * 2 * (size_t)S.N, hipMemcpyDeviceToHost) != hipSuccess) return SDMD_EDEVICE;
    if (leaf && hipMemcpy(leaf, S.leaf, sizeof(int) * ((size_t)S.N + 1), hipMemcpyDeviceToHost) != hipSuccess) return SDMD_EDEVICE;
    return SDMD_OK;
}

extern "C" int sdmd_gpu_stats_get(sdmd_gpu_ctx *c, int32_t s, sdmd_gpu_stats *out) {
    if (!c || s < 0 || s >= c->nsys || !out) return SDMD_EINVAL;
    int rc = sync_from_device(c);
    if (rc) return rc;
    const Sys &S = c->host_sys[s];
    memset(out, 0, sizeof *out);
    out->pops = S.pops; out->frame = S.frame; out->recal = S.recal;
    for (int k = 0; k < 16; k++) out->per_type[k] = S.per_type[k];
    out->pair_evals = S.pair_evals; out->candidates = S.candidates;
    out->normals_used = S.zpos;
    out->currenttime = S.currenttime;
    out->error = S.error;
    out->last_exec = S.last_exec;
    return SDMD_OK;
}

extern "C" int sdmd_gpu_get_trace(sdmd_gpu_ctx *c, int32_t s, sdmd_gpu_pop_rec *out, int64_t max, int64_t *n) {
    if (!c || s < 0 || s >= c->nsys || !n) return SDMD_EINVAL;
    if (c->mode != SDMD_MODE_PLAIN) return SDMD_EUNSUPPORTED;
    int rc = sync_from_device(c);
    if (rc) return rc;
    const Sys &S = c->host_sys[s];
    int64_t k = S.trace_n < max ? S.trace_n : max;
    if (k > 0 && out && hipMemcpy(out, S.trace, sizeof(sdmd_gpu_pop_rec) * (size_t)k, hipMemcpyDeviceToHost) != hipSuccess)
        return SDMD_EDEVICE;
    *n = k;
    return SDMD_OK;
}

extern "C" int sdmd_gpu_get_hashes(sdmd_gpu_ctx *c, int32_t s, int64_t *out, int64_t max, int64_t *n) {
    if (!c || s < 0 || s >= c->nsys || !n) return SDMD_EINVAL;
    if (c->mode != SDMD_MODE_PLAIN) return SDMD_EUNSUPPORTED;
    int rc = sync_from_device(c);
    if (rc) return rc;
    const Sys &S = c->host_sys[s];
    int64_t k = S.hash_n < max ? S.hash_n : max;
    if (k > 0 && out && hipMemcpy(out, S.hashes, sizeof(int64_t) * 2 * (size_t)k, hipMemcpyDeviceToHost) != hipSuccess)
        return SDMD_EDEVICE;
    *n = k;
    return SDMD_OK;
}

// per-phase device time (seconds) of system s when opened with profiling on
extern "C" int sdmd_gpu_phase_times(sdmd_gpu_ctx *c, int32_t s, double *out, int32_t n) {
    if (!c || s < 0 || s >= c->nsys || !out) return SDMD_EINVAL;
    const Sys &S = c->host_sys[s];
    if (!S.prof) return SDMD_ESTATE;
    unsigned long long v[PH_NPH];
    if (hipMemcpy(v, S.prof, sizeof v, hipMemcpyDeviceToHost) != hipSuccess) return SDMD_EDEVICE;
    int dev = 0, khz = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0)
        return SDMD_EDEVICE;
    for (int k = 0; k < n && k < PH_NPH; k++) out[k] = (double)v[k] / (1e3 * khz);
    return SDMD_OK;
}

extern "C" int sdmd_gpu_last_kernel_ms(sdmd_gpu_ctx *c, double *ms) {
    if (!c || !ms) return SDMD_EINVAL;
    *ms = c->last_ms;
    return SDMD_OK;
}

// Energy kernels of the context's mode into `planes` (3 x nsys doubles:
// kinetic, potential, error flag), then the planes into the caller's arrays.
// No allocation: the error plane is read back through a stack buffer.
static int energy_launch(sdmd_gpu_ctx *c, double *planes) {
    if (c->mode == SDMD_MODE_FAST) return sdmd_fast_energy_launch(c, planes);
    hipLaunchKernelGGL(k_energy, dim3(c->nsys, c->echunks), dim3(64 * EWAVES), 0, c->stream, c->dev_sys, c->epart);
    hipLaunchKernelGGL(k_energy_reduce, dim3(c->nsys), dim3(64), 0, c->stream, c->epart, c->echunks, planes);
    return hip_ok(hipGetLastError());
}

static int energy_planes_to_host(sdmd_gpu_ctx *c, const double *planes, double *kinetic, double *potential) {
    const size_t n = (size_t)c->nsys;
    int rc = hip_ok(hipMemcpyAsync(kinetic, planes, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
    if (!rc) rc = hip_ok(hipMemcpyAsync(potential, planes + n, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
    int bad = 0;
    for (size_t s0 = 0; !rc && s0 < n; s0 += 64) {
        double flags[64];
        const size_t m = n - s0 < 64 ? n - s0 : 64;
        rc = hip_ok(hipMemcpyAsync(flags, planes + 2 * n + s0, sizeof(double) * m, hipMemcpyDeviceToHost, c->stream));
        if (!rc) rc = hip_ok(hipStreamSynchronize(c->stream));
        for (size_t k = 0; !rc && k < m; k++) bad |= flags[k] != 0;
    }
    if (!rc) rc = hip_ok(hipStreamSynchronize(c->stream));
    return rc ? rc : (bad ? SDMD_ESTATE : SDMD_OK);     // a table lookup failed or the system is in error
}

extern "C" int sdmd_gpu_energy(sdmd_gpu_ctx *c, double *kinetic, double *potential) {
    if (!c || !kinetic || !potential) return SDMD_EINVAL;
    int rc;
    if (!c->dev_energy && (rc = dev_upload(c, &c->dev_energy, (const double *)nullptr, (size_t)3 * c->nsys)))
        return rc;
    if ((rc = energy_launch(c, c->dev_energy))) return rc;
    return energy_planes_to_host(c, c->dev_energy, kinetic, potential);
}

// ---------------------------------------------------------------- replica exchange on the device
// The REMD server's exchange pass (Server.c:145-192, restated on the host by
// sdmd_remd_rearrange) run by one device thread between event windows, on
// the energies the energy kernel left in its planes, with the server's
// rand() stream (glibc TYPE_3, as sdmd_rand_next) kept in device memory;
// each replica's thermostat temperature is then written where the event
// loop reads it.  The pass is sequential by definition (later replicas see
// earlier swaps, draws happen in order), so one thread runs it.
__device__ int32_t remd_rand_next(sdmd_rand_state &st) {
    const uint32_t v = (uint32_t)st.r[st.f] + (uint32_t)st.r[st.b];
    st.r[st.f] = (int32_t)v;
    if (++st.f >= 31) st.f = 0;
    if (++st.b >= 31) st.b = 0;
    st.calls++;
    return (int32_t)(v >> 1);
}

__global__ void k_remd_exchange(const double *planes, int n, sdmd_remd_temp *T, sdmd_rand_state *rng,
                                long long *counts, double *const *tptr, sdmd_remd_temp *hist, double *ehist,
                                int *err) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const double *epot = planes + n;                 // the potential plane
    for (int k = 0; k < n; k++)
        if (planes[2 * n + k] != 0) *err = 1;         // an energy kernel error: no exchange
    if (*err) return;
    sdmd_rand_state st = *rng;
    for (int i = 0; i < n; i++) {
        if (!T[i].T) continue;
        for (int j = 0; j < n; j++) {
            if (!T[j].T) continue;
            if (T[i].num == T[j].num + 1 || (T[i].num == 1 && T[j].num == 2)) {
                const double beta1 = 1 / T[i].T, beta2 = 1 / T[j].T;
                const double dE = (beta1 - beta2) * (epot[j] - epot[i]);
                const int lo = T[i].num < T[j].num ? T[i].num : T[j].num;
                if (lo >= 1 && lo <= n) counts[2 * (lo - 1)]++;
                bool swap = dE <= 0.0;
                if (!swap) {
                    const double u = 0 + (double)remd_rand_next(st) / ((double)2147483647 / (1 - 0));   // RANDOMVALUE(0, 1)
                    swap = u < exp(-1 * dE);
                }
                if (swap) {
                    const sdmd_remd_temp z = T[i];
                    T[i] = T[j];
                    T[j] = z;
                    if (lo >= 1 && lo <= n) counts[2 * (lo - 1) + 1]++;
                }
                break;
            }
        }
    }
    *rng = st;
    for (int k = 0; k < n; k++) {
        *tptr[k] = T[k].T;                             // targetTemperature = REMD_Temperature.T, REMD.c:100
        if (hist) hist[k] = T[k];
        if (ehist) ehist[k] = epot[k];
    }
}

extern "C" int sdmd_remd_run(sdmd_gpu_ctx *c, sdmd_remd_temp *temps, sdmd_rand_state *rng, int64_t *counts,
                             int32_t cycles, int64_t interval, sdmd_remd_temp *history, double *epot_history) {
    if (!c || !temps || !rng || cycles < 1 || interval < 1) return SDMD_EINVAL;
    const int n = c->nsys;
    for (int k = 0; k < n; k++)
        if (!(temps[k].T >= 0)) return SDMD_EINVAL;
    int rc;
    if (!c->dev_energy && (rc = dev_upload(c, &c->dev_energy, (const double *)nullptr, (size_t)3 * n))) return rc;
    // device copies for this call (freed at its end)
    sdmd_remd_temp *dT = nullptr, *dH = nullptr;
    sdmd_rand_state *dR = nullptr;
    long long *dC = nullptr;
    double **dP = nullptr, *dE = nullptr;
    int *dErr = nullptr;
    double **tp = (double **)malloc(sizeof(double *) * n);
    if (!tp) return SDMD_ENOMEM;
    for (int k = 0; k < n; k++) tp[k] = c->mode == SDMD_MODE_FAST ? sdmd_fast_temperature_addr(c, k) : &c->dev_sys[k].T;
    rc = SDMD_OK;
    const size_t hn = (size_t)cycles * n;
    if (hipMalloc(&dT, sizeof(sdmd_remd_temp) * n) != hipSuccess || hipMalloc(&dR, sizeof(sdmd_rand_state)) != hipSuccess ||
        hipMalloc(&dC, sizeof(long long) * 2 * n) != hipSuccess || hipMalloc(&dP, sizeof(double *) * n) != hipSuccess ||
        hipMalloc(&dErr, sizeof(int)) != hipSuccess ||
        (history && hipMalloc(&dH, sizeof(sdmd_remd_temp) * hn) != hipSuccess) ||
        (epot_history && hipMalloc(&dE, sizeof(double) * hn) != hipSuccess))
        rc = SDMD_EDEVICE;
    long long *zero = (long long *)calloc((size_t)2 * n, sizeof(long long));
    if (!rc && !zero) rc = SDMD_ENOMEM;
    if (!rc) rc = hip_ok(hipMemcpy(dT, temps, sizeof(sdmd_remd_temp) * n, hipMemcpyHostToDevice));
    if (!rc) rc = hip_ok(hipMemcpy(dR, rng, sizeof(sdmd_rand_state), hipMemcpyHostToDevice));
    if (!rc) rc = hip_ok(hipMemcpy(dC, counts ? (const void *)counts : (const void *)zero, sizeof(long long) * 2 * n,
                                   hipMemcpyHostToDevice));
    if (!rc) rc = hip_ok(hipMemcpy(dP, tp, sizeof(double *) * n, hipMemcpyHostToDevice));
    if (!rc) rc = hip_ok(hipMemset(dErr, 0, sizeof(int)));
    // the temperatures the table holds now, before the first window
    if (!rc) {
        for (int k = 0; k < n && !rc; k++)
            rc = hip_ok(hipMemcpy(tp[k], &temps[k].T, sizeof(double), hipMemcpyHostToDevice));
    }
    if (!rc && c->mode == SDMD_MODE_PLAIN) rc = sync_from_device(c);    // host mirror of the plain systems
    for (int cy = 0; cy < cycles && !rc; cy++) {
        if (c->mode == SDMD_MODE_FAST) rc = sdmd_fast_launch_events(c, interval);
        else {
            DISPATCH(c->run_block, launch_run, c, (long long)-interval, 1LL << 62, INFINIT, INFINITY);
            rc = hip_ok(hipGetLastError());
        }
        if (!rc) rc = energy_launch(c, c->dev_energy);
        if (!rc) {
            hipLaunchKernelGGL(k_remd_exchange, dim3(1), dim3(64), 0, c->stream, c->dev_energy, n, dT, dR, dC, dP,
                               dH ? dH + (size_t)cy * n : nullptr, dE ? dE + (size_t)cy * n : nullptr, dErr);
            rc = hip_ok(hipGetLastError());
        }
    }
    if (!rc) rc = hip_ok(hipStreamSynchronize(c->stream));
    int herr = 0;
    if (!rc) rc = hip_ok(hipMemcpy(&herr, dErr, sizeof(int), hipMemcpyDeviceToHost));
    if (!rc) rc = hip_ok(hipMemcpy(temps, dT, sizeof(sdmd_remd_temp) * n, hipMemcpyDeviceToHost));
    if (!rc) rc = hip_ok(hipMemcpy(rng, dR, sizeof(sdmd_rand_state), hipMemcpyDeviceToHost));
    if (!rc && counts) rc = hip_ok(hipMemcpy(counts, dC, sizeof(long long) * 2 * n, hipMemcpyDeviceToHost));
    if (!rc && history) rc = hip_ok(hipMemcpy(history, dH, sizeof(sdmd_remd_temp) * hn, hipMemcpyDeviceToHost));
    if (!rc && epot_history) rc = hip_ok(hipMemcpy(epot_history, dE, sizeof(double) * hn, hipMemcpyDeviceToHost));
    if (!rc) rc = c->mode == SDMD_MODE_FAST ? sdmd_fast_sync(c) : check_errors(c);
    if (!rc && c->mode == SDMD_MODE_FAST)
        for (int k = 0; k < n && !rc; k++)
            if (c->host_sys[k].error) rc = SDMD_ESTATE;
    if (!rc && herr) rc = SDMD_ESTATE;
    HIPV(hipFree(dT)); HIPV(hipFree(dR)); HIPV(hipFree(dC)); HIPV(hipFree(dP)); HIPV(hipFree(dErr));
    if (dH) HIPV(hipFree(dH));
    if (dE) HIPV(hipFree(dE));
    free(tp);
    free(zero);
    return rc;
}

// ---------------------------------------------------------------- allocation-free energy
// Per-system partial results of sdmd_gpu_energy_noalloc (three planes of
// SDMD_NOALLOC_MAX_SYS doubles) in a file-scope device array: every GPU the
// library runs on holds one copy until the process ends.  The kernels write
// every entry they report, so nothing needs clearing between calls; calls
// that overlap on one GPU share the array and race.
static __device__ __align__(256) double scratch[3 * SDMD_NOALLOC_MAX_SYS];

// the array's device address on each GPU, resolved once per device by
// sdmd_gpu_open with that device current (host code never uses the
// array's name as an address)
constexpr int NOALLOC_MAXDEV = 64;
static double *g_scratch[NOALLOC_MAXDEV];
static std::mutex g_scratch_mu;

static int resolve_scratch(int dev, double **out) {
    if (dev < 0 || dev >= NOALLOC_MAXDEV) return SDMD_EDEVICE;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return SDMD_EDEVICE;
        g_scratch[dev] = (double *)p;
    }
    *out = g_scratch[dev];
    return SDMD_OK;
}

extern "C" int sdmd_gpu_energy_noalloc(sdmd_gpu_ctx *c, double *kinetic, double *potential) {
    if (!c || !kinetic || !potential) return SDMD_EINVAL;
    if (c->nsys > SDMD_NOALLOC_MAX_SYS) return SDMD_ERANGE;
    if (!c->scratch) return SDMD_EDEVICE;
    int rc = energy_launch(c, c->scratch);
    return rc ? rc : energy_planes_to_host(c, c->scratch, kinetic, potential);
}

extern "C" int sdmd_gpu_set_temperature(sdmd_gpu_ctx *c, int32_t s, double T) {
    if (!c || s < 0 || s >= c->nsys || !(T > 0)) return SDMD_EINVAL;
    if (c->mode == SDMD_MODE_FAST) return sdmd_fast_set_temperature(c, s, T);
    c->host_sys[s].T = T;
    int rc = hip_ok(hipMemcpyAsync(&c->dev_sys[s].T, &c->host_sys[s].T, sizeof(double), hipMemcpyHostToDevice,
                                   c->stream));
    return rc ? rc : hip_ok(hipStreamSynchronize(c->stream));
}

extern "C" int sdmd_gpu_fast_stats_get(sdmd_gpu_ctx *c, int32_t s, sdmd_gpu_fast_stats *out) {
    if (!c || s < 0 || s >= c->nsys || !out) return SDMD_EINVAL;
    if (c->mode != SDMD_MODE_FAST) return SDMD_EUNSUPPORTED;
    memset(out, 0, sizeof *out);
    return sdmd_fast_stats(c, s, out);
}

extern "C" int sdmd_gpu_autotune(sdmd_gpu_ctx *c, double trial_ms, int32_t *block_out, int32_t *depth_out) {
    if (!c || !(trial_ms > 0)) return SDMD_EINVAL;
    if (c->mode != SDMD_MODE_FAST) return SDMD_EUNSUPPORTED;
    return sdmd_fast_autotune(c, trial_ms, block_out, depth_out);
}

extern "C" int sdmd_gpu_run_graph(sdmd_gpu_ctx *c, int32_t launches, double max_ms) {
    if (!c || launches < 1 || !(max_ms > 0)) return SDMD_EINVAL;
    if (c->mode != SDMD_MODE_FAST) return SDMD_EUNSUPPORTED;
    return sdmd_fast_run_graph(c, launches, max_ms);
}
#endif  // SDMD_PLAIN_RUN
