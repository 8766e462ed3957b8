// sdmd_fast.hip - MI355X (gfx950) screened local-time event engine.
//
// The same event semantics as the reference (Predict, SGThread.c:158-211,
// with BondTime/CollisionTime/PBCandCrossCellTime/ThermostatTime/HBTime/
// HBNeighborTime of TimePrediction.c; DoEvent, Events.c:25-114) on a state
// that needs no O(N) sweep per event:
//
//   local time   every atom keeps (x0, v) valid at its own time t0; event
//                times are absolute, so popping an event touches only the
//                atoms it involves (UpdateData/TimeForward of
//                ToolFunctions.c:23-36 disappear)
//   cells        cell arrays (a count and 64 to 1 024 slots per cell, twice the
//                start's fullest cell) with an FP32 mirror record per slot: offset from the cell's
//                lower corner, time offset from a system epoch, velocity,
//                atom id and type
//   screen       pair times are screened in FP32 on the mirror (cell-relative
//                coordinates keep ~5e-7 A resolution); every candidate whose
//                shell, direction, discriminant or sign decision lies inside
//                its FP32 error band is marked, and the marked candidates
//                plus those whose time interval reaches the smallest upper
//                bound are re-solved in FP64 with the reference formulas;
//                the FP64 minimum is the prediction
//   batches      each round takes every pending event earlier than the
//                smallest third-earliest time of any 64-atom block (when that
//                set is too large, second-earliest, or in a run of a large
//                system up to a time those of a window of time), so the set is
//                exactly a prefix of the event order, and executes
//                concurrently every event whose atoms are at least
//                2 cells (3 when a cell crossing or an H-bond event is
//                involved) and two cell widths from the atoms of every
//                earlier event of the set: no event's re-predictions read
//                the other's atoms, and no event created by one can reach
//                the other's atoms through a single partner, so they
//                commute.  One lane executes one event; the re-predictions
//                are spread over the wavefronts.
//   tree         the per-block minimum, its atom and the block's second
//                minimum live in LDS; a round rescans only the blocks whose
//                atoms changed
//   thermostat   counter-based Philox4x32-10 normals keyed by (seed, system,
//                atom, per-atom draw count), so results do not depend on
//                the batch schedule
//
// FP64 is kept for the clock, the confirmed pair times, the grazing cases
// and the velocity updates (InteractionEvent, Events.c:798-1024).

#include <cstddef>

#include "sdmd_dev.h"

namespace sdmd {

typedef float fvec4 __attribute__((ext_vector_type(4)));   // mirror record half (16 B)

constexpr int FCAP_MIN = 64;      // slots per cell at least (a system's capacity: FSys.cap)
constexpr int FCAP_MAX = 1024;    // ... at most
constexpr int FMAXBLK = 1024;     // 64-atom blocks per system (N <= 65535)
constexpr int FSEL = 64;          // events considered per round
constexpr int FSEL_AIM = 54;      // ... aimed at where a window of time bounds the set
constexpr int FSMALL = 32;        // 64-atom blocks up to which one wavefront selects and executes a round
constexpr int FMAXW = 16;         // wavefronts per workgroup at most
constexpr long long FDRAIN = 1 << 20;   // bound on the pops of a closing drain
constexpr float FINF = 3.0e38f;

// FERR_CAUSAL: an atom was read at a local time later than the reader's
// (the independence rule failed); FERR_DRAIN: a closing drain reached its
// pop bound with events still pending up to the stop time, so the state is
// not a snapshot at one time
// FERR_JOBS: a round's re-predictions were not all completed within
// FJOB_WAIT ticks (the wait is bounded so the launch always ends)
enum { FERR_SELECT = 20, FERR_SLOT = 21, FERR_CAUSAL = 25,
       FERR_DRAIN = 26, FERR_JOBS = 27 };

// phases timed (by wavefront 0) when profiling is on
enum { FPH_SELECT, FPH_EXEC, FPH_STAGE, FPH_SCREEN, FPH_CONFIRM, FPH_OTHER, FPH_TREE, FPH_EVENT, FPH_BOND,
       FPH_SCAN, FPH_COLLECT };

// step radii (squared, FP32) of one constraint entry and bit k set when
// step k carries no energy
constexpr int PROW = 16;          // steps per collision pair at most

struct __attribute__((aligned(16))) ConRad {
    float rad[8];
    unsigned int ez;
    float dmin, dmax;
    int nstep;
};

struct FSys {
    Sys s;
    double *t0;                 // local time of (x, v)
    int *ccnt, *cmem, *slot;    // cell arrays: ccnt[cell], cmem[cell*cap+q], slot[atom]
    int cap;                    // slots per cell: a power of two, twice the start's fullest cell or more
    fvec4 *rec;                // FP32 mirror, two fvec4 per slot
    double *b1, *b2, *b3;       // block's earliest, second and third event times (persisted)
    int *ba, *bb;               // atoms of the earliest and second event
    unsigned int *rctr;         // per-atom draw counter
    // fixed-stride copies of the bond lists (16 slots per atom) and FP32
    // step radii inline with every constraint, so a prediction stages them
    // without a dependent load
    int *bj16;
    double *blo16, *bhi16;
    struct ConRad *crad;
    int *conn;                  // per atom FCONN bytes: its connection row (see FWave)
    int *rowlo;                 // the row's first column (-1: it does not fit its bytes)
    // FP64 shells at a fixed stride, read at a known shell without a
    // dependent load: dmin, dmax, the radii, the energies
    double *prow;               // [NT*NT][2 + 2 * PROW] by resolved collision pair
    double *crow;               // [constraint entry][2 + 2 * FCONSTEP]
    int ncell, nblk;
    float L32[3];
    float eb0, band0;           // the records' rounding in the screen's bands (see ScrBand)
    double Te, rebase_dt;
    double t_stop;              // events later than this stay pending (run_until)
    const void *scrtab;         // ScrTab (FP32 collision table), copied into LDS per launch
    unsigned int key0, key1;
    int validate, max_batch;
    // statistics
    long long batches, deferred, single, screens, confirms, validated, agree, rebases, causal;
    double max_screen_err, max_time_err, tlast;
};

// ---------------------------------------------------------------- fixed view
// (see fixed_view of Sys)
typedef const __attribute__((address_space(4))) FSys FV;
__device__ __forceinline__ FV &fixed_view(const FSys *p) { return *(FV *)p; }
// the same view, read anew: the compiler keeps nothing it read before across
// this point (a hundred values held over the whole event loop would be moved
// through vector registers, two instructions per use; a scalar load fetches
// sixteen words with one)
__device__ __forceinline__ FV &view_anew(FV &F) {
    FV *p = &F;
    asm volatile("" : "+s"(p));
    return *p;
}

// ---------------------------------------------------------------- RNG
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11), Box-Muller normal.
__device__ __forceinline__ void philox10(unsigned int c[4], unsigned int k0, unsigned int k1) {
#pragma unroll
    for (int r = 0; r < 10; r++) {
        const unsigned long long p0 = (unsigned long long)0xD2511F53u * c[0];
        const unsigned long long p1 = (unsigned long long)0xCD9E8D57u * c[2];
        const unsigned int n0 = (unsigned int)(p1 >> 32) ^ c[1] ^ k0;
        const unsigned int n2 = (unsigned int)(p0 >> 32) ^ c[3] ^ k1;
        c[0] = n0; c[1] = (unsigned int)p1; c[2] = n2; c[3] = (unsigned int)p0;
        k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
    }
}

// the four words of draw number `ctr` of atom a
template <class FS>
__device__ __forceinline__ void normal_words(FS &F, int a, unsigned int ctr, unsigned int c[4]) {
    c[0] = (unsigned int)a; c[1] = ctr; c[2] = 0x5344u; c[3] = 0x4d44u;
    philox10(c, F.key0, F.key1);
}
// the standard normal of those words
__device__ double normal_of(unsigned int c0, unsigned int c1, unsigned int c2, unsigned int c3) {
    const unsigned long long w1 = ((unsigned long long)c0 << 32) | c1;
    const unsigned long long w2 = ((unsigned long long)c2 << 32) | c3;
    const double u1 = ((double)(w1 >> 11) + 0.5) * 0x1.0p-53;
    const double u2 = ((double)(w2 >> 11) + 0.5) * 0x1.0p-53;
    return sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
}
// A lower bound of the normal's absolute value in FP32: u1 is rounded up
// (the logarithm's magnitude down), the logarithm and the cosine give up
// 1e-5.  Over all 2^32 words each, against FP64: the hardware's log2 is off by
// 1.9e-6 at most and its cosine by 1.3e-7, and the two bounds keep 7.7e-6 and
// 9.7e-6 of that; the root and the products round by 3e-7, the last factor
// gives up 1e-5.
// The FP64 normal takes about 400 dependent instructions on one lane; a
// thermostat time beyond the earliest event is dismissed without it (all but
// about 1 % of the predictions).
__device__ __forceinline__ float normal_floor(unsigned int c0, unsigned int c2) {
    const float u1 = fmaf((float)c0, 1.000001f, 1.f) * 0x1.0p-32f;
    const float l = -1.3862944f * __builtin_amdgcn_logf(u1) - 1e-5f;        // -2 ln u1
    const float c = fabsf(__builtin_amdgcn_cosf((float)c2 * 0x1.0p-32f)) - 1e-5f;
    return (l > 0 && c > 0) ? 0.99999f * __builtin_amdgcn_sqrtf(l) * c : 0.f;
}

__device__ double fast_normal(FSys &F, int a) {
    const unsigned int ctr = G(F.rctr)[a];
    unsigned int c[4];
    normal_words(F, a, ctr, c);
    G(F.rctr)[a] = ctr + 1;
    return normal_of(c[0], c[1], c[2], c[3]);
}

// ---------------------------------------------------------------- shared counters
// Several wavefronts update the system's counters (held in LDS) at once.
__device__ __forceinline__ void cnt_add(long long &c, long long v) {
    atomicAdd((unsigned long long *)&c, (unsigned long long)v);
}

__device__ __forceinline__ void cnt_max(double &d, double v) {
    unsigned long long *u = (unsigned long long *)&d;
    unsigned long long old = *u;
    while (__longlong_as_double((long long)old) < v) {
        const unsigned long long prev = atomicCAS(u, old, (unsigned long long)__double_as_longlong(v));
        if (prev == old) break;
        old = prev;
    }
}

// ---------------------------------------------------------------- uniform values
// Values every lane of a wave holds alike (the predicted atom's fields) are
// moved to scalar registers, which frees vector registers for the candidates.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ long long uni(long long v) {
    const int lo = __builtin_amdgcn_readfirstlane((int)v);
    const int hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
    return (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double uni(double v) { return __longlong_as_double(uni(__double_as_longlong(v))); }
__device__ __forceinline__ float uni(float v) { return __int_as_float(uni(__float_as_int(v))); }

// ---------------------------------------------------------------- state access
template <class SYS>
__device__ __forceinline__ int cell_id(SYS &S, int cx, int cy, int cz) {
    return cz * S.cellnum[1] * S.cellnum[2] + cy * S.cellnum[1] + cx + 1;
}

struct PosLocal {      // positions at time t from the local-time state, cells from the cell arrays
    const FSys &F;
    double t;
    __device__ void pos(int j, double *p) const {
        const Sys &S = F.s;
        const double dt = t - G(F.t0)[j];
        p[0] = G(S.x)[j] + G(S.vx)[j] * dt;
        p[1] = G(S.y)[j] + G(S.vy)[j] * dt;
        p[2] = G(S.z)[j] + G(S.vz)[j] * dt;
    }
    __device__ int first(int cell) const { return G(F.ccnt)[cell] > 0 ? G(F.cmem)[(size_t)cell * F.cap] : 0; }
    __device__ int next(int cell, int j) const {
        const int q = G(F.slot)[j] + 1;
        return (q > 0 && q < G(F.ccnt)[cell] && q < F.cap) ? G(F.cmem)[(size_t)cell * F.cap + q] : 0;
    }
};

__device__ __forceinline__ void advance(FSys &F, int a, double t) {
    Sys &S = F.s;
    const double dt = t - G(F.t0)[a];
    G(S.x)[a] = G(S.x)[a] + G(S.vx)[a] * dt;
    G(S.y)[a] = G(S.y)[a] + G(S.vy)[a] * dt;
    G(S.z)[a] = G(S.z)[a] + G(S.vz)[a] * dt;
    G(F.t0)[a] = t;
}

// mirror record of atom a (position at t0, expressed at epoch Te)
__device__ __forceinline__ void put_record(FV &F, double Te, int a) {
    SV &S = F.s;
    const int cx = G(S.cx)[a], cy = G(S.cy)[a], cz = G(S.cz)[a];
    const size_t at = (size_t)cell_id(S, cx, cy, cz) * F.cap + G(F.slot)[a];
    fvec4 r0, r1;
    r0.x = (float)(G(S.x)[a] - cx * S.cellsize[1]);
    r0.y = (float)(G(S.y)[a] - cy * S.cellsize[2]);
    r0.z = (float)(G(S.z)[a] - cz * S.cellsize[3]);
    r0.w = (float)(G(F.t0)[a] - Te);
    r1.x = (float)G(S.vx)[a];
    r1.y = (float)G(S.vy)[a];
    r1.z = (float)G(S.vz)[a];
    r1.w = __int_as_float((a << 8) | (G(S.type)[a] & 255));
    G(F.rec)[2 * at] = r0;
    G(F.rec)[2 * at + 1] = r1;
}

// ---------------------------------------------------------------- predicted atom
// Its fields are loaded by one wavefront, one per lane (ScrTab's gather map:
// lanes 0..6 eight bytes each, lanes 7..31 four), and kept in scalar
// registers: every lane uses them, and an LDS read costs a lone wavefront
// more than a hundred cycles each time it is waited for.
struct FAtom {
    double x, y, z, vx, vy, vz, t;
    int i, role, cx, cy, cz, type, hbbond, hbnb, protein, aanum, nbstat, nbnum, nb1, hbit;
    int co;                      // con_off at i
    unsigned int rctr;           // its thermostat draw counter
    int rowlo, spanok;           // static row: first column; its span is < 128 atom ids (byte lookup)
    bool hbscan;                 // a free H-bond atom: its neighbourhood is scanned for partners
    float tfloor;                // lower bound of the next thermostat draw's |normal|
    double pcc;                  // lane 0..2: cell-crossing time along that axis (or infinite)
};

// statistics accumulated per wave, added to the system at the end
struct WStats { long long screen, conf, fp64, cand; };

struct Best {
    double t, pot;
    long long pc;
    int partner, type, sub;
};

template <class SYS>
__device__ __forceinline__ void take(Best &B, SYS &S, double t, double pot, int sub, int type, int j) {
    // JobAssign, TimePrediction.c:1140-1158: strictly earlier and positive
    if (t > 0 && B.t > t) {
        B.t = t; B.pot = pot; B.sub = sub; B.type = type;
        if (j) { B.partner = j; B.pc = G(S.evc)[j]; }
        else { B.partner = INVALID; B.pc = 0; }
    }
}

constexpr int FCON = 16;          // constraint partners staged per predicted atom
constexpr int FCONSTEP = 8;       // steps per staged constraint
constexpr int FMARK = 32;         // words of first-candidate marks
constexpr int FCONN = 128;        // atom ids a row's bytes span

// Per-wavefront LDS.  NL: candidates inside the scan radius listed for the
// screen (25 to 60 at most sizes; a longer list takes the unlisted path).
template <int NL>
struct FWave {
    static constexpr int LIST = NL;
    int nbp[SDMD_NBSLOTS];       // the predicted atom's neighborPartner
    union {
        // the candidates inside the scan radius, in
        // candidate order; first their kinematics, then the screen's result
        struct {
            float l_rr[NL], l_b[NL], l_v2[NL];
        };
        struct {
            float l_t[NL], l_e[NL];              // time, error bound (negative: FP64 decides)
            int l_sh[NL];                        // shell (low byte), constraint slot + 1
        };
    };
    int l_id[NL];                // atom id << 8 | type, as in the mirror record
    int l_k[NL];                 // candidate index; bit 31: its local time is later than the reader's
    // the neighbour cells that hold candidates, in scan order: candidate k of
    // cell c has its record at slot cbase[c] + k; coff[c] is the cell's first
    // candidate (the number of candidates past the last cell)
    int coff[28];
    long long cbase[27];
    fvec4 cof[27];               // cell c's offset times the cell size (x, y, z)
    // bit p: candidate p + 1 is the first of its cell (a window of 64 * FMARK
    // candidates), so that a lane counts bits instead of searching coff
    unsigned long long mark[FMARK];
    // the predicted atom's constraint shells (FP32), CONSTRn lists
    ConRad con[FCON];
    int hbl_n;                   // entries of l_id / l_k left by the screen, -1: none listed
    // connection row by offset from its first column: bits 0-1 BOND and
    // CONSTRAINT, bits 2-6 the constraint's slot + 1 (0: not staged)
    unsigned char conn[FCONN];
    WStats st;                   // the wavefront's statistics (wave-uniform updates)
};
// the list's length by workgroup size (the LDS of a CU holds it all)
constexpr int flist(int W) { return W <= 8 ? 256 : 128; }

// BOND / CONSTRAINT bits of (A, j), the only connection bits CollisionTime
// tests (TimePrediction.c:96-118), with the staged constraint's slot; the
// dynamic slots carry H-bond bits only
template <class FW>
__device__ __forceinline__ int coli_bits(const FW &wm, SV &S, const FAtom &A, int j) {
    if (A.spanok) {
        const unsigned off = (unsigned)(j - A.rowlo);
        return off < 128u ? wm.conn[off] : 0;
    }
    return cmap_get(S, A.i, j) & (SDMD_BOND_CONNECT | SDMD_CONSTRAINT_CONNECT);
}

template <class FW>
__device__ __forceinline__ int fin_nb_list(const FW &wm, const FAtom &A, int j) {
    for (int k = 1; k < SDMD_NBSLOTS; k++) {
        if (wm.nbp[k] == 0) return 0;
        if (wm.nbp[k] == j) return k;
    }
    if (A.nbnum == 0) return 0;
    if (A.nbnum == j) return 5;
    if (A.nbstat == 0) return 0;
    if (A.nbstat == j) return 6;
    return 0;
}

// pair kinematics for atom A (at its time) and j (local state advanced to A.t)
__device__ __forceinline__ void kin_local(FV &F, const FAtom &A, int j, Kin &k, bool *late = nullptr) {
    SV &S = F.s;
    const double dt = A.t - G(F.t0)[j];
    if (late) *late = dt < 0;                  // j's state is later than A's time
    const double vxj = G(S.vx)[j], vyj = G(S.vy)[j], vzj = G(S.vz)[j];
    calc_params_at(S, A.x, A.y, A.z, A.vx, A.vy, A.vz, A.cx, A.cy, A.cz, j, G(S.x)[j] + vxj * dt, G(S.y)[j] + vyj * dt,
                   G(S.z)[j] + vzj * dt, vxj, vyj, vzj, k);
}

// one CollisionTime candidate in FP64 (TimePrediction.c:79-179), exclusions
// already applied; returns +inf when it does not reach JobAssign
// rp: the resolved collision pair of (A.type, type of j) (RightPair,
// ToolFunctions.c:278-292), known from the screen, so the table entry loads
// with j's state instead of after it
__device__ __forceinline__ double coli64(FV &F, const FAtom &A, int j, int bits, int rp, double calib, double &pot, int &sub,
                         bool &reached, bool &late, int *err) {
    SV &S = F.s;
    reached = false;
    pot = 0;
    sub = SDMD_INVALID_INTER;
    Kin k;
    kin_local(F, A, j, k, &late);
    if (!(k.rr <= calib)) return __builtin_inf();
    FP f;
    int cs;
    const int con = bits & SDMD_CONSTRAINT_CONNECT;
    if (con) {
        cs = find_pair(S, A.i, j, K_CONSTRAINT, k.b, k.rr, f, 0, 0, err);
    } else {
        cs = shell_lookup(S, rp >= 0 ? &S.pair[rp] : nullptr, K_COLLISION, k.b, k.rr, f, A.i, j, err);
        if (f.lopot == 0 && f.hipot == 0) return __builtin_inf();
    }
    int s;
    double d2;
    if (k.b < 0 && calc_disc(k, f.lo) > 0) {
        s = -1; d2 = f.lo; pot = f.lopot;
        sub = (cs == 0) ? SDMD_CORECOLLI : SDMD_TBDCAPTR;
    } else {
        s = 1; d2 = f.hi; pot = f.hipot;
        if (con) sub = (cs == 1) ? SDMD_WELLBOUNC : SDMD_TBDESCAP;
        else if (cs == 1) return __builtin_inf();
        else sub = SDMD_TBDESCAP;
    }
    reached = true;
    const double t = calc_time(k, s, d2);
    return (t > 0) ? t : __builtin_inf();
}

// FP32 screen of one collision candidate: time t with absolute error bound e,
// or flag when a decision lies inside the error band (FP64 decides then)
struct Scr { float t, e; bool flag; int ks; };    // ks: radii passed (the shell), valid unless flagged

// One shell description for the screen: hard core, step radii, outer
// limit (all squared), and bit k set when step k carries no energy.
struct Shell {
    float dmin, dmax;
    int nstep;
    unsigned int ezero;
};

// FP32 shell lookup + contact time; `rad(k)` gives step radius k
// The screen's FP32 square roots and reciprocals use the hardware
// instructions (about 1 ulp): every screened quantity carries an error band
// of 1e-5 relative or more, and every decision inside a band goes to FP64.
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }

// How far rounding can move a pair's distance vector: each component is a sum
// of five values of a cell's size at most, each rounded once in FP32, so the
// vector is off by D = sqrt(3) 5 2^-24 cells at most (6e-7 with some room).
// b is then off by D |v|, and r^2 by 2 r D <= 2e-5 r^2 + D^2 / 2e-5.  In cells
// of up to 6.6 and 23 A the bands hold that beside their floors.
struct ScrBand { float eb0, band0; };
static ScrBand screen_band(double cell) {
    const double D = 6e-7 * cell;
    return {(float)fmax(4e-6, D), (float)fmax(1e-5, D * D / 2e-5)};
}

template <class R>
__device__ __forceinline__ Scr screen_shell(const Shell &c, const R &rad, bool con, float rr, float b, float v2, ScrBand sb) {
    Scr o;
    o.t = FINF; o.e = 0; o.flag = false; o.ks = 0;
    const float band = 2e-5f * rr + sb.band0;
    if (rr < c.dmin + band) { o.flag = true; return o; }   // core boundary or inside the core
    // count the radii passed (no early exit; four radii read at a time with
    // unconditional loads clamped to the last step, so a group costs one
    // LDS round trip)
    int ks = 0;
    bool near = false;
    float lo = c.dmin, hi = FINF;
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 4) {
        if (k0 < c.nstep) {
            float dq[4];
#pragma unroll
            for (int u = 0; u < 4; u++) dq[u] = rad(k0 + u < c.nstep ? k0 + u : c.nstep - 1);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if (k0 + u < c.nstep) {
                    const float d = dq[u];
                    near |= fabsf(rr - d) < band;
                    if (rr > d) { ks++; lo = d; }
                    else if (hi == FINF) hi = d;
                }
            }
        }
    }
    if (near) { o.flag = true; return o; }
    o.ks = ks;
    const bool lopot0 = ks ? ((c.ezero >> (ks - 1)) & 1) : true;
    bool hipot0;
    int cs;
    const float eb = 1e-5f * fsqrt(rr * v2) + sb.eb0 * fsqrt(v2) + 1e-20f;
    if (fabsf(b) <= eb) { o.flag = true; return o; }
    if (ks < c.nstep) {
        hipot0 = (c.ezero >> ks) & 1;
        cs = ks == 0 ? 0 : -1;
    } else if (c.dmax > 0) {
        if (rr > c.dmax - band) { o.flag = true; return o; }   // at or beyond the outer limit
        hi = c.dmax;
        hipot0 = true;
        cs = (c.nstep == 0 && b < 0) ? 0 : 1;
    } else {
        // beyond the last step with no outer limit: an approaching pair still
        // reaches the outermost step; a leaving one has no event (collision)
        // or an unbounded one (constraint: left to FP64)
        if (con && !(b < 0)) { o.flag = true; return o; }
        hi = FINF;
        hipot0 = false;
        cs = 1;
    }
    if (!con && lopot0 && hipot0) return o;
    const float disc = b * b - v2 * (rr - lo);
    const float ed = 2.f * fabsf(b) * eb + v2 * band + 4e-6f * (b * b + v2 * rr);
    if (b < 0 && fabsf(disc) <= ed) { o.flag = true; return o; }
    float D;
    if (b < 0 && disc > 0) {
        D = -b + fsqrt(disc);
        o.t = (rr - lo) * frcp(D);
        o.e = 4.f * (band + o.t * (eb + ed * frcp(2.f * fsqrt(disc)))) * frcp(D) + 1e-4f * o.t;
    } else {
        if (!con && cs == 1) return o;
        const float dh = hi - rr;
        const float disc2 = b * b + v2 * dh;
        if (b > 0) {
            D = b + fsqrt(disc2);
            o.t = dh * frcp(D);
            o.e = 4.f * (band + o.t * (eb + (v2 * band + 2.f * b * eb) * frcp(2.f * fsqrt(disc2)))) * frcp(D) + 1e-4f * o.t;
        } else {
            o.t = (-b + fsqrt(disc2)) * frcp(v2);
            o.e = 1e-4f * o.t + 4.f * (eb + band + sb.eb0) * frcp(fsqrt(v2 + 1e-30f));
        }
    }
    if (!(o.t > o.e)) o.flag = true;                         // sign of t uncertain
    return o;
}

// compact FP32 copy of the collision table (RightPair resolved), held in LDS
constexpr int FRAD = 8192;        // steps of the defined pairs' lists in all at most
constexpr int FRADL = 2048;       // ... in the pool (equal lists stored once); the other pairs go to FP64
// indexed by (type_i, type_j) directly: the entry of the resolved pair,
// with that pair's index (one LDS read per candidate)
struct ScrPair {
    float dmin, dmax;
    unsigned short off;          // first radius in the FP32 pool
    unsigned short nstep;
    unsigned short ezero;        // bit k: step k carries no energy (nstep <= 16)
    short rp;                    // resolved pair (RightPair), -1 = none
};
static_assert(sizeof(ScrPair) == 16, "one 16-byte LDS read per screen table entry");
struct ScrTab {
    ScrPair pr[NT * NT];
    float rad[FRADL];
    // per-lane gather map of a predicted atom's fields: lane L loads the
    // 4-byte words gbase[L] + i*gstride[L] + goff[L] (+ gtwo[L]) of atom i
    unsigned long long gbase[64];
    int gstride[64], goff[64], gtwo[64];
};

// ---------------------------------------------------------------- wave helpers
__device__ __forceinline__ float wave_min_f(float t) {     // no NaN
    const unsigned b = __float_as_uint(t), s = (unsigned)((int)b >> 31);
    const unsigned m = wave_umin(b ^ (s | 0x80000000u));
    return __uint_as_float(m ^ ((m >> 31) ? 0x80000000u : 0xffffffffu));
}

__device__ __forceinline__ int wave_sum_i(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);     // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);     // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);     // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);     // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);     // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);     // row_bcast:31
    return lane_get(v, 63);
}

// broadcast a Best from lane src (uniform) to the wave
__device__ __forceinline__ void bcast(Best &B, int src) {
    B.t = lane_get(B.t, src);
    B.pot = lane_get(B.pot, src);
    B.pc = lane_get(B.pc, src);
    B.partner = lane_get(B.partner, src);
    B.type = lane_get(B.type, src);
    B.sub = lane_get(B.sub, src);
}

// wave-ordered min over per-lane candidates with program-order index k:
// the first minimal candidate wins (JobAssign's strict '<')
__device__ __forceinline__ void wave_best(Best &mine, int k, const Best &running, Best &out, int &win) {
    double t = mine.t;
    int kk = (t < running.t && t > 0) ? k : 0x7fffffff;
    if (kk == 0x7fffffff) t = __builtin_inf();
    wave_argmin(t, kk);
    win = kk;
    out = running;
    if (kk != 0x7fffffff) {
        // lane holding kk
        const unsigned long long m = __ballot(k == kk && mine.t == t);
        const int src = m ? __ffsll((long long)m) - 1 : 0;
        Best b = mine;
        bcast(b, src);
        out = b;
    }
}

// ---------------------------------------------------------------- Predict (one atom, one wave)
// Stage the predicted atom: its fields, its connection row and dynamic
// slots (LDS), the 27 neighbour cells and their occupancy prefix (LDS), and
// the bond entry of this lane (lanes < bond count).  No memory fence: the
// LDS data is shared within the wave only, whose LDS operations execute in
// order, so independent global loads stay in flight across the stages.
__device__ __forceinline__ fvec4 cv_load(const fvec4 *p) { return *(gptr_t<const fvec4>)p; }

// the predicted atom's mirror record (position, velocity, time since the epoch)
struct Own { float x, y, z, vx, vy, vz, t; };

struct BondPre {
    int j, sub;
    double lo, hi, xj, yj, zj, vxj, vyj, vzj, t0j;
    long long cj;
};

__device__ __forceinline__ int rl32(int v, int L) { return __builtin_amdgcn_readlane(v, L); }

// c_OX, c_OY, c_OZ with two bits per cell (offset + 1)
constexpr int OFFSETS[3][27] = {
    {0, 1, 0, 0, 0, 1, 1, 1, -1, 0, 0, 0, -1, -1, -1, 0, 0, 1, -1, 1, -1, -1, -1, 1, 1, 1, -1},
    {0, 0, 1, 0, 1, 0, 1, 1, 0, -1, 0, -1, 0, -1, -1, -1, 1, 0, 0, -1, 1, -1, 1, -1, 1, -1, 1},
    {0, 0, 0, 1, 1, 1, 0, 1, 0, 0, -1, -1, -1, 0, -1, 1, -1, -1, 1, 0, 0, 1, -1, -1, -1, 1, 1}};
constexpr unsigned long long pack_offsets(int axis) {
    unsigned long long w = 0;
    for (int c = 0; c < 27; c++) w |= (unsigned long long)(OFFSETS[axis][c] + 1) << (2 * c);
    return w;
}
constexpr unsigned long long OFF_X = pack_offsets(0), OFF_Y = pack_offsets(1), OFF_Z = pack_offsets(2);

// Two memory round trips: (1) every field of atom i, one per lane, through
// the gather map, with its bonded partners' ids; (2) its connection row,
// bond limits and partners' states, constraint entries with their FP32 step
// radii, and the 27 cells' occupancy.  Every load of a level is issued by
// all lanes (indices clamped into range, results masked afterwards), so a
// level costs one memory latency.
template <class FW>
__device__ __forceinline__ void fstage(FV &F, const ScrTab &T, FW &wm, FAtom &A, int i, double t, int &nb, Own &own, BondPre &bp) {
    SV &S = F.s;
    const int lane = threadIdx.x & 63;
    i = uni(i);
    t = uni(t);
    // ---- level 1 (lane map of the host's gather table): the members of
    // FAtom, lanes 48-63 the bonded partners; the role byte is loaded by
    // every lane
    static_assert(SDMD_NBSLOTS == 5 && FCONSTEP == 8, "lane map of the level-1 gather");
    const int *gp = (const int *)T.gbase[lane] + (size_t)i * T.gstride[lane] + T.goff[lane];
    const int lo = G(gp)[0], hi = G(gp)[T.gtwo[lane]];
    const int role = G(S.role)[i];
    const long long w = (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
    const int cx = rl32(lo, 8), cy = rl32(lo, 9), cz = rl32(lo, 10);
    nb = rl32(lo, 27) - rl32(lo, 26);
    const int co = rl32(lo, 28), ncon = rl32(lo, 29) - co;
    if (lane >= 18 && lane < 18 + SDMD_NBSLOTS) wm.nbp[lane - 18] = lo;
    const double p = __longlong_as_double(w);
    A.x = lane_get(p, 0); A.y = lane_get(p, 1); A.z = lane_get(p, 2);
    A.vx = lane_get(p, 3); A.vy = lane_get(p, 4); A.vz = lane_get(p, 5);
    A.t = t; A.i = i; A.role = uni(role); A.cx = cx; A.cy = cy; A.cz = cz; A.co = co;
    A.rctr = (unsigned)rl32(lo, 7);
    A.type = rl32(lo, 11); A.hbbond = rl32(lo, 12); A.hbnb = rl32(lo, 13); A.protein = rl32(lo, 14);
    A.aanum = rl32(lo, 15); A.nbstat = rl32(lo, 16); A.nbnum = rl32(lo, 17); A.nb1 = rl32(lo, 19);
    A.hbit = rl32(lo, 30);
    A.hbscan = A.hbit != SDMD_HBSKIP && A.hbbond <= 0 && (A.role == 'A' || A.role == 'D' || A.role == 'S');
    {
        // own mirror record, as put_record writes it for a state at time t
        const int ax = min(lane, 2), c = ax == 0 ? cx : ax == 1 ? cy : cz;
        const float f = (float)(lane < 3 ? p - c * S.cellsize[ax + 1] : p);
        own.x = lane_get(f, 0); own.y = lane_get(f, 1); own.z = lane_get(f, 2);
        own.vx = lane_get(f, 3); own.vy = lane_get(f, 4); own.vz = lane_get(f, 5);
    }
    // ---- level 2
    const int row = G(F.conn)[i * (FCONN / 4) + (lane & (FCONN / 4 - 1))];
    // bond q on lane 32 + q: its partner id came with level 1 (lane 48 + q)
    const int q = lane - 32;
    const bool bq = q >= 0 && q < nb && q < 16;
    // lanes 32..47 take lanes 48..63 (row-pair swap)
    const int bjs = (int)__builtin_amdgcn_permlane16_swap((unsigned)lo, (unsigned)lo, false, false)[1];
    const int bj = (bq && bjs >= 1 && bjs <= S.N) ? bjs : i;
    double blo = 0, bhi = 0;
    {
        const size_t qq = (size_t)i * 16 + (lane & 15);
        blo = G(F.blo16)[qq];
        bhi = G(F.bhi16)[qq];
    }
    fvec4 c0 = {0, 0, 0, 0}, c1 = c0, c2 = c0;
    if (ncon > 0) {
        const fvec4 *cv = (const fvec4 *)(F.crad + (co + min(lane, ncon - 1)));
        c0 = cv_load(cv); c1 = cv_load(cv + 1); c2 = cv_load(cv + 2);
    }
    const bool own_con = lane < ncon && lane < FCON;
    int cell;
    int ox, oy, oz;                                        // this lane's neighbour cell (lanes 27.. repeat cell 0)
    {
        const int sh2 = lane < 27 ? 2 * lane : 0;
        ox = (int)((OFF_X >> sh2) & 3) - 1; oy = (int)((OFF_Y >> sh2) & 3) - 1; oz = (int)((OFF_Z >> sh2) & 3) - 1;
        int n1 = cx + ox, n2 = cy + oy, n3 = cz + oz;
        if (n1 < 0) n1 = S.cellnum[1] - 1; else if (n1 >= S.cellnum[1]) n1 = 0;
        if (n2 < 0) n2 = S.cellnum[2] - 1; else if (n2 >= S.cellnum[2]) n2 = 0;
        if (n3 < 0) n3 = S.cellnum[3] - 1; else if (n3 >= S.cellnum[3]) n3 = 0;
        cell = cell_id(S, n1, n2, n3);
    }
    int cnt = G(F.ccnt)[cell];
    if (lane >= 27) cnt = 0;
    if (lane < FMARK) wm.mark[lane] = 0;
    // a cell farther from the atom than the scan radius holds no candidate:
    // an atom lies inside its cell until its cell-crossing event.  The margin
    // of 0.02 A holds that event's 1e-8 A, the record's rounding (6e-8 cells,
    // so cells of up to 100 000 A) and the rounding of the sum of squares.
    // The scan radius is 0.9 cells or less, which leaves 17 cells of 27.
    bool reach;
    {
        const float lx = own.x, ly = own.y, lz = own.z;
        const float m = 0.02f;
        const float dx = ox == 0 ? 0.f : fmaxf((ox < 0 ? lx : F.L32[0] - lx) - m, 0.f);
        const float dy = oy == 0 ? 0.f : fmaxf((oy < 0 ? ly : F.L32[1] - ly) - m, 0.f);
        const float dz = oz == 0 ? 0.f : fmaxf((oz < 0 ? lz : F.L32[2] - lz) - m, 0.f);
        const float c2 = (float)((S.cutoffr * SDMD_EXTEND_RATIO) * (S.cutoffr * SDMD_EXTEND_RATIO));
        reach = dx * dx + dy * dy + dz * dz <= c2 + (2e-5f * c2 + F.band0);
    }
    // PBCandCrossCellTime, TimePrediction.c:598-632, one axis per lane
    {
        const int ax = min(lane, 2);
        const double v = ax == 0 ? A.vx : ax == 1 ? A.vy : A.vz;
        const int ci = ax == 0 ? cx : ax == 1 ? cy : cz;
        const double cs = S.cellsize[ax + 1];
        const double tt = (v > 0 ? (ci + 1) * cs - p + ZERO : ci * cs - p - ZERO) / v;
        A.pcc = (v != 0 && tt > 0) ? tt : __builtin_inf();
    }
    // the thermostat draw's lower bound (while the loads above are in flight)
    A.tfloor = 0.f;
    if (S.thermostat) {
        unsigned int c[4];
        normal_words(F, i, A.rctr, c);
        A.tfloor = normal_floor(c[0], c[2]);
    }
    // bonded partners' states (any valid atom on other lanes)
    {
        const int j = bj;
        const double xj = G(S.x)[j], yj = G(S.y)[j], zj = G(S.z)[j];
        const double vxj = G(S.vx)[j], vyj = G(S.vy)[j], vzj = G(S.vz)[j];
        const double t0j = G(F.t0)[j];
        const long long cjj = G(S.evc)[j];
        bp.j = bq ? j : 0;
        bp.xj = xj; bp.yj = yj; bp.zj = zj; bp.vxj = vxj; bp.vyj = vyj; bp.vzj = vzj;
        bp.t0j = t0j; bp.cj = cjj; bp.lo = blo; bp.hi = bhi;
    }
    // ---- connection row and constraint shells (one lane each)
    if (lane < FCONN / 4) ((int *)wm.conn)[lane] = row;
    if (own_con) {
        fvec4 *cl = (fvec4 *)&wm.con[lane];
        cl[0] = c0; cl[1] = c1; cl[2] = c2;
    }
    A.rowlo = rl32(lo, 31);
    A.spanok = A.rowlo >= 0;
    // the cells in reach that hold atoms, packed in scan order, and the marks
    // of their first candidates; one prefix sum for the candidates in reach
    // (high half) and for those of all 27 cells (low half)
    {
        const bool keep = reach && cnt > 0;
        const int incl = scan32_incl(cnt | (keep ? cnt << 16 : 0));
        const int tot = lane_get(incl, 26), n = tot >> 16;
        const int start = (incl >> 16) - cnt;
        const unsigned km = (unsigned)(__ballot(keep) & 0x7ffffffu), below = (1u << (lane & 31)) - 1;
        const int nc = __popc(km), at = __popc(km & below);
        if (lane < 27 && keep) {
            fvec4 co4;
            co4.x = ox * F.L32[0];
            co4.y = oy * F.L32[1];
            co4.z = oz * F.L32[2];
            co4.w = 0.f;
            wm.cof[at] = co4;
            wm.cbase[at] = (long long)cell * F.cap - start;
            wm.coff[at] = start;
            if (start > 0 && start <= 64 * FMARK) atomicOr(&wm.mark[(start - 1) >> 6], 1ull << ((start - 1) & 63));
        } else if (lane < 28) {
            wm.coff[nc + __popc(~km & below)] = n;
        }
        if (lane == 0) wm.st.cand += (tot & 0xffff) - 1;
    }
    wave_sync();
}

// BondTime entry (TimePrediction.c:219-293) from the staged partner state
__device__ __forceinline__ double bond64_pre(FV &F, const FAtom &A, const BondPre &bp, int &sub) {
    SV &S = F.s;
    const int j = bp.j;
    const double dt = A.t - bp.t0j;
    Kin k;
    calc_params_at(S, A.x, A.y, A.z, A.vx, A.vy, A.vz, A.cx, A.cy, A.cz, j, bp.xj + bp.vxj * dt, bp.yj + bp.vyj * dt,
                   bp.zj + bp.vzj * dt, bp.vxj, bp.vyj, bp.vzj, k);
    const double lo = bp.lo, hi = bp.hi;
    double t;
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
    return (t > 0) ? t : __builtin_inf();
}

// cell of candidate k by search (the scans that do not go in order)
template <class FW>
__device__ __forceinline__ int cand_cell(const FW &wm, int k) {
    int lo = 0, hi = 26;                 // largest c with coff[c] <= k
    while (lo < hi) {
        const int m = (lo + hi + 1) >> 1;
        if (wm.coff[m] <= k) lo = m; else hi = m - 1;
    }
    return lo;
}

// the marks of the window of candidates that begins at `base`
template <class FW>
__device__ __forceinline__ void mark_window(FW &wm, int base, int n) {
    const int lane = threadIdx.x & 63;
    if (lane < FMARK) wm.mark[lane] = 0;
    wave_sync();
    if (lane < 27) {
        const int s = wm.coff[lane], p = s - 1 - base;
        if (s < n && p >= 0 && p < 64 * FMARK) atomicOr(&wm.mark[p >> 6], 1ull << (p & 63));
    }
    wave_sync();
}

// the mirror records of candidates base .. base + 64 * FQ - 1, whose loads
// issue together; `first`: cells that begin at or before candidate `base`,
// less one.  Lanes past the last candidate re-read it.
template <int FQ>
struct Group {
    fvec4 r0[FQ], r1[FQ];
    int cq[FQ];
};
template <int FQ, class FW>
__device__ __forceinline__ void load_group(FV &F, const FW &wm, int base, int n, int &first, Group<FQ> &g) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < FQ; q++) {
        if (base + 64 * q < n) {                           // uniform
            const unsigned long long m = (unsigned long long)uni((long long)wm.mark[((base >> 6) + q) & (FMARK - 1)]);
            const int c = first + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
            first += __popcll(m);
            const size_t at = (size_t)(wm.cbase[c] + min(base + lane + 64 * q, n - 1));
            g.cq[q] = c;
            g.r0[q] = G(F.rec)[2 * at];
            g.r1[q] = G(F.rec)[2 * at + 1];
        }
    }
}

// kinematics of a candidate from its mirror record (r0, r1) in neighbour
// cell c, in FP32, against the atom's own record
struct Near { float rr, b, v2, dt; };
template <class FW>
__device__ __forceinline__ Near near_at(const FW &wm, const Own &A, int c, const fvec4 &r0, const fvec4 &r1) {
    Near o;
    o.dt = A.t - r0.w;
    const fvec4 co = wm.cof[c];
    const float rx = A.x - (r0.x + r1.x * o.dt) - co.x;
    const float ry = A.y - (r0.y + r1.y * o.dt) - co.y;
    const float rz = A.z - (r0.z + r1.z * o.dt) - co.z;
    o.rr = rx * rx + ry * ry + rz * rz;
    const float vx = A.vx - r1.x, vy = A.vy - r1.y, vz = A.vz - r1.z;
    o.b = rx * vx + ry * vy + rz * vz;
    o.v2 = vx * vx + vy * vy + vz * vz;
    return o;
}

// FP32 screen of one candidate inside the scan radius
struct CandS {
    float t, e;       // screened time and its absolute error bound (t = FINF: no event)
    int j, bits;
    int rp;           // resolved collision pair (-1: none or a constraint pair)
    int ks, slot;     // shell; staged constraint slot (-1: a collision pair)
    bool flag;        // a decision lies in the error band: FP64 decides
    bool live;        // passed the exclusions
};

template <class FW>
__device__ __forceinline__ void screen_near(FV &F, const ScrTab &T, const FW &wm, const FAtom &A, int id,
                                            float rr, float b, float v2, float rsafe, CandS &o) {
    SV &S = F.s;
    o.t = FINF; o.e = 0; o.flag = false; o.live = false; o.rp = -1; o.ks = 0; o.slot = -1;
    const int j = id >> 8, tj = id & 255;
    o.j = j;
    const int cb = coli_bits(wm, S, A, j);
    o.bits = cb & (SDMD_BOND_CONNECT | SDMD_CONSTRAINT_CONNECT);
    if ((cb & SDMD_BOND_CONNECT) || A.hbbond == j || (A.nb1 && fin_nb_list(wm, A, j))) return;
    o.live = true;
    const bool con = cb & SDMD_CONSTRAINT_CONNECT;
    Shell c;
    const float *rad;
    if (con) {
        const int q = (cb >> 2) - 1;
        o.slot = q;
        if (q < 0) { o.flag = true; return; }             // not staged: FP64 decides
        const ConRad &cr = wm.con[q];
        c.dmin = cr.dmin; c.dmax = cr.dmax; c.nstep = cr.nstep; c.ezero = cr.ez;
        rad = cr.rad;
    } else {
        const ScrPair sp = T.pr[A.type * NT + tj];
        o.rp = sp.rp;
        if (sp.rp < 0 || sp.off == 0xffff) { o.flag = true; return; }
        c.dmin = sp.dmin; c.dmax = sp.dmax; c.nstep = sp.nstep; c.ezero = sp.ezero;
        rad = T.rad + sp.off;
    }
    const Scr sc = screen_shell(c, [&](int k) { return rad[k]; }, con, rr, b, v2, ScrBand{F.eb0, F.band0});
    o.t = sc.t; o.e = sc.e; o.ks = sc.ks; o.flag = sc.flag || (rr > rsafe);
}

// One screened candidate in FP64 (TimePrediction.c:79-179) in the shell the
// screen found: no radius lies inside the screen's band around the pair's
// distance (nor the scan radius), so the FP64 search would end in the same
// shell, and the shell's limits and energies load together with j's state (one round trip).
// Returns +inf when it does not reach JobAssign.
template <class FW>
__device__ __forceinline__ double coli64_shell(FV &F, const ScrTab &T, const FW &wm, const FAtom &A, int id, int ks,
                                               int slot, double &pot, int &sub, long long &pc, bool &late) {
    SV &S = F.s;
    const int j = id >> 8;
    const bool con = slot >= 0;
    const ScrPair sp = T.pr[A.type * NT + (id & 255)];
    const int nstep = con ? wm.con[slot & (FCON - 1)].nstep : (int)sp.nstep, stride = con ? FCONSTEP : PROW;
    const double *row = con ? F.crow + (size_t)(A.co + slot) * (2 + 2 * FCONSTEP)
                            : F.prow + (size_t)max((int)sp.rp, 0) * (2 + 2 * PROW);
    const int kl = max(ks - 1, 0), kh = min(ks, stride - 1);
    const double dmin = G(row)[0], dmax = G(row)[1];
    const double dl = G(row)[2 + kl], el = G(row)[2 + stride + kl], dh = G(row)[2 + kh], eh = G(row)[2 + stride + kh];
    pc = G(S.evc)[j];
    Kin k;
    kin_local(F, A, j, k, &late);
    const double lo = ks > 0 ? dl : dmin, lopot = ks > 0 ? el : 0;
    double hi, hipot;
    int cs;
    if (ks < nstep) { hi = dh; hipot = -1 * eh; cs = ks == 0 ? 0 : -1; }
    else if (dmax > 0) { hi = dmax; hipot = 0; cs = (nstep == 0 && k.b < 0) ? 0 : 1; }
    else { hi = INFINIT; hipot = INFINIT; cs = 1; }
    pot = 0;
    sub = SDMD_INVALID_INTER;
    if (!con && lopot == 0 && hipot == 0) return __builtin_inf();
    int s;
    double d2;
    if (k.b < 0 && calc_disc(k, lo) > 0) {
        s = -1; d2 = lo; pot = lopot;
        sub = (cs == 0) ? SDMD_CORECOLLI : SDMD_TBDCAPTR;
    } else {
        s = 1; d2 = hi; pot = hipot;
        if (con) sub = (cs == 1) ? SDMD_WELLBOUNC : SDMD_TBDESCAP;
        else if (cs == 1) return __builtin_inf();
        else sub = SDMD_TBDESCAP;
    }
    const double t = calc_time(k, s, d2);
    return (t > 0) ? t : __builtin_inf();
}

// FQ: candidates per lane whose records are loaded together

// HBTime's bookkeeping of listed candidate `lane`
struct HBPre { int role, aanum, protein, hbbond; };

// Screened CollisionTime: the candidates inside the scan radius are listed
// in LDS (a quarter of the neighbourhood), screened in FP32 one per lane, and
// the marked ones and those whose interval reaches the smallest upper bound
// are re-solved in FP64; the FP64 minimum (first in scan order on ties)
// competes with the running best under JobAssign's strict '<'.
// A lone wavefront issues a dependent instruction every 8 cycles and an
// independent one every 5 (measured), so what counts is how often the long
// screen runs: once per 64 listed candidates instead of once per 64 scanned.
// VAL: validation mode (the winner of a full FP64 scan compared), kernels of
// their own: as a second form inside the same kernels its registers slowed the
// screened path of the 8-wavefront shape by 14 %
template <int FQ, bool VAL, class FW>
__device__ __forceinline__ void collision_fast(FSys &M, FV &F, unsigned long long *prof, const ScrTab &T, FW &wm, const FAtom &A, const Own &own,
                                               Group<FQ> &g, int first, HBPre &hp, Best &best, long long &nscreen,
                                               long long &nconf, int *err) {
    SV &S = F.s;
    unsigned long long pt = prof ? wall_clock64() : 0;
    const int lane = threadIdx.x & 63;
    const int n = uni(wm.coff[27]);
    const double calib64 = (S.cutoffr * SDMD_EXTEND_RATIO) * (S.cutoffr * SDMD_EXTEND_RATIO);
    const float calib = (float)calib64;
    const float cband = 2e-5f * calib + F.band0, rscan = calib + cband, rsafe = calib - cband;
    int screened = 0, confirmed = 0;                       // wave-uniform
    int my_causal = 0;
    Best mine;
    mine.t = __builtin_inf(); mine.pot = 0; mine.pc = 0; mine.partner = INVALID; mine.type = SDMD_COLI; mine.sub = 0;
    int mink = 0x7fffffff;
    Best full = mine;
    int fullk = 0x7fffffff;
    float myt32 = FINF;
    // FP64 re-solve of candidate k
    auto confirm = [&](int k, int id, int bits, int rp, float t32, int ks, int slot, bool flag) {
        double pot, t;
        int sub;
        bool late;
        long long pc = 0;
        if (flag) {
            bool reached;
            t = coli64(F, A, id >> 8, bits, rp, calib64, pot, sub, reached, late, err);
            pc = G(S.evc)[id >> 8];
        } else {
            t = coli64_shell(F, T, wm, A, id, ks, slot, pot, sub, pc, late);
        }
        my_causal += late ? 1 : 0;             // FP64 check of the screen's FP32 time order
        if (t < mine.t) { mine.t = t; mine.pot = pot; mine.sub = sub; mine.partner = id >> 8; mine.pc = pc; mink = k; myt32 = t32; }
    };
    // ---- the candidates inside the scan radius, in candidate order
    int near = 0;
    for (int base = 0; base < n;) {
#pragma unroll
        for (int q = 0; q < FQ; q++) {
            const int k = base + lane + 64 * q;
            if (base + 64 * q < n) {                       // uniform
                const int id = __float_as_int(g.r1[q].w), j = id >> 8;
                const Near d = near_at(wm, own, g.cq[q], g.r0[q], g.r1[q]);
                const bool nr = k < n && j >= 1 && j <= S.N && j != A.i && (id & 255) < NT && d.rr <= rscan;
                const unsigned long long m = __ballot(nr);
                const int r = near + __builtin_amdgcn_mbcnt_hi((unsigned int)(m >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((unsigned int)m, 0));
                if (nr && r < FW::LIST) {
                    wm.l_rr[r] = d.rr; wm.l_b[r] = d.b; wm.l_v2[r] = d.v2;
                    wm.l_id[r] = id;
                    wm.l_k[r] = k | (d.dt < 0.f ? (int)0x80000000 : 0);
                }
                near += __popcll(m);
            }
        }
        base += 64 * FQ;
        if (base >= n) break;
        if ((base & (64 * FMARK - 1)) == 0) mark_window(wm, base, n);
        load_group<FQ>(F, wm, base, n, first, g);
    }
    wave_sync();
    if (near <= FW::LIST) {
        // HBTime's bookkeeping of the first 64 listed candidates, in flight
        // during the screen
        hp.role = 0;
        if (A.hbscan && lane < near) {
            const int j = wm.l_id[lane] >> 8;
            hp.role = G(S.role)[j]; hp.aanum = G(S.aanum)[j]; hp.protein = G(S.protein)[j]; hp.hbbond = G(S.hbbond)[j];
        }
        float thi = FINF;
        for (int r0 = 0; r0 < near; r0 += 64) {
            const int r = r0 + lane;
            CandS o;
            o.live = false;
            if (r < near) {
            screen_near(F, T, wm, A, wm.l_id[r], wm.l_rr[r], wm.l_b[r], wm.l_v2[r], rsafe, o);
            my_causal += (o.live && wm.l_k[r] < 0) ? 1 : 0;
            if (o.live && !o.flag && o.t < FINF) thi = fminf(thi, o.t + o.e);
            wm.l_t[r] = o.live ? o.t : FINF;
            wm.l_e[r] = (o.live && o.flag) ? -1.f : o.e;
            wm.l_sh[r] = o.ks | ((o.slot + 1) << 8);
            }
            screened += __popcll(__ballot(o.live));
        }
        if (lane == 0) wm.hbl_n = near;
        thi = wave_min_f(thi);
        FPROF(prof, FPH_SCREEN, pt);
        for (int r0 = 0; r0 < near; r0 += 64) {
            const int r = r0 + lane, rl = min(r, near - 1);
            const float t = wm.l_t[rl], e = wm.l_e[rl];
            const int sh = wm.l_sh[rl];
            const bool flag = e < 0.f, need = r < near && (flag || (t < FINF && t - e <= thi));
            confirmed += __popcll(__ballot(need));
            if (need) {
                const int id = wm.l_id[r], slot = ((sh >> 8) & 255) - 1;
                // what the FP64 search of a marked candidate needs
                const int bits = coli_bits(wm, S, A, id >> 8) & (SDMD_BOND_CONNECT | SDMD_CONSTRAINT_CONNECT);
                const int rp = (bits & SDMD_CONSTRAINT_CONNECT) ? -1 : T.pr[A.type * NT + (id & 255)].rp;
                confirm(wm.l_k[r] & 0x7fffffff, id, bits, rp, t, sh & 255, slot, flag);
            }
        }
    } else {
        // more candidates inside the radius than the list holds: bound
        // first, then re-screen and confirm
        float thi = FINF;
        for (int pass = 0; pass < 2; pass++) {
            for (int k0 = 0; k0 < n; k0 += 64) {
                const int k = k0 + lane, kl = min(k, n - 1);
                const int c = cand_cell(wm, kl);
                const size_t at = (size_t)(wm.cbase[c] + kl);
                const fvec4 q0 = G(F.rec)[2 * at], q1 = G(F.rec)[2 * at + 1];
                const int id = __float_as_int(q1.w), j = id >> 8;
                const Near d = near_at(wm, own, c, q0, q1);
                CandS o;
                o.live = false;
                if (k < n && j >= 1 && j <= S.N && j != A.i && (id & 255) < NT && d.rr <= rscan)
                    screen_near(F, T, wm, A, id, d.rr, d.b, d.v2, rsafe, o);
                if (pass == 0) {
                    screened += __popcll(__ballot(o.live));
                    if (o.live) {
                        my_causal += d.dt < 0.f ? 1 : 0;
                        if (!o.flag && o.t < FINF) thi = fminf(thi, o.t + o.e);
                    }
                } else {
                    const bool need = o.live && (o.flag || (o.t < FINF && o.t - o.e <= thi));
                    confirmed += __popcll(__ballot(need));
                    if (need) confirm(k, id, o.bits, o.rp, o.t, o.ks, o.slot, o.flag);
                }
            }
            if (pass == 0) thi = wave_min_f(thi);
        }
    }
    if constexpr (VAL) {
        // every atom of the 27 cells in scan order, from the cell arrays and
        // the FP64 state alone: what the staging drops (a cell taken to be out
        // of reach, a record found under another cell) shows as a disagreement
        const int cl = min(lane, 26);
        int n1 = A.cx + c_OX[cl], n2 = A.cy + c_OY[cl], n3 = A.cz + c_OZ[cl];
        if (n1 < 0) n1 = S.cellnum[1] - 1; else if (n1 >= S.cellnum[1]) n1 = 0;
        if (n2 < 0) n2 = S.cellnum[2] - 1; else if (n2 >= S.cellnum[2]) n2 = 0;
        if (n3 < 0) n3 = S.cellnum[3] - 1; else if (n3 >= S.cellnum[3]) n3 = 0;
        const int cell = cell_id(S, n1, n2, n3);
        const int cnt = lane < 27 ? min(G(F.ccnt)[cell], F.cap) : 0, incl = scan32_incl(cnt);
        const int all = lane_get(incl, 26);
        for (int k0 = 0; k0 < all; k0 += 64) {
            const int k = min(k0 + lane, all - 1);
            int c = 0;                                     // cells that end at or before candidate k
#pragma unroll
            for (int step = 16; step > 0; step >>= 1)
                if (__shfl(incl, c + step - 1, 64) <= k) c += step;
            const int before = __shfl(incl - cnt, c, 64), id = __shfl(cell, c, 64);
            const int j = G(F.cmem)[(size_t)id * F.cap + (k - before)];
            if (k0 + lane < all && j >= 1 && j <= S.N && j != A.i) {
                const int bits = coli_bits(wm, S, A, j) & (SDMD_BOND_CONNECT | SDMD_CONSTRAINT_CONNECT), tj = G(S.type)[j];
                Kin kin;
                bool late, reached;
                kin_local(F, A, j, kin, &late);
                if (!(bits & SDMD_BOND_CONNECT) && A.hbbond != j && !fin_nb_list(wm, A, j) && kin.rr <= calib64) {
                    const int rp = (bits & SDMD_CONSTRAINT_CONNECT) ? -1 : T.pr[A.type * NT + tj].rp;
                    double pot;
                    int sub;
                    my_causal += late ? 1 : 0;
                    const double t = coli64(F, A, j, bits, rp, calib64, pot, sub, reached, late, err);
                    if (t < full.t) { full.t = t; full.pot = pot; full.sub = sub; full.partner = j; fullk = k; }
                }
            }
        }
    }
    FPROF(prof, FPH_CONFIRM, pt);
    nscreen += screened;
    nconf += confirmed;
    if (__ballot(my_causal != 0)) {
        my_causal = wave_sum_i(my_causal);
        if (lane == 0) {
            cnt_add(M.causal, my_causal);
            *err = FERR_CAUSAL;
        }
    }
    // wave argmin (first minimal candidate)
    double tw = mine.t;
    int kw = mink;
    wave_argmin(tw, kw);
    Best win = mine;
    {
        const unsigned long long m = __ballot(mink == kw && kw != 0x7fffffff);
        const int src = m ? __ffsll((long long)m) - 1 : 0;
        bcast(win, src);
        const float w32 = lane_get(myt32, src);
        if (m && lane == 0 && win.t > 0 && w32 < FINF) cnt_max(M.max_screen_err, fabs((double)w32 - win.t) / win.t);
        if (!m) win.t = __builtin_inf();
    }
    if constexpr (VAL) {
        double tf = full.t;
        int kf = fullk;
        wave_argmin(tf, kf);
        const unsigned long long m = __ballot(fullk == kf && kf != 0x7fffffff);
        const int src = m ? __ffsll((long long)m) - 1 : 0;
        Best fw = full;
        bcast(fw, src);
        if (!m) fw.t = __builtin_inf();
        if (lane == 0) {
            cnt_add(M.validated, 1);
            const bool same = (!m && win.t == __builtin_inf()) ||
                              (fw.partner == win.partner && fw.t == win.t && fw.sub == win.sub);
            if (same) cnt_add(M.agree, 1);
            else if (fw.t < __builtin_inf()) cnt_max(M.max_time_err, fabs(win.t - fw.t) / fw.t);
        }
    }
    if (win.t < __builtin_inf() && win.partner > 0 && win.t > 0 && best.t > win.t) {
        best.t = win.t; best.pot = win.pot; best.sub = win.sub; best.type = SDMD_COLI;
        best.partner = win.partner; best.pc = win.pc;
    }
}

// free-atom HBTime candidate (TimePrediction.c:414-478) at local time, in
// two parts: the conditions on j's bookkeeping alone (role pairing, j not
// H-bonded, sequence separation within a chain: TimePrediction.c:420-430),
// then distance, CheckPairMatch, FindPair and the contact time
__device__ __forceinline__ bool hbfree_pre(const FAtom &A, const HBPre &h, int tj) {
    const int ri = A.role, rj = h.role;
    const bool pairok = (ri == 'A' && rj == 'D') || (ri == 'D' && rj == 'A') || (ri == 'S' && tj == 2) ||
                        (rj == 'S' && A.type == 2) || (ri == 'S' && rj == 'S');
    int sep = A.aanum - h.aanum;
    if (sep < 0) sep = -sep;
    return pairok && h.hbbond == 0 && ((A.protein == h.protein && sep >= 4) || A.protein != h.protein);
}

__device__ __forceinline__ bool hbfree_pass(FV &F, const FAtom &A, int j) {
    SV &S = F.s;
    if (j < 1 || j > S.N || j == A.i) return false;
    const HBPre h = {G(S.role)[j], G(S.aanum)[j], G(S.protein)[j], G(S.hbbond)[j]};
    return hbfree_pre(A, h, G(S.type)[j]);
}

__device__ __forceinline__ double hbfree64(FV &F, const FAtom &A, int j, double calib, double &pot, bool &reached, int *err) {
    SV &S = F.s;
    reached = false;
    pot = 0;
    Kin k;
    kin_local(F, A, j, k);
    if (!(k.rr <= calib) || check_pair_match(S, A.i, j, err) < 0) return __builtin_inf();
    FP f;
    const int cs = find_pair(S, A.i, j, K_HB, k.b, k.rr, f, 0, 0, err);
    reached = true;
    if (k.b < 0 && cs == 1 && calc_disc(k, f.lo) > 0) {
        pot = f.lopot;
        double t = calc_time(k, -1, f.lo);
        if (t < 0) t = INFINIT;
        return (t > 0) ? t : __builtin_inf();
    }
    return __builtin_inf();
}

// Predict for atom i at time t (its state is at t); writes the event record
template <int FQ, bool VAL, class FW>
__device__ __forceinline__ void predict_fast(FSys &M, FV &F0, unsigned long long *prof, const ScrTab &T, FW &wm, int i,
                                             double t, WStats &ws, int *err) {
    const int lane = threadIdx.x & 63;
    long long &nscreen = ws.screen, &nconf = ws.conf, &nfp64 = ws.fp64;
    unsigned long long pt = prof ? wall_clock64() : 0;
    FAtom A;
    Own own;
    int nb = 0;
    BondPre bp;                                            // lanes 32 .. 47: one bonded partner each
    fstage(view_anew(F0), T, wm, A, i, t, nb, own, bp);
    FV &F = view_anew(F0);
    SV &S = F.s;
    // the first candidates' records load during the bond times
    const int n = uni(wm.coff[27]);
    int first = 0;
    Group<FQ> g;
    load_group<FQ>(F, wm, 0, n, first, g);
    own.t = (float)(A.t - M.Te);
    FPROF(prof, FPH_STAGE, pt);
    if (nb > 16 && lane == 0) *err = ERR_CELLCAP;      // BondTime's connect[16], TimePrediction.c:188
    Best init;
    init.t = INFINIT; init.pot = 0; init.pc = 0; init.partner = INVALID; init.type = SDMD_INVD; init.sub = 0;
    // BondTime: one lane per bond (lanes 32..), first minimal wins; done
    // before the screen so the staged partner state is dead during it
    Best best = init;
    {
        Best mine = init;
        mine.t = __builtin_inf();
        const int q = lane - 32;
        if (bp.j > 0) {
            int sub;
            mine.t = bond64_pre(F, A, bp, sub);
            mine.sub = sub; mine.pot = 0; mine.type = SDMD_BOND; mine.partner = bp.j; mine.pc = bp.cj;
        }
        Best out;
        int win;
        wave_best(mine, q, best, out, win);
        best = out;
        nfp64 += nb;
    }
    FPROF(prof, FPH_BOND, pt);
    // CollisionTime (screened), against no running best yet
    if (lane == 0) wm.hbl_n = -1;
    wave_sync();
    Best cw = init;
    cw.t = __builtin_inf();
    HBPre hp;
    // (its own view: the constants read before would be held over it, 407
    // vector registers spilled against 228 in the 8-wavefront shape)
    collision_fast<FQ, VAL>(M, view_anew(F0), prof, T, wm, A, own, g, first, hp, cw, nscreen, nconf, err);
    if (prof) pt = wall_clock64();
    // JobAssign order: bonds first, then the collision winner if strictly earlier
    if (cw.partner > 0 && cw.t > 0 && best.t > cw.t) best = cw;
    // PBCandCrossCellTime (each axis's time from the staging)
    {
        const double t_ev = fmin(fmin(lane_get(A.pcc, 0), lane_get(A.pcc, 1)), fmin(lane_get(A.pcc, 2), INFINIT));
        take(best, S, t_ev, 0, SDMD_INVALID_INTER, SDMD_PCC, 0);
    }
    // ThermostatTime, TimePrediction.c:582-595
    if (S.thermostat) {
        const unsigned int ctr = A.rctr;
        if (lane == 0) G(F.rctr)[i] = ctr + 1;
        if (!(S.thermoF * (double)A.tfloor > best.t)) {
            unsigned int c[4];
            normal_words(F, A.i, ctr, c);
            const double z = normal_of(c[0], c[1], c[2], c[3]);
            const double tt = S.thermoF * ((z < 0) ? (-z) : (z));
            take(best, S, tt, 0, SDMD_INVALID_INTER, SDMD_THER, 0);
        }
    }
    // HBTime head, TimePrediction.c:309-330
    const double calib = (S.cutoffr * SDMD_EXTEND_RATIO) * (S.cutoffr * SDMD_EXTEND_RATIO);
    const int hbit = A.hbit;
    if (lane == 0) G(S.hbitype)[i] = SDMD_NOEVENT;
    // The bonded H-bond partner's time (lane 32) and HBNeighborTime's pair
    // times over neighborPartner[1..4] (lane q - 1 for slot q) read state
    // only, so they are solved at once here and applied below in the
    // reference's order (HBTime first, then the slots in order)
    const int nq = min(A.nbstat, SDMD_NBSLOTS - 1);
    const bool hbb = hbit != SDMD_HBSKIP && A.hbbond > 0;
    double pt_t = INFINIT, pt_pot = 0;
    int pt_sub = 0;
    if (lane < nq) {
        // HBNeighborTime slot q, TimePrediction.c:486-579
        const int j = wm.nbp[lane + 1];
        Kin k;
        kin_local(F, A, j, k);
        int host, nb, partner;
        const bool ads = (A.role == 'A' || A.role == 'D' || A.role == 'S');
        if (ads && A.hbbond && G(S.hbnb)[A.hbbond] == j) { host = i; nb = j; partner = A.hbbond; }
        else { host = j; nb = i; partner = G(S.hbbond)[j]; }
        FP f;
        const int cs = find_pair(S, nb, host, K_NEIGHBOR, k.b, k.rr, f, partner, 0, err);
        int s;
        double d2;
        if (k.b < 0 && calc_disc(k, f.lo) > 0) {
            s = -1; d2 = f.lo; pt_pot = f.lopot;
            pt_sub = (cs == 0) ? SDMD_CORECOLLI : SDMD_TBDCAPTR;
        } else {
            s = 1; d2 = f.hi; pt_pot = f.hipot;
            pt_sub = (cs == 1) ? SDMD_WELLBOUNC : SDMD_TBDESCAP;
        }
        pt_t = calc_time(k, s, d2);
        if (pt_t < 0) pt_t = INFINIT;
    } else if (lane == 32 && hbb) {
        // bonded HB partner, TimePrediction.c:330-383
        const int j = A.hbbond;
        Kin k;
        kin_local(F, A, j, k);
        FP f;
        const int cs = find_pair(S, i, j, K_HB, k.b, k.rr, f, 0, 0, err);
        int s;
        double d2;
        if (k.b < 0 && calc_disc(k, f.lo) > 0) {
            s = -1; d2 = f.lo; pt_pot = f.lopot;
            pt_sub = (cs == 0) ? SDMD_CORECOLLI : SDMD_TBDCAPTR;
        } else {
            s = 1; d2 = f.hi; pt_pot = f.hipot;
            pt_sub = (cs == 1) ? SDMD_TBDHBBRIK : SDMD_TBDESCAP;
        }
        pt_t = calc_time(k, s, d2);
        if (pt_t < 0) pt_t = INFINIT;
    }
    if (hbit != SDMD_HBSKIP) {
        if (A.hbbond > 0) {
            const double tt = lane_get(pt_t, 32), pot = lane_get(pt_pot, 32);
            const int sub = lane_get(pt_sub, 32);
            take(best, S, tt, pot, sub, SDMD_HB, A.hbbond);
            nfp64 += 1;
        } else if (A.role == 'A' || A.role == 'D' || A.role == 'S') {
            // free HB atom: scan the neighbourhood in FP64, 128 candidates at
            // a time: the conditions on j's bookkeeping for two candidates
            // per lane (their loads issued together), then the FP64 part for
            // the candidates that pass, packed onto the wave's lanes in
            // candidate order (most candidates fail the role pairing)
            Best mine = best;
            mine.t = __builtin_inf();
            int mink = 0x7fffffff;
            int my = 0;
            const int nl = wm.hbl_n;
            // the candidates the screen listed inside the scan radius, in
            // candidate order; otherwise every candidate, filtered below
            for (int r = lane; r < nl; r += 64) {
                const int id = wm.l_id[r], j = id >> 8, k = wm.l_k[r] & 0x7fffffff;
                if (!(r == lane ? hbfree_pre(A, hp, id & 255) : hbfree_pass(F, A, j))) continue;
                double pot;
                bool reached;
                const double tt = hbfree64(F, A, j, calib, pot, reached, err);
                my += reached;
                if (tt < mine.t) { mine.t = tt; mine.pot = pot; mine.partner = j; mink = k; }
            }
            for (int base = 0; nl < 0 && base < n; base += 128) {
                int jj[2];
                bool ok[2];
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int k = base + 64 * u + lane;
                    jj[u] = 0;
                    if (k < n) {
                        const int c = cand_cell(wm, k);
                        const size_t at = (size_t)(wm.cbase[c] + k);
                        jj[u] = __float_as_int(G(F.rec)[2 * at + 1].w) >> 8;
                    }
                }
#pragma unroll
                for (int u = 0; u < 2; u++) ok[u] = hbfree_pass(F, A, jj[u]);
                const unsigned long long m0 = __ballot(ok[0]), m1 = __ballot(ok[1]);
                const int n0 = __popcll(m0), npass = n0 + __popcll(m1);
                const unsigned int lo = (unsigned int)((1ull << lane) - 1);
                const unsigned int hi = (unsigned int)(((1ull << lane) - 1) >> 32);
                const int r0 = __builtin_amdgcn_mbcnt_hi((unsigned int)(m0 >> 32) & hi,
                                                         __builtin_amdgcn_mbcnt_lo((unsigned int)m0 & lo, 0));
                const int r1 = n0 + __builtin_amdgcn_mbcnt_hi((unsigned int)(m1 >> 32) & hi,
                                                              __builtin_amdgcn_mbcnt_lo((unsigned int)m1 & lo, 0));
                wave_sync();
                if (ok[0]) { wm.l_id[r0] = jj[0] << 8; wm.l_k[r0] = base + lane; }
                if (ok[1]) { wm.l_id[r1] = jj[1] << 8; wm.l_k[r1] = base + 64 + lane; }
                wave_sync();
                for (int r = lane; r < npass; r += 64) {
                    const int j = wm.l_id[r] >> 8, k = wm.l_k[r];
                    double pot;
                    bool reached;
                    const double tt = hbfree64(F, A, j, calib, pot, reached, err);
                    my += reached;
                    if (tt < mine.t) { mine.t = tt; mine.pot = pot; mine.partner = j; mink = k; }
                }
                wave_sync();
            }
            nfp64 += wave_sum_i(my);
            double tw = mine.t;
            int kw = mink;
            wave_argmin(tw, kw);
            const unsigned long long m = __ballot(mink == kw && kw != 0x7fffffff);
            if (m) {
                const int src = __ffsll((long long)m) - 1;
                Best w = mine;
                bcast(w, src);
                take(best, S, w.t, w.pot, SDMD_TBDHBFORM, SDMD_HB, w.partner);
            }
        }
    }
    // HBNeighborTime, TimePrediction.c:486-579: the slots' times (solved
    // above) through JobAssign in slot order; neighborPartnerNum is the
    // winning slot, else the last one
    {
        int flag = 0;
        for (int q = 1; q <= nq; q++) {
            const double tt = lane_get(pt_t, q - 1), pot = lane_get(pt_pot, q - 1);
            const int sub = lane_get(pt_sub, q - 1);
            if (flag == 0) A.nbnum = q;
            nfp64 += 1;
            if (tt > 0 && best.t > tt) {
                take(best, S, tt, pot, sub, SDMD_HBNE, wm.nbp[q]);
                A.nbnum = q;
                flag = 1;
            }
        }
    }
    // WallTime, TimePrediction.c:635-737
    if (S.wall) {
        WallEv w;
        if (wall_time(S, A.y, A.z, A.vy, A.vz, A.type, w, err)) take(best, S, w.t, w.pot, w.sub, SDMD_WALL, 0);
    }
    FPROF(prof, FPH_OTHER, pt);
    if (lane == 0) {
        G(S.evt)[i] = t + best.t;
        G(S.evpot)[i] = best.pot;
        G(S.evpc)[i] = best.pc;
        G(S.evp)[i] = best.partner;
        G(S.evtype)[i] = best.type;
        G(S.evsub)[i] = best.sub;
        G(S.nbnum)[i] = A.nbnum;
    }
}

// ---------------------------------------------------------------- events
__device__ void cell_remove(FSys &F, int a, int cell, int *err) {
    const int q = G(F.slot)[a];
    const int last = G(F.ccnt)[cell] - 1;
    if (q < 0 || q > last || last >= F.cap) { *err = FERR_SLOT; return; }
    const size_t base = (size_t)cell * F.cap;
    if (q != last) {
        const int m = G(F.cmem)[base + last];
        G(F.cmem)[base + q] = m;
        G(F.rec)[2 * (base + q)] = G(F.rec)[2 * (base + last)];
        G(F.rec)[2 * (base + q) + 1] = G(F.rec)[2 * (base + last) + 1];
        G(F.slot)[m] = q;
    }
    G(F.ccnt)[cell] = last;
}

__device__ void cell_insert(FSys &F, int a, int cell, int *err) {
    const int q = G(F.ccnt)[cell];
    if (q >= F.cap) { *err = ERR_CELLCAP; return; }
    G(F.cmem)[(size_t)cell * F.cap + q] = a;
    G(F.slot)[a] = q;
    G(F.ccnt)[cell] = q + 1;
}

// PBCandCrossCellEvent + PBC("part") (Events.c:207-272) on the cell arrays
__device__ void pcc_fast(FSys &F, int i, int *err) {
    Sys &S = F.s;
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
    const int oldc = cell_id(S, old[0], old[1], old[2]);
    int nw[3];
    for (int n = 0; n < 3; n++) {
        int v = (int)(c[n][i] / S.cellsize[n + 1]);
        if (v == S.cellnum[n + 1]) v--;
        if (v < 0 || v >= S.cellnum[n + 1]) { *err = ERR_CELL; return; }
        nw[n] = v;
    }
    for (int n = 0; n < 3; n++) ci[n][i] = nw[n];
    const int newc = cell_id(S, nw[0], nw[1], nw[2]);
    if (newc != oldc) {
        cell_remove(F, i, oldc, err);
        cell_insert(F, i, newc, err);
    }
}

// ThermostatEvent (Events.c:396-420, Andersen, no flow) with the device stream
__device__ void thermostat_fast(FSys &F, int i) {
    Sys &S = F.s;
    double sp[3];
    for (int n = 0; n < 3; n++) {
        int guard = 0;
        do {
            const double variance = S.T / G(S.mass)[i];
            sp[n] = fast_normal(F, i) * sqrt(variance) + 0;
        } while (sp[n] == 0 && ++guard < 8);
    }
    G(S.vx)[i] = sp[0]; G(S.vy)[i] = sp[1]; G(S.vz)[i] = sp[2];
}

// execute one popped event on lane 0 (DoEvent, Events.c:25-114, with the
// counter increments of SGThread.c:100-104); returns the renew count
// mirror record of atom a from values the caller holds (as put_record)
__device__ __forceinline__ void put_record_v(FV &F, double Te, int a, int cx, int cy, int cz, int slot, int type, double x,
                                             double y, double z, double vx, double vy, double vz, double t0) {
    SV &S = F.s;
    const size_t at = (size_t)cell_id(S, cx, cy, cz) * F.cap + slot;
    fvec4 r0, r1;
    r0.x = (float)(x - cx * S.cellsize[1]);
    r0.y = (float)(y - cy * S.cellsize[2]);
    r0.z = (float)(z - cz * S.cellsize[3]);
    r0.w = (float)(t0 - Te);
    r1.x = (float)vx;
    r1.y = (float)vy;
    r1.z = (float)vz;
    r1.w = __int_as_float((a << 8) | (type & 255));
    G(F.rec)[2 * at] = r0;
    G(F.rec)[2 * at + 1] = r1;
}

// one atom's state for a pair event, loaded at once
struct PairAtom {
    double x, y, z, vx, vy, vz, t0, m;
    long long c;
    int cx, cy, cz, slot, type;
};

__device__ __forceinline__ void pair_load(FV &F, int j, PairAtom &q) {
    SV &S = F.s;
    q.x = G(S.x)[j]; q.y = G(S.y)[j]; q.z = G(S.z)[j];
    q.vx = G(S.vx)[j]; q.vy = G(S.vy)[j]; q.vz = G(S.vz)[j];
    q.t0 = G(F.t0)[j]; q.m = G(S.mass)[j]; q.c = G(S.evc)[j];
    q.cx = G(S.cx)[j]; q.cy = G(S.cy)[j]; q.cz = G(S.cz)[j];
    q.slot = G(F.slot)[j]; q.type = G(S.type)[j];
}

// advance to t (as advance()) in registers, stored
__device__ __forceinline__ void pair_advance(FV &F, int j, PairAtom &q, double t) {
    SV &S = F.s;
    const double dt = t - q.t0;
    q.x = q.x + q.vx * dt;
    q.y = q.y + q.vy * dt;
    q.z = q.z + q.vz * dt;
    q.t0 = t;
    G(S.x)[j] = q.x; G(S.y)[j] = q.y; G(S.z)[j] = q.z;
    G(F.t0)[j] = t;
}

// A collision, bond or H-bond-neighbour event of atoms a and p (DoEvent ->
// InteractionEvent without its H-bond branch, Events.c:770-1025), with
// both atoms' state given (loaded with the selection) and the same
// arithmetic as exec_fast's general path (advance, PosLocal, image_near,
// interaction_event): both mirror records are written here.  Returns the
// renewed atoms (1 when the event is stale).
__device__ __forceinline__ int exec_pair(FSys &M, FV &F, int a, int p, int ty, double t, PairAtom &A, PairAtom &P,
                                         long long pca, double pot0, int sub0, int *renew, int *err) {
    SV &S = F.s;
    const double Te = M.Te;
    pair_advance(F, a, A, t);
    renew[0] = a;
    if (pca < P.c) {                                           // HazardCheck, SGThread.c:215-235
        cnt_add(M.s.recal, 1);
        put_record_v(F, Te, a, A.cx, A.cy, A.cz, A.slot, A.type, A.x, A.y, A.z, A.vx, A.vy, A.vz, A.t0);
        return 1;
    }
    if (P.t0 > t) {
        cnt_add(M.causal, 1);
        *err = FERR_CAUSAL;
    }
    pair_advance(F, p, P, t);
    // interaction_event: positions at t through the local-time view
    // (x + v (t - t0) with t0 = t) and the cell-based nearest image
    const double z0 = t - t;
    const double pi0 = A.x + A.vx * z0, pi1 = A.y + A.vy * z0, pi2 = A.z + A.vz * z0;
    double pj[3] = {P.x + P.vx * z0, P.y + P.vy * z0, P.z + P.vz * z0};
    const int ci[3] = {A.cx, A.cy, A.cz}, cj[3] = {P.cx, P.cy, P.cz};
    for (int n = 0; n < 3; n++) {
        if (ci[n] != cj[n]) {
            if (ci[n] == 0 && cj[n] == S.cellnum[n + 1] - 1) pj[n] -= S.box[n + 1];
            else if (ci[n] == S.cellnum[n + 1] - 1 && cj[n] == 0) pj[n] += S.box[n + 1];
        }
    }
    const double r1 = pi0 - pj[0], r2 = pi1 - pj[1], r3 = pi2 - pj[2];
    const double v1 = A.vx - P.vx, v2 = A.vy - P.vy, v3 = A.vz - P.vz;
    const double d2 = r1 * r1 + r2 * r2 + r3 * r3;
    const double b = r1 * v1 + r2 * v2 + r3 * v3;
    const double mu = A.m * P.m / (A.m + P.m);
    double pot = pot0;
    int s = 0;
    bool ok = true;
    switch (sub0) {
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
    default: *err = ERR_SUBTYPE; ok = false; break;
    }
    if (ok) {
        const double phi = (-1 * b + s * sqrt((b * b - 2 * d2 * pot / mu))) / ((A.m + P.m) * d2);
        if (isnan(phi)) {
            *err = ERR_PHI_NAN;
        } else {
            const double fi = P.m * phi, fj = A.m * phi;
            A.vx = A.vx + fi * r1; A.vy = A.vy + fi * r2; A.vz = A.vz + fi * r3;
            P.vx = P.vx - fj * r1; P.vy = P.vy - fj * r2; P.vz = P.vz - fj * r3;
            G(S.vx)[a] = A.vx; G(S.vy)[a] = A.vy; G(S.vz)[a] = A.vz;
            G(S.vx)[p] = P.vx; G(S.vy)[p] = P.vy; G(S.vz)[p] = P.vz;
        }
    }
    cnt_add(M.s.per_type[ty], 1);
    cnt_add(M.s.frame, 1);
    G(S.evc)[a] = A.c + 1;
    G(S.evc)[p] = P.c + 1;
    put_record_v(F, Te, a, A.cx, A.cy, A.cz, A.slot, A.type, A.x, A.y, A.z, A.vx, A.vy, A.vz, A.t0);
    put_record_v(F, Te, p, P.cx, P.cy, P.cz, P.slot, P.type, P.x, P.y, P.z, P.vx, P.vy, P.vz, P.t0);
    renew[1] = p;
    return 2;
}

// every other event (H-bond, thermostat, cell crossing, wall): about 1 % of
// them, kept out of line so that its registers do not count in the loop
__device__ __attribute__((noinline)) int exec_general(FSys &F, int a, int partner, double t, int *renew, int *err) {
    Sys &S = F.s;
    advance(F, a, t);
    renew[0] = a;
    if (partner && G(S.evpc)[a] < G(S.evc)[partner]) {          // HazardCheck, SGThread.c:215-235
        cnt_add(S.recal, 1);
        return 1;
    }
    if (partner) {
        if (G(F.t0)[partner] > t) {
            cnt_add(F.causal, 1);
            *err = FERR_CAUSAL;
        }
        advance(F, partner, t);
    }
    const int ty = G(S.evtype)[a];
    const PosLocal pos{F, t};
    switch (ty) {
    case SDMD_COLI: case SDMD_BOND: case SDMD_HBNE:
        interaction_event(S, pos, a, partner, 0, 0, err);
        break;
    case SDMD_HB: {
        const int nbi = G(S.hbnb)[a], nbj = G(S.hbnb)[partner];
        interaction_event(S, pos, a, partner, nbi, nbj, err);
        hb_event(S, a, partner, nbi, nbj, err);
        break;
    }
    case SDMD_THER: thermostat_fast(F, a); break;
    case SDMD_PCC: pcc_fast(F, a, err); break;
    case SDMD_WALL: {
        double vx = G(S.vx)[a], vy = G(S.vy)[a], vz = G(S.vz)[a];
        wall_event(S, G(S.y)[a], G(S.z)[a], vx, vy, vz, G(S.mass)[a], G(S.evpot)[a], G(S.evsub)[a], err);
        G(S.vx)[a] = vx; G(S.vy)[a] = vy; G(S.vz)[a] = vz;
        break;
    }
    default: *err = ERR_EVENTTYPE; return 1;
    }
    if (ty >= 0 && ty < 16) cnt_add(S.per_type[ty], 1);
    cnt_add(S.frame, 1);
    G(S.evc)[a]++;
    if (partner) G(S.evc)[partner]++;
    if (partner) { renew[1] = partner; return 2; }
    return 1;
}

// a selected event's record and the state of its atoms (P of the partner, or
// of the atom itself)
struct Pending {
    int a, p, ty, sub;           // p: partner, 0 = none
    double t, pot;
    long long pca;
    signed char ra, rp;          // roles
    PairAtom A, P;
};
__device__ __forceinline__ void pending_load(FV &F, int a, double t, Pending &e) {
    SV &S = F.s;
    const int p0 = G(S.evp)[a];
    e.a = a; e.t = t;
    e.ty = G(S.evtype)[a]; e.sub = G(S.evsub)[a]; e.pot = G(S.evpot)[a]; e.pca = G(S.evpc)[a];
    e.ra = G(S.role)[a];
    pair_load(F, a, e.A);
    e.p = (p0 > 0 && p0 <= S.N) ? p0 : 0;
    const int q = e.p ? e.p : a;
    e.rp = G(S.role)[q];
    pair_load(F, q, e.P);
}

__device__ __forceinline__ int exec_fast(FSys &M, FV &F, Pending &e, int *renew, int *err) {
    if (e.p && e.p != e.a && (e.ty == SDMD_COLI || e.ty == SDMD_BOND || e.ty == SDMD_HBNE))
        return exec_pair(M, F, e.a, e.p, e.ty, e.t, e.A, e.P, e.pca, e.pot, e.sub, renew, err);
    const int nr = exec_general(M, e.a, e.p, e.t, renew, err);
    put_record(F, M.Te, renew[0]);                     // the pair path writes its own records
    if (nr > 1) put_record(F, M.Te, renew[1]);
    return nr;
}

// ---------------------------------------------------------------- tree blocks
// Block b covers atoms 64b+1 .. 64b+64.  Returns its earliest event (t1,
// a1), the next one (t2, a2) and the third time t3.  An atom whose own event
// names a1 (or a2) as partner while a1's (a2's) names it back is the same
// pair event seen from the other side: the earlier one's execution
// re-predicts it, and the earlier one's independence test covers its atoms,
// so it is skipped when ranking.
//
// A wavefront scans four blocks at once, one per row of 16 lanes with four
// atoms per lane: the reductions stay inside rows (DPP moves only) and serve
// four blocks with the instructions that one block takes.
// Times are compared as two ordered unsigned words, high words first.
template <int CTRL>
__device__ __forceinline__ unsigned row_umin_step(unsigned v) {
    return min(v, (unsigned)__builtin_amdgcn_update_dpp(-1, (int)v, CTRL, 0xF, 0xF, false));
}
// the row's smallest word, in all its lanes (quad permutations, half-row and
// row mirrors)
__device__ __forceinline__ unsigned row_umin(unsigned v) {
    return row_umin_step<0x140>(row_umin_step<0x141>(row_umin_step<0x4E>(row_umin_step<0xB1>(v))));
}
struct RowScan {
    unsigned hi[4], lo[4];       // times of this lane's atoms as ordered words
    int k[4], p[4];              // atoms (0x7fffffff: none) and their partners
};
// the row's smallest time; with TAKE also its atom (the lowest on equal
// times), which leaves the scan with its mirror
template <bool TAKE>
__device__ __forceinline__ double row_first(RowScan &r, int &atom) {
    const unsigned H = row_umin(min(min(r.hi[0], r.hi[1]), min(r.hi[2], r.hi[3])));
    unsigned l = 0xffffffffu;
#pragma unroll
    for (int u = 0; u < 4; u++) l = min(l, r.hi[u] == H ? r.lo[u] : 0xffffffffu);
    const unsigned L = row_umin(l);
    if (TAKE) {
        unsigned a = 0x7fffffffu;
#pragma unroll
        for (int u = 0; u < 4; u++) a = min(a, (r.hi[u] == H && r.lo[u] == L) ? (unsigned)r.k[u] : 0x7fffffffu);
        const int K = (int)row_umin(a);
        unsigned q = 0xffffffffu;                // the atom's partner (one lane holds it)
#pragma unroll
        for (int u = 0; u < 4; u++) q = min(q, r.k[u] == K ? (unsigned)r.p[u] : 0xffffffffu);
        const int P = (int)row_umin(q);
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (r.k[u] == K || (r.k[u] == P && r.p[u] == K)) {
                order_words(__builtin_inf(), r.hi[u], r.lo[u]);
                r.k[u] = 0x7fffffff;
                r.p[u] = 0;
            }
        atom = K;
    }
    const unsigned s = (H >> 31) ? 0u : 0xffffffffu;             // order_words undone
    return __longlong_as_double((long long)(((unsigned long long)(H ^ (s | 0x80000000u)) << 32) | (L ^ s)));
}

// the earliest (t1, a1) and second (t2, a2) events of this row's block b that
// are not the mirror of an earlier one, and its third time t3 (b < 0: none)
__device__ __forceinline__ void block_scan4(FV &F, int b, double &t1, int &a1, double &t2, int &a2, double &t3) {
    const int l = threadIdx.x & 15, N = F.s.N;
    RowScan r;
    double t[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int a = b * 64 + 16 * u + l + 1;
        const bool in = b >= 0 && a <= N;
        const int q = in ? a : 1;
        t[u] = G(F.s.evt)[q];
        r.p[u] = G(F.s.evp)[q];
        r.k[u] = in ? a : 0x7fffffff;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        if (r.k[u] == 0x7fffffff) { t[u] = __builtin_inf(); r.p[u] = 0; }
        order_words(t[u], r.hi[u], r.lo[u]);
    }
    int none;
    t1 = row_first<true>(r, a1);
    t2 = row_first<true>(r, a2);
    t3 = row_first<false>(r, none);
}

// ---------------------------------------------------------------- helper workgroups
// A system's re-predictions of a round can be shared with helper workgroups
// on other CUs of the owner's XCD.  The owner workgroup publishes the
// round's jobs in global memory; every wavefront of the system's workgroups
// -- the owner's own included -- claims jobs from one word until none is
// left, and the owner waits for the count of completed jobs.  The owner
// never needs a helper (its own wavefronts take whatever is unclaimed), so
// the protocol cannot deadlock on a helper that is not resident.
//
// Ordering uses the XCD's shared L2: a workgroup reads its XCD from the
// hardware (XCC_ID), the owner records it in the job record, and a helper
// takes jobs only when it runs on that XCD.  Writes are published by waiting
// for them to complete (they write through the CU's L1 into the L2) before
// the agent-scope atomic that announces them; the reader, after the atomic
// that observes them, runs an agent-scope acquire (its L1 copies are
// dropped; a workgroup-scope invalidate does not drop lines other CUs
// wrote).  No L2 write-back is needed, as no other XCD takes part.
constexpr long long FHELP_IDLE = 1000000000LL;   // ticks (10 s at 100 MHz): a helper with no owner activity leaves
constexpr long long FJOB_WAIT = 200000000LL;     // ticks (2 s): the owner's bound on one round's predictions

// What helpers poll, what they count and what they read lie in cache lines of
// their own: with the done count beside the polled word a round of 64 systems
// of 1 536 atoms spent 2.7 us before a helper's prediction began and 3.5 us
// after the last one ended.
struct FJob {                   // one re-prediction: its time, the FP32 mirror's epoch, the atom
    double t, Te;
    int a, pad[3];
};
struct __attribute__((aligned(256))) FJobs {
    unsigned long long word;    // jobs of the round << 32 | next job index; JOB_STOP in the index: the owner has left
    unsigned long long pad0[31];
    int done;                   // helper jobs of the round completed, + JOB_FAILED for a failed one
    int pad1[63];
    int err;                    // first error of a helper's prediction
    int xcc;                    // the owner's XCD (-1: helpers stay out)
    int pad2[62];
    FJob job[2 * FSEL];
};
constexpr unsigned JOB_STOP = 0x80000000u;   // (a late claim's increments do not reach it)
constexpr int JOB_FAILED = 0x10000;

// helpers' statistics (the owner's live in FSys), summed by the host
struct FHelp {
    long long screens, confirms, pair_evals, candidates, validated, agree, causal;
    double max_screen_err, max_time_err;
};

__device__ __forceinline__ unsigned long long job_load(unsigned long long *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int int_load(int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// s_waitcnt vmcnt(0): this wave's vector-memory operations (its stores
// included) have completed in the L2.  Written as an asm statement with a
// memory clobber: the compiler neither moves memory operations across it nor
// drops it (the s_waitcnt builtin was found removed from the event loop by
// the wait-count pass, and it does not order memory operations)
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void acquire_agent() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent"); }
// the XCD this wavefront runs on (hwreg XCC_ID, bits 3:0)
__device__ __forceinline__ int xcc_id() { return __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 15; }

// claim the next unassigned job of the published round (-1: none left)
__device__ __forceinline__ int job_claim(FJobs *J) {
    const unsigned long long old = __hip_atomic_fetch_add(&J->word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return (unsigned)old < (unsigned)(old >> 32) ? (int)(unsigned)old : -1;
}

__device__ __forceinline__ void job_done(FJobs *J, bool failed) {
    __hip_atomic_fetch_add(&J->done, failed ? 1 + JOB_FAILED : 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------- shared memory
template <int W>
struct FShared {
    long long run_clock_end, run_count_end;   // the launch's bounds (thread 0)
    double window;                            // span of event times collected per round
    double b1[FMAXBLK], b2[FMAXBLK], b3[FMAXBLK];
    int ba[FMAXBLK], bb[FMAXBLK];
    double red_t[W], red_t1[W], red_t3[W];
    int red_a[W];
    double sel_t[FSEL];
    int sel_a[FSEL], sel_rank[FSEL];  // selected set: atom, number of earlier events in the set
    // per selected event: cells of target and partner (packed x<<20|y<<10|z),
    // whether it writes beyond its two atoms' state (cell crossing, H-bond),
    // their positions at the event time
    int pre_ca[FSEL], pre_cp[FSEL], pre_fl[FSEL];
    float pre_pa[FSEL][3], pre_pp[FSEL][3];
    unsigned long long conflict;
    int nset;                          // events in the selected set
    int nsel, nex, nren, nlight, next_ren, err, stop, drain;
    long long drain_end;
    // renewed atoms: H-bond-capable ones from the front (nren), the others
    // from the back (nlight)
    int ren_a[2 * FSEL];
    double ren_t[2 * FSEL];
    unsigned int dmask[FMAXBLK / 32];   // blocks touched this round (bit per block)
    FWave<flist(W)> w[W];
};

template <int W>
__device__ __forceinline__ void fsys_load(FSys &dst, const FSys *src) {
    const int n = (int)(sizeof(FSys) / sizeof(int));
    for (int k = threadIdx.x; k < n; k += 64 * W) ((int *)&dst)[k] = ((const int *)src)[k];
    __syncthreads();
}

template <int W>
__device__ __forceinline__ void fsys_store(FSys *dst, const FSys &src) {
    __syncthreads();
    const int n = (int)(sizeof(FSys) / sizeof(int));
    for (int k = threadIdx.x; k < n; k += 64 * W) ((int *)dst)[k] = ((const int *)&src)[k];
}

// FP32 mirror re-expressed at a new epoch (positions at Te, time offsets 0);
// the FP64 state is not touched
template <int W>
__device__ void rebase(FSys &M, FV &F, double Te) {
    __syncthreads();
    if (threadIdx.x == 0) { M.Te = Te; M.rebases++; }   // single writer between barriers
    __syncthreads();
    SV &S = F.s;
    for (int a = threadIdx.x + 1; a <= S.N; a += 64 * W) {
        const int cx = G(S.cx)[a], cy = G(S.cy)[a], cz = G(S.cz)[a];
        const size_t at = (size_t)cell_id(S, cx, cy, cz) * F.cap + G(F.slot)[a];
        const double dt = Te - G(F.t0)[a];
        fvec4 r0;
        r0.x = (float)((G(S.x)[a] + G(S.vx)[a] * dt) - cx * S.cellsize[1]);
        r0.y = (float)((G(S.y)[a] + G(S.vy)[a] * dt) - cy * S.cellsize[2]);
        r0.z = (float)((G(S.z)[a] + G(S.vz)[a] * dt) - cz * S.cellsize[3]);
        r0.w = 0.f;
        G(F.rec)[2 * at] = r0;
    }
    __syncthreads();
}


// ---------------------------------------------------------------- kernels
// bulk Predict(1..N) at the system time and the block minima
template <int W>
__device__ __forceinline__ void tab_load(ScrTab &dst, const void *src) {
    const int n = (int)(sizeof(ScrTab) / sizeof(int));
    for (int k = threadIdx.x; k < n; k += 64 * W) ((int *)&dst)[k] = ((const int *)src)[k];
    __syncthreads();
}

#ifndef SDMD_FAST_WAVES
// cell arrays from the reference's linked lists (list order), every cell
__global__ __launch_bounds__(256) void k_fast_cells(FSys *systems) {
    FSys &F = systems[blockIdx.x];
    const Sys &S = F.s;
    for (int c = 1 + blockIdx.y * 256 + threadIdx.x; c <= F.ncell; c += 256 * gridDim.y) {
        int q = 0;
        for (int a = G(S.celllist)[S.N + c]; a && q < F.cap; a = G(S.celllist)[a], q++) {
            G(F.cmem)[(size_t)c * F.cap + q] = a;
            G(F.slot)[a] = q;
        }
        G(F.ccnt)[c] = q;
    }
}

// bond lists at a fixed stride of 16 (BondTime's connect[16]), connection
// rows as bytes and the constraints' tables: FP32 radii and energy bits inline (up to 8 steps are
// staged) and FP64 shells at a fixed stride (a constraint of more steps than
// a row holds is not staged, and then not read from here).  Derived on the
// device: 20 MB for 26 080 atoms, which took longer to write on the host and
// to copy than all the rest of opening a system.
__global__ __launch_bounds__(256) void k_fast_derive(FSys *systems) {
    FV &F = fixed_view(systems + blockIdx.x);
    SV &S = F.s;
    const int tid = blockIdx.y * 256 + threadIdx.x, all = 256 * gridDim.y, N = S.N;
    for (int k = tid; k < (N + 1) * 16; k += all) {
        const int a = k >> 4, e = a > 0 ? G(S.bond_off)[a] + (k & 15) : 0;
        const bool in = a > 0 && e < G(S.bond_off)[a + 1];
        G(F.bj16)[k] = in ? G(S.bond_j)[e] : 0;
        G(F.blo16)[k] = in ? G(S.bond_dmin)[e] : 0.0;
        G(F.bhi16)[k] = in ? G(S.bond_dmax)[e] : 0.0;
    }
    // an atom's connection row as bytes over its span (row and span small
    // enough; otherwise it is searched in memory): bits 0-1 BOND and
    // CONSTRAINT, bits 2-6 the slot + 1 of a constraint that is staged
    for (int a = tid; a <= N; a += all) {
        const int o = a > 0 ? G(S.cmap_off)[a] : 0, n = a > 0 ? G(S.cmap_off)[a + 1] - o : 0;
        const int lo = n > 0 ? G(S.cmap_j)[o] : 0, hi = n > 0 ? G(S.cmap_j)[o + min(n, 64) - 1] : 0;
        const bool fits = n <= 64 && hi - lo < FCONN;
        for (int k = 0; k < FCONN / 4; k++) G(F.conn)[a * (FCONN / 4) + k] = 0;
        G(F.rowlo)[a] = fits ? lo : -1;
        unsigned char *bytes = (unsigned char *)(F.conn + a * (FCONN / 4));
        const int co = a > 0 ? G(S.con_off)[a] : 0;
        for (int k = o; fits && k < o + n; k++) {
            const int rc = G(S.cmap_con)[k], slot = rc - co;              // rc < 0: no constraint
            const bool staged = rc >= 0 && slot >= 0 && slot < FCON && G(S.con)[max(rc, 0)].nstep <= FCONSTEP;
            G(bytes)[G(S.cmap_j)[k] - lo] = (unsigned char)((G(S.cmap_bits)[k] & (SDMD_BOND_CONNECT | SDMD_CONSTRAINT_CONNECT)) |
                                                            (staged ? (slot + 1) << 2 : 0));
        }
    }
    const int nc = G(S.con_off)[N + 1];
    for (int k = tid; k < nc; k += all) {
        const int step0 = G(S.con)[k].step0, nstep = min((int)G(S.con)[k].nstep, FCONSTEP);
        double *row = F.crow + (size_t)k * (2 + 2 * FCONSTEP);
        G(row)[0] = G(S.con)[k].dmin;
        G(row)[1] = G(S.con)[k].dmax;
        unsigned ez = 0;
        for (int q = 0; q < FCONSTEP; q++) {
            const double dq = q < nstep ? G(S.sd)[step0 + q] : 0.0, eq = q < nstep ? G(S.se)[step0 + q] : 0.0;
            G(row)[2 + q] = dq;
            G(row)[2 + FCONSTEP + q] = eq;
            G(F.crad)[k].rad[q] = (float)dq;
            if (q < nstep && eq == 0) ez |= 1u << q;
        }
        G(F.crad)[k].ez = ez;
        G(F.crad)[k].dmin = (float)G(S.con)[k].dmin;
        G(F.crad)[k].dmax = (float)G(S.con)[k].dmax;
        G(F.crad)[k].nstep = G(S.con)[k].nstep;
    }
}

// linked cell lists from the cell arrays of one system, for a download
__global__ __launch_bounds__(256) void k_fast_lists(FSys *systems, int sys) {
    FSys &F = systems[sys];
    const Sys &S = F.s;
    for (int c = 1 + blockIdx.x * 256 + threadIdx.x; c <= F.ncell; c += 256 * gridDim.x) {
        int head = 0;
        for (int q = G(F.ccnt)[c] - 1; q >= 0; q--) {
            const int a = G(F.cmem)[(size_t)c * F.cap + q];
            G(S.celllist)[a] = head;
            head = a;
        }
        G(S.celllist)[S.N + c] = head;
    }
}

// mirror records of every atom, before the bulk prediction reads them
__global__ __launch_bounds__(256) void k_fast_records(FSys *systems) {
    FV &F = fixed_view(systems + blockIdx.x);
    for (int a = 1 + blockIdx.y * 256 + threadIdx.x; a <= F.s.N; a += 256 * gridDim.y) put_record(F, F.Te, a);
}

// Bulk Predict(1..N): a prediction reads positions, velocities and counters
// but no other atom's event record, so the atoms are spread over gridDim.y
// workgroups per system (one wavefront per atom at a time).  Bound by the
// instruction count of a prediction (about 9 us on one wavefront); with
// one workgroup per system a 26 080-atom system took 58 ms on one CU.
template <int W, bool VAL>
__global__ __launch_bounds__(64 * W) void k_fast_predict(FSys *systems) {
    __shared__ FSys Fl;
    __shared__ FWave<flist(W)> w[W];
    __shared__ ScrTab tab;
    FSys &Fg = systems[blockIdx.x];
    FV &C = fixed_view(systems + blockIdx.x);
    fsys_load<W>(Fl, &Fg);
    tab_load<W>(tab, Fl.scrtab);
    FSys &F = Fl;
    Sys &S = F.s;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    if (tid == 0) {                         // statistics of this workgroup only
        F.validated = F.agree = F.causal = 0;
        F.max_screen_err = F.max_time_err = 0;
    }
    __syncthreads();
    WStats &ws = w[wave].st;                // in LDS: no registers held across the loop
    ws.screen = ws.conf = ws.fp64 = ws.cand = 0;
    wave_sync();
    int err = 0;
    for (int i = 1 + blockIdx.y * W + wave; i <= S.N; i += W * gridDim.y) {
        predict_fast<4, VAL>(F, C, nullptr, tab, w[wave], i, G(F.t0)[i], ws, &err);
        if (__ballot(err != 0)) break;              // uniform across the wave
    }
    if (err) atomicCAS(&Fg.s.error, 0, err);
    if (lane == 0) {
        cnt_add(Fg.screens, ws.screen);
        cnt_add(Fg.confirms, ws.conf);
        cnt_add(Fg.s.pair_evals, ws.fp64 + ws.conf);
        cnt_add(Fg.s.candidates, ws.cand);
    }
    __syncthreads();
    if (tid == 0) {
        if (F.validated) cnt_add(Fg.validated, F.validated);
        if (F.agree) cnt_add(Fg.agree, F.agree);
        if (F.causal) cnt_add(Fg.causal, F.causal);
        cnt_max(Fg.max_screen_err, F.max_screen_err);
        cnt_max(Fg.max_time_err, F.max_time_err);
    }
}

// the block minima of every system, four 64-atom blocks per wavefront
__global__ __launch_bounds__(256) void k_fast_blocks(FSys *systems) {
    FV &F = fixed_view(systems + blockIdx.x);
    for (int b0 = 4 * (blockIdx.y * 4 + (threadIdx.x >> 6)); b0 < F.nblk; b0 += 16 * gridDim.y) {
        const int b = b0 + ((threadIdx.x & 63) >> 4);
        double t1, t2, t3;
        int a1, a2;
        block_scan4(F, b < F.nblk ? b : -1, t1, a1, t2, a2, t3);
        if ((threadIdx.x & 15) == 0 && b < F.nblk) {
            G(F.b1)[b] = t1; G(F.ba)[b] = a1; G(F.b2)[b] = t2; G(F.bb)[b] = a2; G(F.b3)[b] = t3;
        }
    }
}

// CalKinetE + CalPotenE (ToolFunctions.c:626-752) of every system at its
// snapshot time T (the earliest pending event, the time a download reports):
// positions are x + v (T - t0); one wavefront per atom i, two lanes per
// neighbour cell, for partners j > i.  A chain of dependent loads per pair
// bounds it, so the atoms are spread over the GPU: gridDim.y workgroups per
// system, each leaving its sums in `part` (k_energy_reduce adds them).  One
// workgroup per system with one thread per atom took 4.0 ms for 64 systems of
// 1 536 atoms.
__global__ __launch_bounds__(64 * EWAVES) void k_fast_energy(FSys *systems, double *part) {
    const FSys &F = systems[blockIdx.x];
    const Sys &S = F.s;
    const int tid = threadIdx.x, lane = tid & 63;
    double tm = __builtin_inf();
    for (int b = lane; b < F.nblk; b += 64) tm = fmin(tm, G(F.b1)[b]);
    double T = wave_min_d(tm);
    if (!(T < INFINIT)) T = F.tlast;
    const int N = S.N;
    const double cut2 = S.cutoffr * S.cutoffr;
    const int c = min(lane >> 1, 26);
    Sum2 ke = {0, 0}, pe = {0, 0};
    int err = 0;
    for (int i = 1 + blockIdx.y * EWAVES + (tid >> 6); i <= N; i += EWAVES * gridDim.y) {
        const double dti = T - G(F.t0)[i];
        const double vi[3] = {G(S.vx)[i], G(S.vy)[i], G(S.vz)[i]};
        const double xi = G(S.x)[i] + vi[0] * dti, yi = G(S.y)[i] + vi[1] * dti, zi = G(S.z)[i] + vi[2] * dti;
        if (lane == 0) ke.add(0.5 * G(S.mass)[i] * (vi[0] * vi[0] + vi[1] * vi[1] + vi[2] * vi[2]));
        int cc[3] = {G(S.cx)[i] + c_OX[c], G(S.cy)[i] + c_OY[c], G(S.cz)[i] + c_OZ[c]};
        double sh[3] = {0, 0, 0};
        for (int k = 0; k < 3; k++) {
            if (cc[k] < 0) { cc[k] = S.cellnum[k + 1] - 1; sh[k] = -1 * S.box[k + 1]; }
            else if (cc[k] >= S.cellnum[k + 1]) { cc[k] = 0; sh[k] = S.box[k + 1]; }
        }
        const int cell = cell_id(S, cc[0], cc[1], cc[2]);
        const int cnt = lane < 54 ? min(G(F.ccnt)[cell], F.cap) : 0;
        for (int q = lane & 1; q < cnt; q += 2) {
            const int j = G(F.cmem)[(size_t)cell * F.cap + q];
            if (j <= i || j > N) continue;
            const double dtj = T - G(F.t0)[j];
            const double vj[3] = {G(S.vx)[j], G(S.vy)[j], G(S.vz)[j]};
            const double xj = G(S.x)[j] + vj[0] * dtj, yj = G(S.y)[j] + vj[1] * dtj, zj = G(S.z)[j] + vj[2] * dtj;
            const double r1 = xi - (xj + sh[0]), r2 = yi - (yj + sh[1]), r3 = zi - (zj + sh[2]);
            const double rr = r1 * r1 + r2 * r2 + r3 * r3;
            if (rr > cut2) continue;
            pe.add(pair_energy(S, i, j, r1, r2, r3, rr, vi, vj, &err));
        }
    }
    energy_partial(ke, pe, err || S.error, part);
}

#endif  // SDMD_FAST_WAVES

// A helper workgroup: its wavefronts claim the owner's published jobs
// (re-predictions) until the owner stops, then add their statistics to hp.
template <int W, int FQ, bool VAL>
__device__ __forceinline__ void helper_loop(FSys &F, FV &C, const ScrTab &tab, FShared<W> &sh, FJobs *J, FHelp *hp, int xcc) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    WStats &ws = sh.w[wave].st;             // in LDS: no registers held across the loop
    ws.screen = ws.conf = ws.fp64 = ws.cand = 0;
    wave_sync();
    int near = -1;                               // 1: on the owner's XCD (fixed for the launch, set before any job)
    for (;;) {
        int q = -1, quit = 0;
        if (lane == 0) {
            long long idle0 = (long long)wall_clock64();
            for (;;) {
                const unsigned long long w = job_load(&J->word);
                if ((unsigned)w < (unsigned)(w >> 32)) {
                    if (near < 0) near = int_load(&J->xcc) == xcc;
                    if (!near) { quit = 1; break; }
                    q = job_claim(J);
                    if (q >= 0) break;
                    continue;
                }
                if ((unsigned)w & JOB_STOP) { quit = 1; break; }
                if ((long long)wall_clock64() - idle0 > FHELP_IDLE) { quit = 1; break; }
                __builtin_amdgcn_s_sleep(2);
            }
        }
        q = lane_get(q, 0);
        quit = lane_get(quit, 0);
        if (quit) break;
        acquire_agent();                         // drop stale L1 lines: the owner's writes, from the L2
        const int a = J->job[q].a;
        const double t = J->job[q].t, Te = J->job[q].Te;
        if (lane == 0) F.Te = Te;                // every wave of the round writes the same epoch
        int err = 0;
        predict_fast<FQ, VAL>(F, C, nullptr, tab, sh.w[wave], a, t, ws, &err);
        const bool failed = __ballot(err != 0) != 0;
        if (err) atomicCAS(&J->err, 0, err);
        wait_stores();                           // the event record is in the L2 before the count
        if (lane == 0) job_done(J, failed);
    }
    if (lane == 0) {
        atomicAdd((unsigned long long *)&hp->screens, (unsigned long long)ws.screen);
        atomicAdd((unsigned long long *)&hp->confirms, (unsigned long long)ws.conf);
        atomicAdd((unsigned long long *)&hp->pair_evals, (unsigned long long)(ws.fp64 + ws.conf));
        atomicAdd((unsigned long long *)&hp->candidates, (unsigned long long)ws.cand);
    }
    __syncthreads();
    if (tid == 0) {
        atomicAdd((unsigned long long *)&hp->validated, (unsigned long long)F.validated);
        atomicAdd((unsigned long long *)&hp->agree, (unsigned long long)F.agree);
        atomicAdd((unsigned long long *)&hp->causal, (unsigned long long)F.causal);
        cnt_max(hp->max_screen_err, F.max_screen_err);
        cnt_max(hp->max_time_err, F.max_time_err);
    }
}

// the event loop: rounds of concurrent independent events until `npops`
// pops are done or the device clock passes `budget` ticks (100 MHz).
// Workgroup b serves system (b % 8) + 8 * ((b / 8) / (1 + H)) as owner
// (role 0) or helper (roles 1..H), so with round-robin dispatch over the 8
// XCDs all workgroups of a system share one XCD's L2.
template <int W, int FQ, bool VAL>
__global__ __launch_bounds__(64 * W) void k_fast_run(FSys *systems, FJobs *jobs, FHelp *help, int nsys, int H,
                                                     long long npops, long long budget, double t_end) {
    __shared__ FSys Fl;
    __shared__ FShared<W> sh;
    __shared__ ScrTab tab;
    const int sys = (blockIdx.x & 7) + 8 * ((blockIdx.x >> 3) / (H + 1));
    const int role = (blockIdx.x >> 3) % (H + 1);
    if (sys >= nsys) return;                     // uniform per workgroup
    FJobs *J = jobs + sys;
    fsys_load<W>(Fl, &systems[sys]);
    if (threadIdx.x == 0) Fl.t_stop = t_end;
    tab_load<W>(tab, Fl.scrtab);
    FSys &F = Fl;
    FV &C = fixed_view(systems + sys);
    Sys &M = F.s;                              // counters
    SV &S = C.s;
    unsigned long long *const prof = S.prof;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int xcc = xcc_id();
    if (role > 0) {
        if (tid == 0) {                          // statistics of this helper only; no phase clocks
            F.validated = F.agree = F.causal = 0;
            F.max_screen_err = F.max_time_err = 0;
        }
        __syncthreads();
        helper_loop<W, FQ, VAL>(F, C, tab, sh, J, help + sys, xcc);
        return;
    }
    if (H > 0 && tid == 0) {                     // helpers on this XCD may join
        __hip_atomic_store(&J->xcc, xcc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        wait_stores();
    }
    const int nblk = C.nblk;
    for (int b = tid; b < nblk; b += 64 * W) {
        sh.b1[b] = G(C.b1)[b]; sh.b2[b] = G(C.b2)[b]; sh.b3[b] = G(C.b3)[b];
        sh.ba[b] = G(C.ba)[b]; sh.bb[b] = G(C.bb)[b];
    }
    if (tid == 0) { sh.err = M.error; sh.stop = 0; sh.drain = 0; }
    if (tid < FMAXBLK / 32) sh.dmask[tid] = 0;
    __syncthreads();
    if (tid == 0) {                       // npops < 0: -npops executed events
        sh.window = __builtin_inf();
        sh.run_clock_end = (long long)wall_clock64() + budget;
        sh.run_count_end = npops < 0 ? M.frame - npops : M.pops + npops;
    }
    WStats &ws = sh.w[wave].st;             // in LDS: no registers held across the loop
    ws.screen = ws.conf = ws.fp64 = ws.cand = 0;
    wave_sync();
    const int cap = C.max_batch > 0 ? min(C.max_batch, FSEL) : FSEL;
    const bool small = nblk <= FSMALL;
    // A run of a number of pops or events ends with the round that reaches
    // it, so its rounds keep their sets; a run up to a time has the same
    // result whatever they are.
    const bool wide = !small && llabs(npops) >= (1LL << 32);
    unsigned long long pt = prof ? wall_clock64() : 0;
    while (true) {
        // ---- selection: every event earlier than the smallest third time of
        // any block (each block's two earliest), or, when that set is too
        // large, earlier than the smallest second time (each block's earliest)
        //
        // Wavefront 0 collects the set, loads the events' atoms, tests their
        // independence and executes them, one event per lane, with the loaded
        // state in registers: a barrier or a hand-over through LDS costs as
        // much as 50 instructions.  Up to FSMALL blocks (few events) no other
        // wavefront takes part before the re-predictions; of more blocks the
        // scans and the pair tests are spread over the workgroup.
        double m3 = __builtin_inf(), m2 = __builtin_inf(), m1 = __builtin_inf();
        int a1 = 0x7fffffff;
        for (int b = small ? lane : tid; b < nblk; b += small ? 64 : 64 * W) {
            m3 = fmin(m3, sh.b3[b]);
            m2 = fmin(m2, sh.b2[b]);
            const double t = sh.b1[b];
            if (t < m1 || (t == m1 && sh.ba[b] < a1)) { m1 = t; a1 = sh.ba[b]; }
        }
        m3 = wave_min_d(m3);
        if (!small) m2 = wave_min_d(m2);                      // only needed where a set can be too large
        wave_argmin(m1, a1);
        const double tcap = nextafter(F.t_stop, __builtin_inf());
        double theta = fmin(m2, tcap), theta3 = fmin(m3, tcap), tmin = m1;
        int amin = a1;
        if (!small) {
            if (lane == 0) { sh.red_t[wave] = m2; sh.red_t3[wave] = m3; sh.red_t1[wave] = m1; sh.red_a[wave] = a1; }
            __syncthreads();
            for (int w = 0; w < W; w++) {
                theta = fmin(theta, sh.red_t[w]);
                theta3 = fmin(theta3, sh.red_t3[w]);
                if (sh.red_t1[w] < tmin || (sh.red_t1[w] == tmin && sh.red_a[w] < amin)) { tmin = sh.red_t1[w]; amin = sh.red_a[w]; }
            }
        }
        FPROF(prof, FPH_SCAN, pt);
        const bool old_epoch = tmin - F.Te > C.rebase_dt;     // uniform
        if (tid == 0) {
            // Once the pop or time budget is spent, drain: execute what is
            // still pending up to the latest executed time, so that every
            // atom's local time is at most that time and every pending event
            // is later -- the state is then a snapshot at one time.
            const bool spent = (npops < 0 ? M.frame : M.pops) >= sh.run_count_end;
            if (!sh.drain && (spent || (long long)wall_clock64() > sh.run_clock_end)) {
                sh.drain = 1;
                if (F.tlast < F.t_stop) F.t_stop = F.tlast;
                sh.drain_end = M.pops + FDRAIN;
            }
            const bool pending = tmin < INFINIT && tmin <= F.t_stop;
            if (sh.drain && M.pops >= sh.drain_end && pending && !sh.err) sh.err = FERR_DRAIN;
            if (sh.err || !pending || amin < 1 || amin > S.N || (sh.drain && M.pops >= sh.drain_end))
                sh.stop = 1;
            sh.nsel = 0;
            sh.next_ren = 0;
            sh.conflict = 0;
        }
        if (!small || old_epoch) {
            __syncthreads();
            if (sh.stop) break;
            if (old_epoch) rebase<W>(F, C, tmin);
        }
        // collect the prefix set
        if (small) {                                          // at most 2 * FSMALL events: no overflow
            wave_sync();
            if (wave == 0 && !sh.stop) {
                const int b = min(lane, nblk - 1);
                const double u1 = sh.b1[b], u2 = sh.b2[b];
                const bool in1 = lane < nblk && u1 < theta3, in2 = lane < nblk && u2 < theta3;
                const unsigned long long k1 = __ballot(in1), k2 = __ballot(in2), below = (1ull << lane) - 1;
                const int n1 = __popcll(k1), s1 = __popcll(k1 & below), s2 = n1 + __popcll(k2 & below);
                if (in1) { sh.sel_t[s1] = u1; sh.sel_a[s1] = sh.ba[b]; }
                if (in2) { sh.sel_t[s2] = u2; sh.sel_a[s2] = sh.bb[b]; }
                if (lane == 0) sh.nsel = n1 + __popcll(k2);
            }
            wave_sync();
        } else {
            auto collect = [&](double before, bool second) {
                for (int b = tid; b < nblk; b += 64 * W) {
                    if (sh.b1[b] < before) {
                        const int slotk = atomicAdd(&sh.nsel, 1);
                        if (slotk < FSEL) { sh.sel_t[slotk] = sh.b1[b]; sh.sel_a[slotk] = sh.ba[b]; }
                    }
                    if (second && sh.b2[b] < before) {
                        const int slotk = atomicAdd(&sh.nsel, 1);
                        if (slotk < FSEL) { sh.sel_t[slotk] = sh.b2[b]; sh.sel_a[slotk] = sh.bb[b]; }
                    }
                }
            };
            // Any time up to theta3 bounds a prefix of the event order.  Where
            // that of theta3 is too large (more than about 200 blocks), the
            // events of a window of time are taken that holds about FSEL_AIM
            // of them, the window following the counts seen: a round costs
            // 20 us beside its predictions, and the blocks' second times,
            // the other bound at hand, leave only 27 events of 408 blocks.
            const double reach = wide ? fmin(theta3, tmin + sh.window) : theta3;
            collect(reach, true);
            __syncthreads();
            int found = sh.nsel;
            if (wide) {
                double w = sh.window;
                if (found > FSEL) {
                    __syncthreads();
                    const double fit = (double)FSEL_AIM / found, span = reach - tmin;
                    // the counts scatter: the window shrinks no faster than it grows
                    w = w < 1e300 ? span * fmax(fit, 0.8) : span * fit;
                    if (tid == 0) sh.nsel = 0;
                    __syncthreads();
                    collect(fmax(theta, tmin + span * fit), true);
                    __syncthreads();
                    found = sh.nsel;
                } else if (reach < theta3) {                  // the window was the bound
                    w *= fmin(fmax((double)FSEL_AIM / max(found, 1), 0.8), 1.25);
                }
                if (tid == 0) sh.window = w;                  // read next after the coming barriers
            }
            if (found > FSEL) {
                __syncthreads();
                if (tid == 0) sh.nsel = 0;
                __syncthreads();
                collect(theta, false);
                __syncthreads();
            }
        }
        FPROF(prof, FPH_COLLECT, pt);
        int ns = 0;
        Pending ev;
        ev.a = 0x7fffffff;
        ev.ra = ev.rp = 0;
        ev.t = __builtin_inf();
        if (wave == 0 && !sh.stop) {
            ns = sh.nsel;
            const bool single = (ns == 0 || ns > FSEL);
            if (single) {
                if (lane == 0) { ev.t = tmin; ev.a = amin; }
                ns = 1;
            } else if (lane < ns) {
                ev.t = sh.sel_t[lane]; ev.a = sh.sel_a[lane];
            }
            // cells, kind and positions (at the event time) of each event's
            // target and partner, for the independence test
            if (lane < ns && ev.a >= 1 && ev.a <= S.N) {
                pending_load(C, ev.a, ev.t, ev);
                sh.pre_ca[lane] = (ev.A.cx << 20) | (ev.A.cy << 10) | ev.A.cz;
                sh.pre_cp[lane] = (ev.P.cx << 20) | (ev.P.cy << 10) | ev.P.cz;
                sh.pre_fl[lane] = (ev.ty == SDMD_PCC || ev.ty == SDMD_HB) ? 1 : 0;
                const double da = ev.t - ev.A.t0, dp = ev.t - ev.P.t0;
                sh.pre_pa[lane][0] = (float)(ev.A.x + ev.A.vx * da);
                sh.pre_pa[lane][1] = (float)(ev.A.y + ev.A.vy * da);
                sh.pre_pa[lane][2] = (float)(ev.A.z + ev.A.vz * da);
                sh.pre_pp[lane][0] = (float)(ev.P.x + ev.P.vx * dp);
                sh.pre_pp[lane][1] = (float)(ev.P.y + ev.P.vy * dp);
                sh.pre_pp[lane][2] = (float)(ev.P.z + ev.P.vz * dp);
            }
            sh.sel_a[lane] = ev.a;
            sh.sel_t[lane] = ev.t;
            sh.sel_rank[lane] = 0;
            if (lane == 0) {
                sh.nset = ns;
                F.batches++;
                if (single) F.single++;
            }
        }
        if (small) wave_sync();
        else __syncthreads();
        // independence: every pair of the set, spread over the workgroup (no
        // sorting: the pair's time order is compared directly); the later
        // event k of a pair conflicts with the earlier one l when an atom of
        // l lies within D - 1 cells (Chebyshev, periodic) of an atom of k
        // -- D = 2, so neither event's predictions read the other's atoms;
        // D = 3 when either writes beyond its atoms' state (a cell crossing
        // moves an atom into a neighbouring cell, an H-bond event rewrites
        // its neighbours' bookkeeping) -- or when the two atoms are closer
        // than two cell widths (>= twice the cut-off, so an event created by
        // one cannot reach the other's atoms through a single partner)
        if (!small || wave == 0) {
            const int nset = small ? ns : sh.nset;
            const int npair = nset * (nset - 1) / 2;
            const int n1 = S.cellnum[1], n2 = S.cellnum[2], n3 = S.cellnum[3];
            const float bx = (float)S.box[1], by = (float)S.box[2], bz = (float)S.box[3];
            const float cmin = (float)fmin(S.cellsize[1], fmin(S.cellsize[2], S.cellsize[3]));
            const float R2 = 4.f * cmin * cmin;
            const float ix = 1.f / bx, iy = 1.f / by, iz = 1.f / bz;
            unsigned long long mine = 0;
            for (int q = small ? lane : tid; q < npair; q += small ? 64 : 64 * W) {
                int i = (int)((1.f + sqrtf(1.f + 8.f * (float)q)) * 0.5f);
                while (i * (i - 1) / 2 > q) i--;
                while ((i + 1) * i / 2 <= q) i++;
                const int j = q - i * (i - 1) / 2;
                const bool jfirst = sh.sel_t[j] < sh.sel_t[i] || (sh.sel_t[j] == sh.sel_t[i] && sh.sel_a[j] < sh.sel_a[i]);
                const int k = jfirst ? i : j, l = jfirst ? j : i;      // l is the earlier event
                if (nset > cap) atomicAdd(&sh.sel_rank[k], 1);
                const int D = 2 + ((sh.pre_fl[k] | sh.pre_fl[l]) ? 1 : 0);
                auto far = [&](int u, int v) {
                    int dx = abs((u >> 20) - (v >> 20)), dy = abs(((u >> 10) & 1023) - ((v >> 10) & 1023)),
                        dz = abs((u & 1023) - (v & 1023));
                    dx = min(dx, n1 - dx); dy = min(dy, n2 - dy); dz = min(dz, n3 - dz);
                    return max(dx, max(dy, dz)) >= D;
                };
                auto apart = [&](const float *u, const float *v) {      // minimum image
                    float dx = u[0] - v[0], dy = u[1] - v[1], dz = u[2] - v[2];
                    dx -= bx * rintf(dx * ix);
                    dy -= by * rintf(dy * iy);
                    dz -= bz * rintf(dz * iz);
                    return dx * dx + dy * dy + dz * dz >= R2;
                };
                const int ka = sh.pre_ca[k], kp = sh.pre_cp[k], la = sh.pre_ca[l], lp = sh.pre_cp[l];
                const float *xka = sh.pre_pa[k], *xkp = sh.pre_pp[k], *xla = sh.pre_pa[l], *xlp = sh.pre_pp[l];
                const bool indep = far(ka, la) && far(ka, lp) && far(kp, la) && far(kp, lp) &&
                                   apart(xka, xla) && apart(xka, xlp) && apart(xkp, xla) && apart(xkp, xlp);
                if (!indep) mine |= 1ull << k;
            }
            mine = wave_or64(mine);
            if (lane == 0 && mine) atomicOr(&sh.conflict, mine);
        }
        if (small) wave_sync();
        else __syncthreads();
        FPROF(prof, FPH_SELECT, pt);
        // ---- execution: the independent events among the `cap` earliest of
        // the set, one lane per event
        int err = 0;
        if (wave == 0) {
            const bool ok = lane < ns && ev.a >= 1 && ev.a <= S.N && !((sh.conflict >> lane) & 1) && sh.sel_rank[lane] < cap;
            const int nex = __popcll(__ballot(ok));
            if (lane == 0) {
                sh.nex = nex;
                F.deferred += ns - nex;
            }
            int renew[2] = {0, 0}, nr = 0;
            if (ok) nr = exec_fast(F, C, ev, renew, &err);
            // H-bond-capable atoms (acceptor, donor, sulfur) scan their
            // neighbourhood for H-bond partners: the longest predictions of a
            // round, queued first so the waves finish together
            const unsigned long long below = (1ull << lane) - 1;
            int nh = 0, nl = 0;
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const signed char ro = r ? ev.rp : ev.ra;        // renew[1] is the partner
                const bool heavy = ro == 'A' || ro == 'D' || ro == 'S';
                const unsigned long long mh = __ballot(r < nr && heavy), ml = __ballot(r < nr && !heavy);
                if (r < nr) {
                    const int slot = heavy ? nh + __popcll(mh & below) : 2 * FSEL - 1 - (nl + __popcll(ml & below));
                    sh.ren_a[slot] = renew[r];
                    sh.ren_t[slot] = ev.t;
                }
                nh += __popcll(mh);
                nl += __popcll(ml);
            }
            if (lane == 0) { sh.nren = nh; sh.nlight = nl; }
            const double last = -wave_min_d(ok ? -ev.t : __builtin_inf());
            if (lane == 0 && nex > 0 && F.tlast < last) F.tlast = last;
        }
        if (err) atomicCAS(&sh.err, 0, err);
        __syncthreads();
        if (sh.stop) break;
        const int nex = sh.nex;
        if (nex < 1) {                                     // no selectable event: stop with an error
            if (tid == 0) sh.err = FERR_SELECT;
            break;
        }
        FPROF(prof, FPH_EVENT, pt);
        // re-prediction of every renewed atom, one wave per atom; a wave takes
        // the next atom when it finishes one (prediction times vary)
        const int nheavy = sh.nren, nlight = sh.nlight;
        const int nren = nheavy + nlight;             // <= 2 * nex <= 2 * FSEL: the two ends do not meet
        auto ren_at = [&](int r) { return r < nheavy ? r : 2 * FSEL - nlight + (r - nheavy); };
        err = 0;
        // Jobs 0 .. W - 1 are the owner's wavefronts' own; the others are
        // published for the helpers and for owner wavefronts that finish
        // early.  A round with no more jobs than wavefronts stays on this CU:
        // nothing is published or waited for (59 atoms: 14.2 -> 11.2 us per
        // round's predictions).
        const bool shared = H > 0 && nren > W;
        if (shared) {
            for (int r = tid; r < nren; r += 64 * W) {
                const int q = ren_at(r);
                J->job[r].a = sh.ren_a[q];
                J->job[r].t = sh.ren_t[q];
                J->job[r].Te = F.Te;
            }
            if (tid == 0) J->done = 0;
            // the barrier does not wait for other wavefronts' stores: each
            // wave waits for its own (event execution, job list) to complete
            // in the L2 before the word announces the round
            wait_stores();
            __syncthreads();
            if (tid == 0)
                __hip_atomic_store(&J->word, (unsigned long long)nren << 32 | W, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        // one prediction call site for all forms: after its own job a wave
        // takes the next one from the LDS counter or from the job word
        for (int r = wave < nren ? wave : -1; r >= 0;) {
            const int q = ren_at(r);
            predict_fast<FQ, VAL>(F, C, prof, tab, sh.w[wave], sh.ren_a[q], sh.ren_t[q], ws, &err);
            if (shared && r >= W && lane == 0) job_done(J, false);
            if (__ballot(err != 0)) break;          // uniform across the wave
            r = -1;
            if (lane == 0 && sh.err == 0 && nren > W) {
                if (shared) {
                    r = job_claim(J);
                } else {
                    r = W + atomicAdd(&sh.next_ren, 1);
                    if (r >= nren) r = -1;
                }
            }
            r = lane_get(r, 0);
        }
        if (shared) {
            if (err) atomicCAS(&sh.err, 0, err);
            if (tid == 0) {
                // every claimed job completes (its wavefront is running); an
                // error ends the wait, and the loop with it
                const long long w0 = (long long)wall_clock64();
                int done;
                while ((done = int_load(&J->done)) < nren - W && *(volatile int *)&sh.err == 0) {
                    if ((long long)wall_clock64() - w0 > FJOB_WAIT) { atomicCAS(&sh.err, 0, FERR_JOBS); break; }
                }
                acquire_agent();                        // the helpers' event records, from the L2
                if (done >= JOB_FAILED) {
                    const int he = int_load(&J->err);
                    atomicCAS(&sh.err, 0, he ? he : (int)FERR_JOBS);
                }
            }
        }
        for (int r = tid; r < nren; r += 64 * W) {
            const int b = (sh.ren_a[ren_at(r)] - 1) >> 6;
            if (b >= 0 && b < nblk) atomicOr(&sh.dmask[b >> 5], 1u << (b & 31));
        }
        if (err) atomicCAS(&sh.err, 0, err);
        __syncthreads();
        if (tid == 0) M.pops += nex;
        // the touched blocks, each once, in ascending order (every wavefront
        // makes its own list from the mask)
        int *dirty = sh.w[wave].l_id;
        int nd;
        {
            static_assert(FMAXBLK / 32 <= 32, "the touched-block mask fits lanes 0..31");
            static_assert(FWave<flist(W)>::LIST >= 2 * FSEL, "a round touches at most 2 * FSEL blocks");
            const unsigned int m = (lane < FMAXBLK / 32) ? sh.dmask[lane] : 0u;
            const int c = __popc(m);
            const int incl = scan32_incl(c);
            int o = incl - c;
            for (unsigned int mm = m; mm; mm &= mm - 1) dirty[o++] = lane * 32 + __builtin_ctz(mm);
            nd = lane_get(incl, 31);
            wave_sync();
        }
        FPROF(prof, FPH_EXEC, pt);
        // ---- tree: rescan the touched blocks, four per wavefront at a time
        for (int d0 = 4 * wave; d0 < nd; d0 += 4 * W) {
            const int d = d0 + (lane >> 4), b = d < nd ? dirty[d] : -1;
            double t1, t2, t3;
            int a1b, a2b;
            block_scan4(C, b, t1, a1b, t2, a2b, t3);
            if ((lane & 15) == 0 && b >= 0) {
                sh.b1[b] = t1; sh.ba[b] = a1b; sh.b2[b] = t2; sh.bb[b] = a2b; sh.b3[b] = t3;
            }
        }
        __syncthreads();
        if (tid < FMAXBLK / 32) sh.dmask[tid] = 0u;       // next set after the coming barriers
        FPROF(prof, FPH_TREE, pt);
    }
    if (H > 0 && tid == 0)                        // helpers leave once their current job is done
        __hip_atomic_store(&J->word, (unsigned long long)JOB_STOP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int b = tid; b < nblk; b += 64 * W) {
        G(C.b1)[b] = sh.b1[b]; G(C.b2)[b] = sh.b2[b]; G(C.b3)[b] = sh.b3[b];
        G(C.ba)[b] = sh.ba[b]; G(C.bb)[b] = sh.bb[b];
    }
    if (lane == 0) {
        atomicAdd((unsigned long long *)&F.screens, (unsigned long long)ws.screen);
        atomicAdd((unsigned long long *)&F.confirms, (unsigned long long)ws.conf);
        atomicAdd((unsigned long long *)&M.pair_evals, (unsigned long long)(ws.fp64 + ws.conf));
        atomicAdd((unsigned long long *)&M.candidates, (unsigned long long)ws.cand);
    }
    __syncthreads();
    if (tid == 0) {
        if (sh.err) M.error = sh.err;
        M.currenttime = F.tlast;
    }
    fsys_store<W>(&systems[sys], Fl);
}

// The event loop for workgroups of W wavefronts.  This file is compiled for
// each W with SDMD_FAST_WAVES = W, once with and once without SDMD_FAST_VALIDATE
// (the units build in parallel; each holds the event loop of its W), and once
// without either for the host side and the bulk prediction.
struct FastRun {
    hipStream_t stream;
    FSys *sys;
    FJobs *jobs;
    FHelp *help;
    int nsys, helpers, depth;
    long long npops, budget;
    double t_end;
};
template <int W, bool VAL> void fast_launch_run(const FastRun &r);

#ifdef SDMD_FAST_WAVES
#ifdef SDMD_FAST_VALIDATE
constexpr bool FVALIDATE = true;
#else
constexpr bool FVALIDATE = false;
#endif
// one workgroup per system and role, 8 * ceil(nsys / 8) * (1 + helpers) in
// all; validation has one staging depth (which does not change results)
template <int W, bool VAL>
void fast_launch_run(const FastRun &r) {
    const dim3 g(8 * ((r.nsys + 7) / 8) * (1 + r.helpers)), b(64 * W);
    auto *run = &k_fast_run<W, 4, VAL>;
    if constexpr (!VAL)
        if (r.depth == 2) run = &k_fast_run<W, 2, VAL>;
    hipLaunchKernelGGL(run, g, b, 0, r.stream, r.sys, r.jobs, r.help, r.nsys, r.helpers, r.npops, r.budget, r.t_end);
}
template void fast_launch_run<SDMD_FAST_WAVES, FVALIDATE>(const FastRun &);
#endif

}  // namespace sdmd

#ifndef SDMD_FAST_WAVES
// ==================================================================== host side
namespace sdmd {
// reset every system's job word before a launch (a kernel, not a memset, so
// it can sit in a captured graph)
__global__ void k_fast_jobs_reset(FJobs *jobs, int nsys) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nsys) {
        jobs[s].word = 0;
        jobs[s].done = 0;
        jobs[s].err = 0;
        jobs[s].xcc = -1;
    }
}
}  // namespace sdmd

using namespace sdmd;

struct sdmd::FastState {
    FSys *host;
    FSys *dev;
    int waves;                 // wavefronts per workgroup (events in flight per round per pass)
    int tuned;                 // waves is the autotuner's choice
    int autoshape;             // the number of helpers was left to the engine, and the shape with it
    int depth;                 // candidates per lane staged in registers (FQ)
    int validate;
    hipGraph_t graph;          // captured launch sequence (sdmd_gpu_run_graph)
    hipGraphExec_t gexec;
    int g_launches;
    long long g_budget;
    int helpers;               // helper workgroups per system (0: owners only)
    int hmax;                  // most helpers per system the GPU holds beside the owners
    FJobs *jobs;               // device: per-system job words and lists
    FHelp *help;               // device: helpers' statistics
    FHelp *hhelp;              // host copy
};

// helper workgroups per system that fit beside the owners: one workgroup
// per CU (the kernel's LDS), systems spread over the 8 XCDs, each system's
// workgroups on one XCD
static int helpers_that_fit(int nsys) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) !=
            hipSuccess || cus < 8)
        return 0;
    const int per_xcd = (nsys + 7) / 8;
    const int h = cus / 8 / per_xcd - 1;
    return h < 0 ? 0 : (h > 15 ? 15 : h);
}

template <typename T>
static int fdev_alloc(sdmd_gpu_ctx *c, T **dst, const T *src, size_t n) {
    return dev_upload(c, dst, src, n);
}

int sdmd_fast_open(sdmd_gpu_ctx *c, const sdmd_gpu_opts *o) {
    FastState *fs = (FastState *)calloc(1, sizeof(FastState));
    if (!fs) return SDMD_ENOMEM;
    c->fast = fs;
    fs->waves = c->block / 64;
    fs->depth = 4;
    if (fs->waves < 1 || fs->waves > FMAXW) return SDMD_EINVAL;
    fs->validate = o ? o->validate : 0;
    fs->host = (FSys *)calloc((size_t)c->nsys, sizeof(FSys));
    if (!fs->host) return SDMD_ENOMEM;
    int rc;
    sdmd_arena ar = {};
    for (int s = 0; s < c->nsys; s++) {
        const sdmd_system_desc *d = c->desc[s];
        FSys &F = fs->host[s];
        F.s = c->host_sys[s];
        const Sys &S = F.s;
        if (!S.steps_sorted) return SDMD_EUNSUPPORTED;
        const int N = d->natom;
        const long ncell = (long)d->cellnum[0] * d->cellnum[1] * d->cellnum[2];
        F.ncell = (int)ncell;
        F.nblk = (N + 63) / 64;
        if (F.nblk > FMAXBLK || N >= (1 << 23)) return SDMD_EUNSUPPORTED;
        if (d->cellnum[0] >= 1024 || d->cellnum[1] >= 1024 || d->cellnum[2] >= 1024) return SDMD_EUNSUPPORTED;
        for (int k = 0; k < 3; k++) F.L32[k] = (float)d->cellsize[k];
        const ScrBand sb = screen_band(fmax(d->cellsize[0], fmax(d->cellsize[1], d->cellsize[2])));
        F.eb0 = sb.eb0;
        F.band0 = sb.band0;
        F.Te = d->currenttime;
        F.tlast = d->currenttime;
        F.rebase_dt = 0.5;
        F.t_stop = INFINIT;
        const unsigned long long seed = (o && o->seed) ? o->seed : (unsigned long long)d->seed;
        F.key0 = (unsigned int)seed;
        F.key1 = (unsigned int)(seed >> 32) ^ (0x9E3779B9u * (unsigned int)(s + 1));
        F.validate = fs->validate;
        F.max_batch = o ? o->max_batch : 0;
        // cell arrays from the reference's linked lists (LIFO order kept),
        // with room for twice the fullest cell (cells fill and empty as the
        // atoms move; a cell past its capacity stops the run with an error)
        int fullest = 0;
        for (long cell = 1; cell <= ncell; cell++) {
            int n = 0;
            for (int a = d->celllist[N + cell]; a && n <= N; a = d->celllist[a], n++)
                if (a < 0 || a > N) return SDMD_EINVAL;
            if (n > N) return SDMD_EINVAL;                 // a cycle in the list
            fullest = n > fullest ? n : fullest;
        }
        int cap = FCAP_MIN;
        while (cap < 2 * fullest && cap < FCAP_MAX) cap *= 2;
        if (fullest > cap) return SDMD_EUNSUPPORTED;
        F.cap = cap;
        double *t0 = (double *)malloc(sizeof(double) * ((size_t)N + 1));
        if (!t0) return SDMD_ENOMEM;
        for (int a = 0; a <= N; a++) t0[a] = d->currenttime;
        arena_add(&ar, &F.t0, (const double *)t0, (size_t)N + 1);
        free(t0);
        arena_add(&ar, &F.ccnt, (const int *)nullptr, (size_t)ncell + 1);
        arena_add(&ar, &F.slot, (const int *)nullptr, (size_t)N + 1);
        if ((rc = fdev_alloc(c, &F.cmem, (const int *)nullptr, ((size_t)ncell + 1) * cap)) ||
            (rc = fdev_alloc(c, &F.rec, (const fvec4 *)nullptr, ((size_t)ncell + 1) * cap * 2))) {
                    return rc;
        }
        arena_add(&ar, &F.b1, (const double *)nullptr, (size_t)F.nblk);
        arena_add(&ar, &F.b2, (const double *)nullptr, (size_t)F.nblk);
        arena_add(&ar, &F.b3, (const double *)nullptr, (size_t)F.nblk);
        arena_add(&ar, &F.ba, (const int *)nullptr, (size_t)F.nblk);
        arena_add(&ar, &F.bb, (const int *)nullptr, (size_t)F.nblk);
        arena_add(&ar, &F.rctr, (const unsigned int *)nullptr, (size_t)N + 1);
        {
            // bond lists and constraint tables at fixed strides, written by
            // k_fast_derive from the lists already on the device
            const size_t nc = (size_t)(d->con_off[N + 1] > 0 ? d->con_off[N + 1] : 1), n16 = ((size_t)N + 1) * 16;
            const size_t bytes[7] = {n16 * sizeof(int), n16 * sizeof(double), n16 * sizeof(double), nc * sizeof(ConRad),
                                     nc * (2 + 2 * FCONSTEP) * sizeof(double), ((size_t)N + 1) * FCONN,
                                     ((size_t)N + 1) * sizeof(int)};
            void **dst[7] = {(void **)&F.bj16, (void **)&F.blo16, (void **)&F.bhi16, (void **)&F.crad,
                             (void **)&F.crow, (void **)&F.conn, (void **)&F.rowlo};
            size_t at[7], all = 0;
            for (int k = 0; k < 7; k++) { at[k] = all; all += (bytes[k] + 255) & ~(size_t)255; }
            char *block = nullptr;
            if (hipMalloc((void **)&block, all) != hipSuccess) return SDMD_EDEVICE;
            if ((rc = dev_keep(c, block))) return rc;
            for (int k = 0; k < 7; k++) *dst[k] = block + at[k];
            const int PR = 2 + 2 * PROW;
            // the collision table's rows are one copy for systems of equal tables
            const sdmd_system_desc *d0 = c->desc[0];
            int top = 0;
            for (int k = 0; k < NT * NT; k++)
                top = d->pair[k].step0 + d->pair[k].nstep > top ? d->pair[k].step0 + d->pair[k].nstep : top;
            const bool shared = s > 0 && top <= d0->nstep_pool && !memcmp(d->pair, d0->pair, sizeof(sdmd_pair) * NT * NT) &&
                                !memcmp(d->step_d, d0->step_d, sizeof(double) * top) &&
                                !memcmp(d->step_e, d0->step_e, sizeof(double) * top);
            double *prows = (double *)calloc(shared ? 1 : (size_t)NT * NT * PR, sizeof(double));
            if (!prows) return SDMD_ENOMEM;
            auto fill = [&](double *r, const sdmd_pair &p, int stride) {
                r[0] = p.dmin;
                r[1] = p.dmax;
                for (int k = 0; k < p.nstep && k < stride; k++) {
                    r[2 + k] = d->step_d[p.step0 + k];
                    r[2 + stride + k] = d->step_e[p.step0 + k];
                }
            };
            for (int k = 0; k < NT * NT && !shared; k++) fill(prows + (size_t)k * PR, d->pair[k], PROW);
            if (shared) F.prow = fs->host[0].prow;
            else arena_add(&ar, &F.prow, (const double *)prows, (size_t)NT * NT * PR);
            free(prows);
        }
        if ((rc = arena_commit(c, &ar))) return rc;
        // FP32 screen table: RightPair (ToolFunctions.c:278-292) resolved for
        // every type pair, the pair's limits and its step radii
        ScrTab *tb = (ScrTab *)calloc(1, sizeof(ScrTab));
        if (!tb) return SDMD_ENOMEM;
        auto back = [](int t) { return t == 3 ? 1 : t == 4 ? 2 : t == 27 ? 26 : t; };
        int pool = 0, stored = 0, nlist = 0;
        static thread_local int lists[NT * NT][3];      // first step, steps, place in the pool
        rc = SDMD_OK;
        // every defined pair's entry; equal lists of radii stored once
        ScrPair *ent = (ScrPair *)calloc(NT * NT, sizeof(ScrPair));
        if (!ent) { free(tb); return SDMD_ENOMEM; }
        for (int p = 0; p < NT * NT; p++) {
            const sdmd_pair &pp = d->pair[p];
            ent[p].rp = -1;
            if (!(pp.dmin > 0)) continue;
            if (pp.nstep > 16 || pool + pp.nstep > FRAD) { rc = SDMD_EUNSUPPORTED; break; }
            ScrPair &sp = ent[p];
            sp.dmin = (float)pp.dmin;
            sp.dmax = (float)pp.dmax;
            sp.nstep = (unsigned short)pp.nstep;
            sp.ezero = 0;
            sp.rp = (short)p;
            float list[16];
            for (int k = 0; k < pp.nstep; k++) {
                list[k] = (float)d->step_d[pp.step0 + k];
                if (d->step_e[pp.step0 + k] == 0) sp.ezero |= (unsigned short)(1u << k);
            }
            pool += pp.nstep;
            // a list already stored: that of an earlier pair with the same steps
            int q = 0;
            while (q < nlist && (lists[q][0] != pp.step0 || lists[q][1] != pp.nstep)) q++;
            if (q == nlist && stored + pp.nstep <= FRADL) {
                lists[q][0] = pp.step0; lists[q][1] = pp.nstep; lists[q][2] = stored;
                memcpy(tb->rad + stored, list, sizeof(float) * pp.nstep);
                stored += pp.nstep;
                nlist++;
            }
            sp.off = q < nlist ? (unsigned short)lists[q][2] : 0xffff;
        }
        for (int t1 = 0; t1 < NT; t1++)
            for (int t2 = 0; t2 < NT; t2++) {
                const int a = back(t1), b = back(t2);
                const int cand[4] = {t1 * NT + t2, a * NT + t2, t1 * NT + b, a * NT + b};
                int r = -1;
                for (int q = 0; q < 4 && r < 0; q++)
                    if (d->pair[cand[q]].dmin > 0) r = cand[q];
                if (r >= 0) tb->pr[t1 * NT + t2] = ent[r];
                else tb->pr[t1 * NT + t2].rp = -1;
            }
        free(ent);
        // the gather map of fstage's first level (device addresses of this
        // system's arrays)
        {
            const Sys &Sh = F.s;
            auto setg = [&](int L, const void *base, int stride, int off, int two) {
                tb->gbase[L] = (unsigned long long)(uintptr_t)base;
                tb->gstride[L] = stride;
                tb->goff[L] = off;
                tb->gtwo[L] = two;
            };
            for (int L = 0; L < 64; L++) setg(L, Sh.cx, 1, 0, 0);
            setg(7, F.rctr, 1, 0, 0);
            for (int q = 0; q < 16; q++) setg(48 + q, F.bj16, 16, q, 0);
            const void *d8[7] = {Sh.x, Sh.y, Sh.z, Sh.vx, Sh.vy, Sh.vz, Sh.evc};
            for (int L = 0; L < 7; L++) setg(L, d8[L], 2, 0, 1);
            const void *d4[10] = {Sh.cx, Sh.cy, Sh.cz, Sh.type, Sh.hbbond, Sh.hbnb, Sh.protein, Sh.aanum, Sh.nbstat,
                                  Sh.nbnum};
            for (int L = 0; L < 10; L++) setg(8 + L, d4[L], 1, 0, 0);
            for (int k = 0; k < SDMD_NBSLOTS; k++) setg(18 + k, Sh.nbp, SDMD_NBSLOTS, k, 0);
            setg(26, Sh.bond_off, 1, 0, 0); setg(27, Sh.bond_off, 1, 1, 0);
            setg(28, Sh.con_off, 1, 0, 0); setg(29, Sh.con_off, 1, 1, 0);
            setg(30, Sh.hbitype, 1, 0, 0); setg(31, F.rowlo, 1, 0, 0);
        }
        if (rc == SDMD_OK) {
            ScrTab *dt = nullptr;
            rc = fdev_alloc(c, &dt, (const ScrTab *)tb, 1);
            F.scrtab = dt;
        }
        free(tb);
        if (rc) return rc;
    }
    if ((rc = fdev_alloc(c, &fs->dev, fs->host, (size_t)c->nsys))) return rc;
    hipLaunchKernelGGL(k_fast_cells, dim3(c->nsys, 64), dim3(256), 0, c->stream, fs->dev);
    hipLaunchKernelGGL(k_fast_derive, dim3(c->nsys, 64), dim3(256), 0, c->stream, fs->dev);
    if (hipGetLastError() != hipSuccess) return SDMD_EDEVICE;
    if ((rc = fdev_alloc(c, &fs->jobs, (const FJobs *)nullptr, (size_t)c->nsys))) return rc;
    if ((rc = fdev_alloc(c, &fs->help, (const FHelp *)nullptr, (size_t)c->nsys))) return rc;
    fs->hhelp = (FHelp *)calloc((size_t)c->nsys, sizeof(FHelp));
    if (!fs->hhelp) return SDMD_ENOMEM;
    fs->hmax = helpers_that_fit(c->nsys);
    const int want = o ? o->helpers : 0;
    if (want < -1) return SDMD_EINVAL;
    fs->helpers = want < 0 ? 0 : (want == 0 ? fs->hmax : (want < fs->hmax ? want : fs->hmax));
    fs->autoshape = want == 0;
    return SDMD_OK;
}

static int fast_sync_from(sdmd_gpu_ctx *c) {
    FastState *fs = c->fast;
    if (hipMemcpyAsync(fs->host, fs->dev, sizeof(FSys) * c->nsys, hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
        hipMemcpyAsync(fs->hhelp, fs->help, sizeof(FHelp) * c->nsys, hipMemcpyDeviceToHost, c->stream) !=
            hipSuccess ||
        hipStreamSynchronize(c->stream) != hipSuccess)
        return SDMD_EDEVICE;
    for (int s = 0; s < c->nsys; s++) {
        c->host_sys[s] = fs->host[s].s;
        c->host_sys[s].pair_evals += fs->hhelp[s].pair_evals;       // predictions run by helper workgroups
        c->host_sys[s].candidates += fs->hhelp[s].candidates;
    }
    return SDMD_OK;
}

int sdmd_fast_sync(sdmd_gpu_ctx *c) { return fast_sync_from(c); }

// Wavefronts per workgroup of a launch.  With helper workgroups a round's
// re-predictions (10 to 40) find more wavefronts than they need, and one
// wavefront per SIMD, with all registers of the SIMD, is the fastest a
// prediction gets: us per round with 4 / 8 wavefronts per workgroup 20 / 28
// (59 atoms), 35 / 40 (64 systems of 1 536), 47 / 52 (26 080); ms for 2 000
// events of each of 32, 64, 96 and 128 systems of 1 536 atoms (7, 3, 1 and 1
// helpers) 10.4 / 14.8, 11.2 / 15.0, 14.3 / 16.2 and 14.4 / 16.4.  Without
// helpers the owner's wavefronts are all there are: 45 / 35 ms for 6 000
// events of 26 080 atoms.  A caller that asks for a number of helpers gets the
// workgroups asked for with it; the autotuner's choice is taken as it is.
static int run_waves(const FastState *fs) {
    return (!fs->tuned && fs->autoshape && fs->helpers > 0 && fs->waves > 4) ? 4 : fs->waves;
}

template <bool VAL>
static void launch_shape(int waves, const FastRun &r) {
    switch (waves) {
    case 4: fast_launch_run<4, VAL>(r); break;
    case 8: fast_launch_run<8, VAL>(r); break;
    case 12: fast_launch_run<12, VAL>(r); break;
    case 16: fast_launch_run<16, VAL>(r); break;
    default: fast_launch_run<1, VAL>(r); break;
    }
}

// the event loop for the context's shape (wavefronts x staging depth x
// helper workgroups), after a reset of the job words
static void launch_run(sdmd_gpu_ctx *c, long long pops, long long budget, double t_end) {
    FastState *fs = c->fast;
    hipLaunchKernelGGL(k_fast_jobs_reset, dim3((c->nsys + 255) / 256), dim3(256), 0, c->stream, fs->jobs, c->nsys);
    const FastRun r = {c->stream, fs->dev, fs->jobs, fs->help, c->nsys, fs->helpers, fs->depth, pops, budget, t_end};
    if (fs->validate) launch_shape<true>(run_waves(fs), r);
    else launch_shape<false>(run_waves(fs), r);
}

static int budget_ticks(double max_ms, long long *out) {
    *out = 1LL << 62;
    if (max_ms > 0) {
        int dev = 0, khz = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0)
            return SDMD_EDEVICE;
        *out = (long long)(max_ms * khz);
    }
    return SDMD_OK;
}

// every system's device error word (0 = none) after a sync
static int fast_errors(sdmd_gpu_ctx *c) {
    for (int s = 0; s < c->nsys; s++)
        if (c->fast->host[s].s.error) return SDMD_ESTATE;
    return SDMD_OK;
}

// one window of `events` more executed events per system, enqueued on the
// context's stream without waiting (the device REMD loop)
int sdmd_fast_launch_events(sdmd_gpu_ctx *c, long long events) {
    launch_run(c, -events, 1LL << 62, INFINIT);
    return hipGetLastError() == hipSuccess ? SDMD_OK : SDMD_EDEVICE;
}

// device address of system s's thermostat temperature
double *sdmd_fast_temperature_addr(sdmd_gpu_ctx *c, int s) { return &c->fast->dev[s].s.T; }

int sdmd_fast_prepare(sdmd_gpu_ctx *c) {
    FastState *fs = c->fast;
    HIPV(hipEventRecord(c->ev0, c->stream));
    // predictions: enough workgroups of 8 wavefronts to fill the GPU, at
    // least one atom per wavefront; a workgroup's set-up (50 KB of tables
    // into LDS) costs about one prediction
    int maxn = 1;
    for (int s = 0; s < c->nsys; s++) maxn = fs->host[s].s.N > maxn ? fs->host[s].s.N : maxn;
    const int want = (maxn + 7) / 8, fit = (1024 + c->nsys - 1) / c->nsys;
    const dim3 gp(c->nsys, want < fit ? want : fit), ga(c->nsys, gp.y < 64 ? gp.y : 64);
    hipLaunchKernelGGL(k_fast_records, ga, dim3(256), 0, c->stream, fs->dev);
    if (fs->validate) hipLaunchKernelGGL((k_fast_predict<8, true>), gp, dim3(512), 0, c->stream, fs->dev);
    else hipLaunchKernelGGL((k_fast_predict<8, false>), gp, dim3(512), 0, c->stream, fs->dev);
    hipLaunchKernelGGL(k_fast_blocks, ga, dim3(256), 0, c->stream, fs->dev);
    if (hipGetLastError() != hipSuccess) return SDMD_EDEVICE;   // launch rejected (shape, resources)
    HIPV(hipEventRecord(c->ev1, c->stream));
    if (hipStreamSynchronize(c->stream) != hipSuccess) return SDMD_EDEVICE;
    float ms = 0;
    HIPV(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    if (fast_sync_from(c)) return SDMD_EDEVICE;
    return fast_errors(c);
}

int sdmd_fast_run(sdmd_gpu_ctx *c, long long pops, double max_ms, double t_end) {
    FastState *fs = c->fast;
    long long budget;
    if (budget_ticks(max_ms, &budget)) return SDMD_EDEVICE;
    HIPV(hipEventRecord(c->ev0, c->stream));
    launch_run(c, pops, budget, t_end);
    if (hipGetLastError() != hipSuccess) return SDMD_EDEVICE;
    HIPV(hipEventRecord(c->ev1, c->stream));
    if (hipStreamSynchronize(c->stream) != hipSuccess) return SDMD_EDEVICE;
    float ms = 0;
    HIPV(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    if (fast_sync_from(c)) return SDMD_EDEVICE;
    return fast_errors(c);
}

// positions at the clock (earliest pending event), event times relative to it
int sdmd_fast_download(sdmd_gpu_ctx *c, int s, sdmd_system_desc *out) {
    FastState *fs = c->fast;
    if (fast_sync_from(c)) return SDMD_EDEVICE;
    const FSys &F = fs->host[s];
    const Sys &S = F.s;
    if (S.error) return SDMD_ESTATE;         // e.g. an incomplete drain: not a snapshot at one time
    // every array is wanted here (the plain engine leaves out missing ones)
    for (const void *p : {(void *)out->x, (void *)out->y, (void *)out->z, (void *)out->vx, (void *)out->vy, (void *)out->vz,
                          (void *)out->type, (void *)out->cellx, (void *)out->celly, (void *)out->cellz,
                          (void *)out->hb_bond, (void *)out->hb_itype, (void *)out->nb_partner,
                          (void *)out->nb_partnernum, (void *)out->nb_status, (void *)out->dyn_j, (void *)out->dyn_bits,
                          (void *)out->ev_partner, (void *)out->ev_type, (void *)out->ev_sub, (void *)out->ev_counter,
                          (void *)out->ev_pcounter, (void *)out->ev_time, (void *)out->ev_pot, (void *)out->celllist})
        if (!p) return SDMD_EDEVICE;
    const int N = S.N;
    const size_t N1 = (size_t)N + 1;
    double *t0 = (double *)malloc(sizeof(double) * N1);
    double *b1 = (double *)malloc(sizeof(double) * (size_t)F.nblk);
    if (!t0 || !b1) { free(t0); free(b1); return SDMD_ENOMEM; }
    // the lists from the cell arrays on the device, then every array that a
    // run changes in one copy
    const int blocks = (F.ncell + 255) / 256;
    hipLaunchKernelGGL(k_fast_lists, dim3(blocks < 1024 ? blocks : 1024), dim3(256), 0, c->stream, fs->dev, s);
    int rc = hip_ok(hipGetLastError());
    if (rc == SDMD_OK) rc = hip_ok(hipMemcpyAsync(t0, F.t0, sizeof(double) * N1, hipMemcpyDeviceToHost, c->stream));
    if (rc == SDMD_OK)
        rc = hip_ok(hipMemcpyAsync(b1, F.b1, sizeof(double) * (size_t)F.nblk, hipMemcpyDeviceToHost, c->stream));
    if (rc == SDMD_OK) rc = sdmd_dyn_download(c, s);
    if (rc != SDMD_OK) HIPV(hipStreamSynchronize(c->stream));   // no copy in flight when the buffers go
    if (rc == SDMD_OK) sdmd_dyn_scatter(c, s, out);
    if (rc == SDMD_OK) {
        double T = INFINIT;
        for (int b = 0; b < F.nblk; b++) if (b1[b] < T) T = b1[b];
        if (!(T < INFINIT)) T = F.tlast;
        for (int a = 1; a <= N; a++) {
            const double dt = T - t0[a];
            out->x[a] = out->x[a] + out->vx[a] * dt;
            out->y[a] = out->y[a] + out->vy[a] * dt;
            out->z[a] = out->z[a] + out->vz[a] * dt;
            out->ev_time[a] -= T;
        }
        out->currenttime = T;
    }
    free(t0); free(b1);
    return rc;
}

// energies of every system into out's three planes (kinetic, potential,
// error flag; energy_planes_to_host reads them back)
int sdmd_fast_energy_launch(sdmd_gpu_ctx *c, double *out) {
    hipLaunchKernelGGL(k_fast_energy, dim3(c->nsys, c->echunks), dim3(64 * EWAVES), 0, c->stream, c->fast->dev,
                       c->epart);
    hipLaunchKernelGGL(k_energy_reduce, dim3(c->nsys), dim3(64), 0, c->stream, c->epart, c->echunks, out);
    return hipGetLastError() == hipSuccess ? SDMD_OK : SDMD_EDEVICE;
}

// the thermostat's target temperature of one system (REMD exchanges set it)
int sdmd_fast_set_temperature(sdmd_gpu_ctx *c, int s, double T) {
    FastState *fs = c->fast;
    fs->host[s].s.T = T;
    c->host_sys[s].T = T;
    if (hipMemcpyAsync(&fs->dev[s].s.T, &fs->host[s].s.T, sizeof(double), hipMemcpyHostToDevice, c->stream) !=
            hipSuccess || hipStreamSynchronize(c->stream) != hipSuccess)
        return SDMD_EDEVICE;
    return SDMD_OK;
}

int sdmd_fast_stats(sdmd_gpu_ctx *c, int s, sdmd_gpu_fast_stats *out) {
    if (fast_sync_from(c)) return SDMD_EDEVICE;
    const FSys &F = c->fast->host[s];
    out->batches = F.batches;
    out->deferred = F.deferred;
    out->single = F.single;
    out->screens = F.screens;
    out->confirms = F.confirms;
    out->validated = F.validated;
    out->agree = F.agree;
    out->rebases = F.rebases;
    const FHelp &h = c->fast->hhelp[s];          // predictions run by helper workgroups
    out->screens += h.screens;
    out->confirms += h.confirms;
    out->validated += h.validated;
    out->agree += h.agree;
    out->causal = F.causal + h.causal;
    out->max_screen_rel_err = F.max_screen_err > h.max_screen_err ? F.max_screen_err : h.max_screen_err;
    out->max_time_rel_err = F.max_time_err > h.max_time_err ? F.max_time_err : h.max_time_err;
    out->clock = F.tlast;
    out->helpers = c->fast->helpers;
    return SDMD_OK;
}

// A sequence of `launches` event-loop launches (each bounded by max_ms of
// device time) captured once into a HIP graph and replayed; the graph is
// rebuilt when the shape, count or bound changes.
int sdmd_fast_run_graph(sdmd_gpu_ctx *c, int launches, double max_ms) {
    FastState *fs = c->fast;
    long long budget;
    if (launches < 1 || budget_ticks(max_ms, &budget)) return SDMD_EINVAL;
    const int key = ((launches * 16 + fs->helpers) * 64 + run_waves(fs)) * 8 + fs->depth;
    if (!fs->gexec || fs->g_launches != key || fs->g_budget != budget) {
        if (fs->gexec) { HIPV(hipGraphExecDestroy(fs->gexec)); fs->gexec = nullptr; }
        if (fs->graph) { HIPV(hipGraphDestroy(fs->graph)); fs->graph = nullptr; }
        if (hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) return SDMD_EDEVICE;
        bool launched = true;
        for (int k = 0; k < launches; k++) {
            launch_run(c, 1LL << 60, budget, INFINIT);
            launched = launched && hipGetLastError() == hipSuccess;
        }
        const bool captured = hipStreamEndCapture(c->stream, &fs->graph) == hipSuccess;
        if (!launched || !captured) {
            if (fs->graph) { HIPV(hipGraphDestroy(fs->graph)); fs->graph = nullptr; }
            return SDMD_EDEVICE;
        }
        if (hipGraphInstantiate(&fs->gexec, fs->graph, nullptr, nullptr, 0) != hipSuccess) {
            fs->gexec = nullptr;
            return SDMD_EDEVICE;
        }
        fs->g_launches = key;
        fs->g_budget = budget;
    }
    HIPV(hipEventRecord(c->ev0, c->stream));
    if (hipGraphLaunch(fs->gexec, c->stream) != hipSuccess) return SDMD_EDEVICE;
    HIPV(hipEventRecord(c->ev1, c->stream));
    if (hipStreamSynchronize(c->stream) != hipSuccess) return SDMD_EDEVICE;
    float ms = 0;
    HIPV(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    if (fast_sync_from(c)) return SDMD_EDEVICE;
    return fast_errors(c);
}

// Time each workgroup shape (wavefronts per system x candidates staged per
// lane) on the live systems for trial_ms of device time and keep the one that
// executes the most events per millisecond; the systems advance meanwhile.
int sdmd_fast_autotune(sdmd_gpu_ctx *c, double trial_ms, int32_t *block_out, int32_t *depth_out) {
    FastState *fs = c->fast;
    static const int shapes[][2] = {{4, 4}, {8, 4}, {12, 4}, {16, 4}, {4, 2}, {8, 2}, {12, 2}, {16, 2}};
    double best = -1;
    int bw = fs->waves, bq = fs->depth;
    fs->tuned = 1;                               // the trials run the shapes as named
    for (const auto &sh : shapes) {
        fs->waves = sh[0];
        fs->depth = sh[1];
        long long ev0 = 0, ev1 = 0;
        for (int s = 0; s < c->nsys; s++) ev0 += fs->host[s].s.frame;
        int rc = sdmd_fast_run(c, 1LL << 60, trial_ms, INFINIT);
        if (rc) return rc;
        for (int s = 0; s < c->nsys; s++) ev1 += fs->host[s].s.frame;
        const double rate = (double)(ev1 - ev0) / (c->last_ms > 0 ? c->last_ms : 1.0);
        if (rate > best) { best = rate; bw = sh[0]; bq = sh[1]; }
    }
    fs->waves = bw;
    fs->depth = bq;
    // helper workgroups for the kept shape: all that fit (the trials above),
    // half of them, none
    int bh = fs->helpers;
    const int hs[2] = {fs->hmax / 2, 0};
    for (int k = 0; k < 2; k++) {
        if (hs[k] == bh || (k == 0 && hs[0] == 0)) continue;
        const int keep = fs->helpers;
        fs->helpers = hs[k];
        long long ev0 = 0, ev1 = 0;
        for (int s = 0; s < c->nsys; s++) ev0 += fs->host[s].s.frame;
        int rc = sdmd_fast_run(c, 1LL << 60, trial_ms, INFINIT);
        if (rc) return rc;
        for (int s = 0; s < c->nsys; s++) ev1 += fs->host[s].s.frame;
        const double rate = (double)(ev1 - ev0) / (c->last_ms > 0 ? c->last_ms : 1.0);
        if (rate > best) { best = rate; bh = hs[k]; }
        fs->helpers = keep;
    }
    fs->helpers = bh;
    c->block = 64 * bw;
    if (block_out) *block_out = 64 * bw;
    if (depth_out) *depth_out = bq;
    return SDMD_OK;
}

void sdmd_fast_close(sdmd_gpu_ctx *c) {
    if (!c->fast) return;
    if (c->fast->gexec) HIPV(hipGraphExecDestroy(c->fast->gexec));
    if (c->fast->graph) HIPV(hipGraphDestroy(c->fast->graph));
    free(c->fast->host);
    free(c->fast->hhelp);
    free(c->fast);
    c->fast = nullptr;
}
#endif  // SDMD_FAST_WAVES
