// pdmd_engine.hip -- gfx950 kernels of the PRIME20 discontinuous-MD event
// loop.  One workgroup owns one system for a whole launch and commits its
// events in the reference's serial order, on up to seven event wavefronts (64
// lanes each) and one calendar wavefront.
//   * Each round takes up to W calendar entries; the pair events among them
//     run side by side, one per wavefront, and the round commits the prefix
//     the serial order would have run the same way (footprint marks per bead
//     in LDS, no new calendar key ahead of a later one of the round).
//   * Inside an event the wavefront issues every collision-time prediction
//     the event triggers (full recomputes of the colliding pair and of the
//     down beads that pointed at it, single-pair updates of the down set) as
//     one batch of 64-byte gathers, one lane per pair, FP64 in the
//     reference's evaluation order (no contraction).
//   * The calendar is a leaf per bead, in LDS when the system fits, else in
//     HBM, and a time per 16 leaves in LDS.  While events run, the calendar
//     wavefront brings those times up to date and collects the least entries,
//     from which and from the events' new entries the next round is taken.
//   * Neighbour-list rebuilds (coarse-cell counting sort, a wavefront per
//     cell), free flight and displacement checks at the sync event run on all
//     wavefronts of the system; at start-up and where an update is forced
//     their steps are launches over the whole GPU.
// Many systems in one launch run concurrently, one workgroup each.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>
#include <mutex>
#include <type_traits>

#include "pdmd_device.h"
#include "pdmd_engine.h"

namespace pdmd {
namespace {

constexpr int kW = 64;
constexpr int kBlk = 16;
constexpr int kSup = 64;
constexpr int kNumbin = 2000;
constexpr int kMaxBlist = 160;
constexpr double kLt = 1e-10;
constexpr double kSm = 5e-12;
constexpr int kMaxWaves = 8;  // most wavefronts in one system's workgroup

__device__ inline int lane_id() { return (int)(threadIdx.x & (kW - 1)); }
__device__ inline int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// Phase timers (device clock cycles summed into SysState::phase[k]) when
// built with -DPDMD_PHASE_TIMERS; no code otherwise.  Phases: 0 selection,
// 1 pair event before rescheduling, 2 reschedule loads and work list,
// 3 reschedule predictions, 4 down-set updates, 5 leaf writes,
// 7 sync event without rebuild, 8 list rebuild, 9 full events(),
// 10 ghost event before rescheduling, 11 reschedule rows and work list,
// 12 reschedule down-set scan, 13 rebuild count, 14 sync count; list
// rebuild steps: 16 cells and histogram, 17 scan, 19 sorted
// copies, 20 neighbour search; multi-wavefront rounds: 21 rounds of two or
// more pair events, 22 entries popped in them, 23 entries committed, 24
// footprint marks up to the first round barrier, 25 footprint checks up to
// the second, 26 new keys up to the third, 27 the wait for the other wavefronts,
// 28 rounds cut by a footprint conflict or an event that cannot speculate,
// 29 rounds cut by the key order; round selection: 30 the pops, 31 the
// pool collected again for them; rescheduling batches: 32 pair predictions made
// in them, 33 their 64-lane passes (32 / (64 * 33) is their lane occupancy);
// down-set work outside the batches: 34 single-pair updates predicted one
// per lane, 35 full recomputes run one bead at a time, 36 events rescheduled
// by the generic form.
enum { kPhSelect = 0, kPhPair = 1, kPhLoads = 2, kPhPred = 3, kPhDown = 4, kPhLeaf = 5,
       kPhSync = 7, kPhLists = 8, kPhEvents = 9, kPhGhost = 10, kPhRows = 11, kPhScan = 12, kPhNRebuild = 13,
       kPhNSync = 14, kPhLCells = 16, kPhLScan = 17, kPhLCopy = 19, kPhLSearch = 20,
       kPhNRound = 21, kPhNPopped = 22, kPhNCommit = 23, kPhBMark = 24, kPhBCheck = 25, kPhBKeys = 26,
       kPhBTail = 27, kPhNCutMark = 28, kPhNCutKey = 29, kPhSelPop = 30, kPhSelCopy = 31, kPhNPred = 32,
       kPhNPredPass = 33, kPhNSingle = 34, kPhNFull = 35, kPhNGeneric = 36 };
#ifdef PDMD_PHASE_TIMERS
#define PH_BEGIN(v) long long v = clock64()
#define PH_END(S, k, v)                                                                                  \
    do {                                                                                                 \
        if (threadIdx.x == 0)                                                                            \
            atomicAdd((unsigned long long*)&(S).st->phase[k], (unsigned long long)(clock64() - (v)));   \
        v = clock64();                                                                                   \
    } while (0)
#define PH_COUNT(S, k)                                                                      \
    do {                                                                                    \
        if (threadIdx.x == 0) atomicAdd((unsigned long long*)&(S).st->phase[k], 1ull);     \
    } while (0)
#define PH_RESET(v) v = clock64()
#define PH_ADDN(S, k, n)                                                                                  \
    do {                                                                                                  \
        if (threadIdx.x == 0) atomicAdd((unsigned long long*)&(S).st->phase[k], (unsigned long long)(n)); \
    } while (0)
// a per-lane count, summed over the wavefront where it is added
#define PH_LANE_DECL(v) int v = 0
#define PH_LANE_INC(v) ++v
#define PH_LANE_ADD(S, k, v)                                            \
    do {                                                                \
        int ph_s_ = v;                                                  \
        for (int ph_o_ = 32; ph_o_ > 0; ph_o_ >>= 1) ph_s_ += __shfl_xor(ph_s_, ph_o_, 64); \
        PH_ADDN(S, k, ph_s_);                                           \
    } while (0)
#else
#define PH_BEGIN(v) \
    do {            \
    } while (0)
#define PH_END(S, k, v) \
    do {                \
    } while (0)
#define PH_COUNT(S, k) \
    do {               \
    } while (0)
#define PH_RESET(v) \
    do {            \
    } while (0)
#define PH_ADDN(S, k, n) \
    do {                 \
    } while (0)
#define PH_LANE_DECL(v) \
    do {                \
    } while (0)
#define PH_LANE_INC(v) \
    do {               \
    } while (0)
#define PH_LANE_ADD(S, k, v) \
    do {                     \
    } while (0)
#endif

// Global-memory access through the generic pointers of SysDev, as global_*
// operations (a flat operation would also hold back every LDS wait).
#define GLB __attribute__((address_space(1)))
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
template <class T>
__device__ inline T gld(const T* p) {
    static_assert(sizeof(T) % 16 == 0, "16-byte multiple");
    u32x4 t[sizeof(T) / 16];
    const GLB u32x4* q = (const GLB u32x4*)p;
#pragma unroll
    for (int k = 0; k < (int)(sizeof(T) / 16); ++k) t[k] = q[k];
    T r;
    __builtin_memcpy(&r, t, sizeof(T));
    return r;
}
template <class T>
__device__ inline void gst(T* p, const T& v) {
    static_assert(sizeof(T) % 16 == 0, "16-byte multiple");
    u32x4 t[sizeof(T) / 16];
    __builtin_memcpy(t, &v, sizeof(T));
    GLB u32x4* q = (GLB u32x4*)p;
#pragma unroll
    for (int k = 0; k < (int)(sizeof(T) / 16); ++k) q[k] = t[k];
}
template <class T>
__device__ inline T gl1(const T* p) {
    return *(const GLB T*)p;
}
template <class T>
__device__ inline void gs1(T* p, T v) {
    *(GLB T*)p = v;
}
__device__ inline int2 gl2(const int2* p) {
    const unsigned long long v = gl1(reinterpret_cast<const unsigned long long*>(p));
    return make_int2((int)(unsigned)v, (int)(unsigned)(v >> 32));
}
__device__ inline void gs2(int2* p, int2 v) {
    gs1(reinterpret_cast<unsigned long long*>(p), (unsigned long long)(unsigned)v.x | ((unsigned long long)(unsigned)v.y << 32));
}

// The workgroup's dynamic LDS.  Views into it are kept as offsets and
// turned into pointers from this array where they are used, so the compiler
// keeps LDS accesses as ds_* operations (a pointer stored in a struct and
// passed on would become a flat pointer).
extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

// the scaled tables sit at the start of the LDS, the system's SysDev right
// after them (field reads become LDS reads in every function)
constexpr int kSdOff = (int)((sizeof(DevTables) + 15) / 16 * 16);
__device__ inline const DevTables& tabs() { return *reinterpret_cast<const DevTables*>(smem); }
__device__ inline const SysDev& sdev() { return *reinterpret_cast<const SysDev*>(smem + kSdOff); }

// ------------------------------------------------------------------------
// project RNG (counter-based splitmix64) and a logarithm from basic ops
// ------------------------------------------------------------------------
__device__ inline uint64_t sm64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}
__device__ inline double rng_u01(uint64_t seed, int stream, uint64_t ctr) {
    const uint64_t key = sm64(seed ^ (0x5851F42D4C957F2Dull * (uint64_t)(stream + 1)));
    return (double)(sm64(key + ctr) >> 11) * (1.0 / 9007199254740992.0);
}
// log x = e ln2 + 2 atanh((m-1)/(m+1)), m in [1/sqrt2, sqrt2]; identical
// bits to the CPU oracle's restatement
__device__ double dlog(double x) {
    uint64_t b = (uint64_t)__double_as_longlong(x);
    int e = (int)((b >> 52) & 0x7ff);
    int adj = 0;
    if (e == 0) {
        x = x * 18014398509481984.0;
        b = (uint64_t)__double_as_longlong(x);
        e = (int)((b >> 52) & 0x7ff);
        adj = -54;
    }
    e = e - 1023 + adj;
    b = (b & 0x000FFFFFFFFFFFFFull) | 0x3FF0000000000000ull;
    double m = __longlong_as_double((long long)b);
    if (m > 1.4142135623730951) {
        m = m * 0.5;
        e = e + 1;
    }
    const double s = (m - 1.0) / (m + 1.0);
    const double z = s * s;
    double p = 2.0 / 25.0;
    p = p * z + 2.0 / 23.0;
    p = p * z + 2.0 / 21.0;
    p = p * z + 2.0 / 19.0;
    p = p * z + 2.0 / 17.0;
    p = p * z + 2.0 / 15.0;
    p = p * z + 2.0 / 13.0;
    p = p * z + 2.0 / 11.0;
    p = p * z + 2.0 / 9.0;
    p = p * z + 2.0 / 7.0;
    p = p * z + 2.0 / 5.0;
    p = p * z + 2.0 / 3.0;
    const double lm = 2.0 * s + (s * z) * p;
    const double de = (double)e;
    return de * 6.93147180369123816490e-01 + (de * 1.90821492927058770002e-10 + lm);
}

// ------------------------------------------------------------------------
// pair codes: closed form of make_code.f from two topo words, overrides
// ------------------------------------------------------------------------
// without a branch: the same-chain rules come from a table over the two bead
// kinds and their residue distance, clamped to 4 either way (DevTables::statc,
// chain_code).  As a switch, every rule that some lane needed ran on its own.
__device__ inline int static_t(const DevTables& T, int ta, int tb) {
    const int ka = topo_kind(ta), ra = topo_res(ta), kb = topo_kind(tb), rb = topo_res(tb);
    const bool swap = ka > kb || (ka == kb && ra > rb);
    const int k4 = swap ? kb * 4 + ka : ka * 4 + kb, d = swap ? ra - rb : rb - ra;
    int same = T.statc[k4 * 9 + min(max(d, -4), 4) + 4];
    const bool hp = topo_hp(ta) && topo_hp(tb);
    same = same == 16 && !hp ? 1 : same;
    // -Dchaptype=2 builds no code inside a second-species chain
    // (make_code.f:349,366; its side-chain loop finds no firstside2 entry)
    same = topo_free(ta) ? 1 : same;
    // -Dno_h zeroes hp only where make_code.f:80-104 reads it (different
    // chains); the same-chain loops read hp1/hp2 (make_code.f:174-186)
    // and none between two second-species chains (make_code.f:519-547)
    const bool rr = ka == 3 && kb == 3, well = rr && hp && !topo_noh(ta) && !(topo_free(ta) && topo_free(tb));
    const bool nc = (ka == 1 && kb == 2) || (ka == 2 && kb == 1);
    const int tn = ka == 1 ? ta : tb, tc = ka == 1 ? tb : ta;
    const bool pro = topo_pro(tn) && topo_chain(tn) < topo_chain(tc);
    const int other = well ? 16 : (nc && !pro ? 15 : 1);
    const int r = topo_chain(ta) == topo_chain(tb) ? same : other;
    // under -Dno_hbs make_code.f skips every code-15 assignment (:114-170,
    // :192-208, :348-365): those pairs keep the hard-core code 1
    return r == 15 && topo_nohbs(ta) ? 1 : r;
}
// Where nbor.f finds the pair {a, b}, as one 64-bit key: the cell it scans
// (cell_add.f's linear index, cells in ascending order), the place of that
// cell's own bead in its list, the other cell's place in the scan
// (cell_link.f's half stencil; 0 for the own cell), the other bead's place.
// A bead's neighbour rows in nbor.f's order are its rows sorted by this key.
// a and b: the beads' fine cells (10 bits per axis) and list places.
__device__ inline unsigned fine_lin(int f, int nc) {
    return 1u + (unsigned)((f & 1023) + 2) + (unsigned)((((f >> 10) & 1023) + 2) + ((f >> 20) + 2) * nc) * (unsigned)nc;
}
// la: fine_lin of a's cell
__device__ inline unsigned long long nbor_key(int M, const DevTables& T, int2 a, unsigned la, int2 b) {
    const int fa = a.x, fb = b.x, pa = a.y & 0xFFFF, pb = b.y & 0xFFFF;
    int at = 62;  // (dx + 2) + 5 (dy + 2) + 25 (dz + 2) of the periodic offset, each in [-2, 2]
    const int mul[3] = {1, 5, 25};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        // periodic offset in [-(M / 2), M - M / 2), in [-2, 2] for neighbours
        int t = ((fb >> (10 * q)) & 1023) - ((fa >> (10 * q)) & 1023);
        t += t < 0 ? M : 0;
        at += mul[q] * (t < M - M / 2 ? t : t - M);
    }
    const int h = T.halfst[at], g = T.halfst[124 - at];
    const bool own = at == 62, by_a = own || h > 0;
    const unsigned lin = by_a ? la : fine_lin(fb, M + 4);
    const unsigned first = own ? min(pa, pb) : (by_a ? pa : pb);
    const unsigned rest = own ? max(pa, pb) : (by_a ? (unsigned)(h << 10 | pb) : (unsigned)(g << 10 | pa));
    return ((unsigned long long)lin << 26) | (first << 16) | rest;
}

// ev_code(row, col) with row's override slots o
__device__ inline int dyn_code(int4 o, int col, int stat) {
    if (o.x >= 0 && (o.x >> 8) == col) return o.x & 0xff;
    if (o.y >= 0 && (o.y >> 8) == col) return o.y & 0xff;
    if (o.z >= 0 && (o.z >> 8) == col) return o.z & 0xff;
    if (o.w >= 0 && (o.w >> 8) == col) return o.w & 0xff;
    return stat;
}
// single-lane writer of ev_code(row, col) = code (keeps an override only
// where it differs from the static code)
__device__ void set_code(const SysDev&, int row, int col, int code, int& status) {
    const SysDev& S = sdev();

    int4 o = gld(S.ovr + (row));
    const int stat = static_t(tabs(), gl1(&S.rec[row].topo), gl1(&S.rec[col].topo));
    if (o.x >= 0 && (o.x >> 8) == col) o.x = -1;
    if (o.y >= 0 && (o.y >> 8) == col) o.y = -1;
    if (o.z >= 0 && (o.z >> 8) == col) o.z = -1;
    if (o.w >= 0 && (o.w >> 8) == col) o.w = -1;
    if (code != stat) {
        const int v = (col << 8) | code;
        if (o.x < 0) o.x = v;
        else if (o.y < 0) o.y = v;
        else if (o.z < 0) o.z = v;
        else if (o.w < 0) o.w = v;
        else status = kErrOverrideSlots;
    }
    gst(S.ovr + (row), o);
}

// ------------------------------------------------------------------------
// predictors: core.f, bond.f, sqwel.f, sqshlder.f, nc_sqwel.f
// ------------------------------------------------------------------------
struct Geo {
    double rx, ry, rz, b, r2, v2;
};
// x - round(x) (round: halves away from zero), from the half-to-even
// rounding instruction: the two differ only where the remainder is exactly
// one half, whose sign is then the opposite of x's
__device__ inline double min_image(double x) {
    const double d = x - __builtin_rint(x);
    return fabs(d) == 0.5 ? copysign(0.5, -x) : d;
}
__device__ inline void geo(const Rec& a, const Rec& c, double tf, Geo& g) {
    const double vx = a.vx - c.vx, vy = a.vy - c.vy, vz = a.vz - c.vz;
    const double rx = min_image(a.x - c.x + vx * tf);
    const double ry = min_image(a.y - c.y + vy * tf);
    const double rz = min_image(a.z - c.z + vz * tf);
    g.rx = rx;
    g.ry = ry;
    g.rz = rz;
    g.b = rx * vx + ry * vy + rz * vz;
    g.r2 = rx * rx + ry * ry + rz * rz;
    g.v2 = vx * vx + vy * vy + vz * vz;
}
__device__ inline void bond_window(const DevTables& T, int code, double2 bw, double& blmin, double& blmax) {
    if (code >= 10) {
        blmin = bw.x;
        blmax = bw.y;
    } else {
        blmin = T.ev_param[2][code];
        blmax = T.ev_param[3][code];
    }
}
// collision time of a pair with ev_code `code` from its geometry g at the
// current false time (ia, ic: identities, the lower bead's first; bonded:
// the two are H-bonded; bwa: the lower bead's own bond window); tij keeps
// its preset (1e9) and type its value when no event is predicted.
// Every predictor of core.f, bond.f, sqwel.f, sqshlder.f and nc_sqwel.f has
// the same shape: an inner radius^2 A and an outer radius^2 B with
//   dA = b^2 - v^2 (r^2 - A),  dB = b^2 - v^2 (r^2 - B)
// and one of four roots: approach to A, (-b - sqrt dA)/v^2; exit through B,
// (-b + sqrt dB)/v^2; entry through B, (-b - sqrt dB)/v^2; and the stable
// exit form of bond.f:63, -(r^2 - B)/(sqrt dB + b).  The per-class rules
// below only choose A, B, the root and the type, by selects without a
// branch: the lanes of a batch hold pairs of different classes, and every
// class a divergent branch would run on its own.
__device__ inline void predict_geo(const DevTables& T, int code, int ia, int ic, bool bonded, double2 bwa,
                                   const Geo& g, double& tij, int& type) {
    const double b = g.b, r2 = g.r2, v2 = g.v2;
    const bool sqz = code >= 22 && code <= 26;
    const bool is_core = code <= 3 || (code >= 17 && code <= 26);
    const bool is_bond = code >= 4 && code <= 12;
    const bool is_nc = code == 15, is_well = code == 16, is_shl = code >= 40;
    const int cc = min((unsigned)code, 50u);
    // inner and outer radii squared
    const double ssq = T.sigma_sq[ia][ic];
    const double pe = T.ev_param[1][cc];
    const double q = T.sqz610[sqz ? code - 21 : 0][ia > ic ? ia : ic];
    const double wsq = *(is_shl ? &T.shlddia_sq[ia][ic] : &T.welldia_sq[ia][ic]);
    const double blmin = code >= 10 ? bwa.x : T.ev_param[2][cc], blmax = code >= 10 ? bwa.y : T.ev_param[3][cc];
    // the bonded N-C pair: core scaled by ev_param(1,15) twice, inside the
    // well by construction (nc_sqwel.f:76-101)
    const bool nc_own = is_nc && ia + ic != 5;
    const bool ncb = nc_own && bonded, ncu = nc_own && !bonded;
    const bool wl = (is_nc && !nc_own) || is_well || is_shl;
    double A = ssq * (pe * pe);         // core.f:27-31
    A = sqz ? A * (q * q) : A;
    A = wl || ncu ? ssq : A;            // sqwel.f, sqshlder.f, nc_sqwel.f: hard core unscaled
    A = ncb ? ssq * pe * pe : A;
    A = is_bond ? blmin * blmin : A;    // bond.f:19-31,70-81
    const double B = is_bond ? blmax * blmax : wsq;
    const double dA = b * b - v2 * (r2 - A);
    const double diff = r2 - B;
    const double dB = b * b - v2 * diff;
    const bool in = b < 0.0, pA = dA > 0.0, pB = dB > 0.0, inside = diff < 0.0;
    // root: r1 approach A, r2_ exit B, r3 enter B, r4 stable exit B
    const bool r1 = in && pA && (is_core || is_bond || ncb || (wl && inside));
    const bool r2_ = !r1 && ((is_bond && in && pB) || ncb || (wl && inside));
    const bool r3 = in && pB && (ncu || (wl && !inside));
    const bool r4 = is_bond && !in && pB;
    // types: N-C H-bond well 1/16/7, side-chain well 1/8/4, shoulder 1/10/12
    const int ex = is_bond ? 3 : (ncb || is_well ? 8 : (is_nc ? 16 : 10));
    const int en = ncu ? 9 : (is_nc ? 7 : (is_well ? 4 : 12));
    const int ty = r1 ? (is_bond ? 2 : 1) : (r2_ ? ex : (r4 ? 3 : en));
    const double sq = sqrt(r1 ? dA : dB);
    const double num = r4 ? -diff : (r2_ ? -b + sq : -b - sq);
    const double den = r4 ? sq + b : v2;
    const double t = num / den;
    const bool any = r1 || r2_ || r3 || r4;
    tij = any ? t : tij;
    type = any ? ty : type;
    if (!(is_core || is_bond || is_nc || is_well || is_shl)) type = -99;  // codes 13, 14, 27..39: error in ev_code matrix
}
__device__ inline void predict(const DevTables& T, int code, const Rec& a, const Rec& c, bool bonded, double2 bwa,
                               double tf, double& tij, int& type) {
    Geo g;
    geo(a, c, tf, g);
    predict_geo(T, code, dyn_ident(a.dyn), dyn_ident(c.dyn), bonded, bwa, g, tij, type);
}

// ------------------------------------------------------------------------
// wave helpers
// ------------------------------------------------------------------------
__device__ inline Rec shfl_rec(const Rec& r, int src) {
    Rec o;
    o.x = __shfl(r.x, src, kW);
    o.y = __shfl(r.y, src, kW);
    o.z = __shfl(r.z, src, kW);
    o.vx = __shfl(r.vx, src, kW);
    o.vy = __shfl(r.vy, src, kW);
    o.vz = __shfl(r.vz, src, kW);
    o.bm = __shfl(r.bm, src, kW);
    o.topo = __shfl(r.topo, src, kW);
    o.dyn = __shfl(r.dyn, src, kW);
    return o;
}
// Hand-off through LDS between the lanes of one wavefront: LDS operations
// of a wavefront complete in program order, so only the compiler's ordering
// is needed (no wait for outstanding global loads).
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// Hand-off of global-memory and LDS writes between the lanes of one
// wavefront (the stores complete before any lane reads past this point).
// Event-level code synchronises only its own wavefront: the other
// wavefronts of a system's workgroup meet it at the round barriers.
__device__ inline void wave_sync_mem() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
}
// Barrier of every wavefront of the system's workgroup, for the steps that
// all of them run together (list rebuilds, full rescans).
__device__ inline void wg_sync(int nw) {
    if (nw > 1)
        __syncthreads();
    else
        wave_sync_mem();
}

// scalar-register copies of wave-uniform values: what depends on them
// branches and addresses on the scalar unit instead of masking lanes
__device__ inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline int4 uni(int4 v) { return make_int4(uni(v.x), uni(v.y), uni(v.z), uni(v.w)); }
__device__ inline double uni(double v) {
    return __hiloint2double(uni(__double2hiint(v)), uni(__double2loint(v)));
}

// DPP lane moves: CTRL row_shr:n = 0x110+n, row_bcast:15 = 0x142,
// row_bcast:31 = 0x143; lanes without a valid source keep their own value
template <int CTRL, int RM>
__device__ inline int dpp_i(int v) {
    return __builtin_amdgcn_update_dpp(v, v, CTRL, RM, 0xf, false);
}
template <int CTRL, int RM>
__device__ inline double dpp_d(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = dpp_i<CTRL, RM>((int)b), hi = dpp_i<CTRL, RM>((int)(b >> 32));
    return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}
__device__ inline double readlane_d(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}
__device__ inline unsigned long long readlane_u64(unsigned long long v, int l) {
    return (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)v, l) |
           ((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(v >> 32), l) << 32);
}
// lanes of mask before this one (without a mask of the lanes below, which
// would stay in two registers)
__device__ inline int before_me(unsigned long long mask) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}
// first non-zero status of the wave (0 if none); wave-uniform
__device__ inline int wave_status(int v) {
    const unsigned long long m = __ballot(v != 0);
    return m ? __builtin_amdgcn_readlane(v, __ffsll((long long)m) - 1) : 0;
}
__device__ inline double wave_max(double v) {
    double o;
    o = dpp_d<0x111, 0xf>(v); v = o > v ? o : v;
    o = dpp_d<0x112, 0xf>(v); v = o > v ? o : v;
    o = dpp_d<0x114, 0xf>(v); v = o > v ? o : v;
    o = dpp_d<0x118, 0xf>(v); v = o > v ? o : v;
    o = dpp_d<0x142, 0xa>(v); v = o > v ? o : v;
    o = dpp_d<0x143, 0xc>(v); v = o > v ? o : v;
    return readlane_d(v, 63);
}
__device__ inline int wave_imax(int v) {
    v = max(v, dpp_i<0x111, 0xf>(v));
    v = max(v, dpp_i<0x112, 0xf>(v));
    v = max(v, dpp_i<0x114, 0xf>(v));
    v = max(v, dpp_i<0x118, 0xf>(v));
    v = max(v, dpp_i<0x142, 0xa>(v));
    v = max(v, dpp_i<0x143, 0xc>(v));
    return __builtin_amdgcn_readlane(v, 63);
}
// min of predictions (t, position) carrying partner and type
__device__ inline void wave_min_pred(double& t, int& p, int& m, int& ty) {
    for (int s = 1; s < kW; s <<= 1) {
        const double ot = __shfl_xor(t, s, kW);
        const int op = __shfl_xor(p, s, kW);
        const int om = __shfl_xor(m, s, kW);
        const int oty = __shfl_xor(ty, s, kW);
        if (ot < t || (ot == t && op < p)) {
            t = ot;
            p = op;
            m = om;
            ty = oty;
        }
    }
}

// Calendar key of one entry: order (bin, time, later add first), payload
// partner and type.  bc = bin << 8 | (coltype + 2); ip = index << 16 |
// (partner + 2).  Equal bins and times, which only bit-identical event
// times give, are settled by the entries' add stamps: the reference's
// bucket lists put each add at the head (add_tbin.f:28-32) and its stable
// sort keeps list order among equal times (main.F90:521-545), so the entry
// added last is taken first.
struct Key {
    double t;
    int bc;
    unsigned ip;
};
constexpr int kEmptyBc = INT_MAX;
constexpr int kStampBits = 20;  // adds per event: up to N + 4 in a sync's list rebuild
__device__ inline unsigned long long mk_stamp(long long coll, int sub) {
    return ((unsigned long long)coll << kStampBits) | (unsigned long long)(unsigned)sub;
}
// stamps live in HBM and are read and written at the device's L2 (other
// wavefronts of the workgroup write them)
__device__ inline void stamp_set(int k, unsigned long long v) {
    __hip_atomic_store((GLB unsigned long long*)(sdev().stamp + k), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned long long stamp_get(int k) {
    return __hip_atomic_load((GLB unsigned long long*)(sdev().stamp + k), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// a before b in the order above, with a's and b's stamps given (entries not
// yet written: a round's new keys)
__device__ inline bool key_less_st(const Key& a, unsigned long long sa, const Key& b, unsigned long long sb) {
    const int ab = a.bc >> 8, bb = b.bc >> 8;
    if (ab != bb) return ab < bb;
    if (a.t != b.t) return a.t < b.t;
    if (a.bc == kEmptyBc || sa == sb) return a.ip < b.ip;
    return sa > sb;
}
// a before b, both entries of the calendar (their stamps written).  Only
// shared order proxies come here, a few times in a million entries: out of
// line, so that the event loop's code stays small.
__device__ __noinline__ bool key_less(Key a, Key b) {
    const int ab = a.bc >> 8, bb = b.bc >> 8;
    if (ab != bb) return ab < bb;
    if (a.t != b.t) return a.t < b.t;
    if (a.bc == kEmptyBc || a.ip == b.ip) return a.ip < b.ip;
    const unsigned long long sa = stamp_get((int)(a.ip >> 16)), sb = stamp_get((int)(b.ip >> 16));
    return sa != sb ? sa > sb : a.ip < b.ip;
}
__device__ inline Key empty_key() {
    Key e;
    e.t = 0.0;
    e.bc = kEmptyBc;
    e.ip = 0xFFFFFFFFu;
    return e;
}
__device__ inline int key_bin(const Key& k) { return k.bc >> 8; }
__device__ inline int key_ct(const Key& k) { return (k.bc & 0xff) - 2; }
__device__ inline int key_idx(const Key& k) { return (int)(k.ip >> 16); }
__device__ inline int key_p(const Key& k) { return (int)(k.ip & 0xFFFFu) - 2; }
__device__ inline Key leaf_key(const Leaf& lf, int idx) {
    const int bin = leaf_bin(lf.meta);
    if (bin < 0) return empty_key();
    Key k;
    k.t = lf.tim;
    k.bc = (bin << 8) | (leaf_ct(lf.meta) + 2);
    k.ip = ((unsigned)idx << 16) | (unsigned)(lf.nptnr + 2);
    return k;
}
__device__ inline Key readlane_key(const Key& k, int l) {
    Key r;
    r.t = readlane_d(k.t, l);
    r.bc = __builtin_amdgcn_readlane(k.bc, l);
    r.ip = (unsigned)__builtin_amdgcn_readlane((int)k.ip, l);
    return r;
}

// per-system register state
struct Sc {
    double tfalse, t, interval, interval_max, t_fact, n_forced, sortsize, tbin_off, old_tfalse;
    long long coll, numghosts, nupdates, nforced, target;
    unsigned long long rc0, rc1;
    int nbin, status;
    long long nev[32];  // tally by resolved coltype (main.F90:926)
};

__device__ inline int calc_bin(const Sc& c, double tim, bool uncond, int& status) {
    if (!uncond && !(tim < c.interval_max)) return -1;
    int j = (int)((tim + c.tbin_off) / c.sortsize) + 1;
    if (j > kNumbin) j = kNumbin;  // -Ddebugging clamp, add_tbin.f:20-23
    if (j < 0) {
        // a negative time already reported (events.f:59-73 stops there) keeps its status
        if (!status) status = kErrBin;
        return -1;
    }
    // inserted behind the scan position: the reference's bucket scan
    // (main.F90:496-498) never returns to it before the next rebuild
    return j < c.nbin ? -1 : j;
}

// the same from values (calc_bin stays apart: through this one the loop spills a
// register more, 0.4 % of a 128-bead system's time)
__device__ inline int bin_of(double interval_max, double tbin_off, double sortsize, int nbin, double tim, int& status) {
    if (!(tim < interval_max)) return -1;
    int j = (int)((tim + tbin_off) / sortsize) + 1;
    if (j > kNumbin) j = kNumbin;
    if (j < 0) {
        if (!status) status = kErrBin;
        return -1;
    }
    return j < nbin ? -1 : j;
}

// flags: kPairReadsSp = the outcome resolution read the shoulder set or an
// H-bond partner; kPairWroteSp = the event rewrote them
constexpr int kPairReadsSp = 1, kPairWroteSp = 2;
struct Pair {  // the event's colliding pair (j < 0 for a ghost event)
    int i, j, flags, pad;
    Rec ri, rj;
    double2 bwi, bwj;
    int4 xi, xj;
};

constexpr int kMaxSpec = 8;  // full recomputes batched with the pair's own
// per-owner minimum of a prediction batch: LDS atomics on (time, position)
struct MinSlot {
    unsigned long long tkey;
    unsigned packed;  // position << 21 | (type + 1) << 16 | partner
    int pad;
};
// a down-set bead whose full recompute is batched with the pair's
struct SpecInfo {
    Rec r;
    double2 bw;
    int4 x;
    int l, nu, nx, off;
};
// a down-set bead's own data, read by the lanes that predict its single-pair
// updates inside the batch
struct DownInfo {
    Rec r;
    int4 o;
    double2 bw;
};
// time as an unsigned key with the order of the doubles (-0 as +0)
__device__ inline unsigned long long t_order(double t) {
    if (t == 0.0) t = 0.0;
    const unsigned long long b = (unsigned long long)__double_as_longlong(t);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}


// lanes of the selection: the pool's candidates, then the committed
// events' new entries, then up to 8 popped entries that were not committed
constexpr int kCandMax = 24, kFreshMax = 32;
// One round of a multi-wavefront system: the popped calendar entries (in
// key order, one per wavefront) and what each wavefront reports back.
struct Batch {
    Key key[kMaxWaves];   // popped entries
    Key knew[kMaxWaves];  // least key among the wavefront's new calendar entries
    unsigned long long knew_st[kMaxWaves];  // its add stamp
    int ty[kMaxWaves];    // resolved type of each event
    int nbl;              // blocks to rescan in wavefront 0's list (multi-pass forms)
    int st[kMaxWaves];    // status after each event
    int wdone[kMaxWaves]; // the wavefront's committed entries are written
    int st_rep[kMaxWaves];  // status of its replayed updates
    int K;                // entries popped this round (0: stop)
    int cut;              // first wavefront whose event is not committed
    int rebuild;          // the round's sync event rebuilds the lists
    unsigned long long moved;    // largest displacement of a sync event, as ordered bits
    // The pool the next round is selected from: every calendar entry whose
    // proxy lies below `edge` and that the round in flight has not popped is
    // in cand (as of the round's start) or, rewritten by a committed event
    // of the round, in that event's wavefront's share of fresh.
    double edge;
    double width;                // time the edge lies ahead of the round's last event
    int ncand;
    int full;                    // the pool is not complete: collect it again before selecting
    int nfresh[kMaxWaves];
    int order[kMaxWaves];        // lane of the entry of each rank (selection)
    Key cand[kCandMax];
    Key fresh[kFreshMax];
    // blocks with rewritten entries, a bit per block and a word per 64
    // blocks, by the round's parity: one is written while the other is
    // worked off
    unsigned long long dirty[2][kSup];
    int gbead;            // the bead of a ghost event leading the round
    long long t0;         // start of a budgeted launch (wall_clock64)
    Leaf pseudo[3];       // the ghost, sync and output entries across a list rebuild
    int share[3];         // taken so far of a list rebuild's search, sort and events
};
// Order proxy of a calendar key: a positive double with the bin in its
// exponent field (bins 1 to kNumbin = 2000 of 2046 values) and the top 52
// bits below the sign of the time in its mantissa (negative times as 0);
// +infinity for no entry.  Proxies order keys as key_less does except that
// distinct keys may share one; the reductions below take the minimum proxy
// and settle shared proxies with key_less.  As doubles they need one
// instruction per step for the minimum where 64-bit integers need a compare
// and two selects, and no proxy is a NaN or a denormal (bins start at 1).
__device__ inline double key_proxy(const Key& k) {
    const long long b = __double_as_longlong(k.t);
    const int hi = (int)(b >> 32);
    const unsigned h = (unsigned)max(hi, 0), l = hi < 0 ? 0u : (unsigned)b;
    const unsigned ph = ((unsigned)(k.bc >> 8) << 20) | (h >> 11), pl = (h << 21) | (l >> 11);
    const bool none = k.bc == kEmptyBc;
    return __hiloint2double(none ? 0x7FF00000 : (int)ph, none ? 0 : (int)pl);
}
constexpr int kInfHi = 0x7FF00000;
__device__ inline bool proxy_none(double p) { return __double2hiint(p) == kInfHi; }
// v_min_f64 without the quieting of its operands that the compiler puts
// before it; the wait states that a lane move of the result needs follow
__device__ inline double min_raw(double a, double b) {
    double r;
    asm("v_min_f64 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// a lane move in which every lane has a source (row_ror:n = 0x120 + n)
template <int CTRL>
__device__ inline double ror_d(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// minimum over each row of 16 lanes, in all of its lanes
__device__ inline double row_min(double v) {
    v = min_raw(v, ror_d<0x121>(v));
    v = min_raw(v, ror_d<0x122>(v));
    v = min_raw(v, ror_d<0x124>(v));
    return min_raw(v, ror_d<0x128>(v));
}
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
// minimum over the wave, in every lane
__device__ inline double wave_min(double v) {
    v = row_min(v);
    {
        const unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
        const u32x2 l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const u32x2 h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        v = min_raw(__hiloint2double((int)h.x, (int)l.x), __hiloint2double((int)h.y, (int)l.y));
    }
    {
        const unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
        const u32x2 l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const u32x2 h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        v = min_raw(__hiloint2double((int)h.x, (int)l.x), __hiloint2double((int)h.y, (int)l.y));
    }
    return v;
}
// the lane of the least key among the lanes of `tie`, which share a proxy
__device__ __noinline__ int tie_lane(Key k, unsigned long long tie) {
    int src = __ffsll((long long)tie) - 1;
    Key r = readlane_key(k, src);
    unsigned long long rest = tie & (tie - 1);
    while (rest) {
        const int o_src = __ffsll((long long)rest) - 1;
        const Key o = readlane_key(k, o_src);
        rest &= rest - 1;
        if (key_less(o, r)) {
            r = o;
            src = o_src;
        }
    }
    return src;
}
// minimum over the wave, returned to every lane
__device__ inline Key key_min_wave(const Key& k) {
    const double p = key_proxy(k), m = wave_min(p);
    if (proxy_none(readlane_d(m, 0))) return empty_key();
    const unsigned long long tie = __ballot(p == m);
    return readlane_key(k, (tie & (tie - 1)) ? uni(tie_lane(k, tie)) : __ffsll((long long)tie) - 1);
}
// the lane of the least key among the lanes of `tie`, which share a proxy,
// with their add stamps given per lane (new entries, not yet written)
__device__ __noinline__ int tie_lane_st(Key k, unsigned long long st, unsigned long long tie) {
    int src = __ffsll((long long)tie) - 1;
    Key r = readlane_key(k, src);
    unsigned long long rs = readlane_u64(st, src);
    unsigned long long rest = tie & (tie - 1);
    while (rest) {
        const int o_src = __ffsll((long long)rest) - 1;
        rest &= rest - 1;
        const Key o = readlane_key(k, o_src);
        const unsigned long long os = readlane_u64(st, o_src);
        if (key_less_st(o, os, r, rs)) {
            r = o;
            rs = os;
            src = o_src;
        }
    }
    return src;
}
// minimum over the wave of keys with their add stamps, returned to every
// lane with its stamp
__device__ inline Key key_min_wave_st(const Key& k, unsigned long long st, unsigned long long& out_st) {
    const double p = key_proxy(k), mn = wave_min(p);
    out_st = 0;
    if (proxy_none(readlane_d(mn, 0))) return empty_key();
    const unsigned long long tie = __ballot(p == mn);
    const int src = (tie & (tie - 1)) ? uni(tie_lane_st(k, st, tie)) : __ffsll((long long)tie) - 1;
    out_st = readlane_u64(st, src);
    return readlane_key(k, src);
}

// LDS views, one set per wavefront: the calendar tree, the master scalars
// and the round record are shared, the work lists are the wavefront's own
struct Lds {
    int o_blk, o_wm, o_wx, o_blist, o_pair, o_sc, o_leaf, o_wd, o_wt, o_wy, o_slot, o_spec, o_down;
    int o_msc, o_batch, o_mark, o_one, o_pool;
    int nwr;  // wavefronts of a list rebuild that have scratch in the pool
    Leaf* leaf;  // calendar leaves in HBM when they do not fit in LDS
    unsigned mark_mask;  // footprint mark of bead b: word b & mark_mask
    int nblk, nsup, maxw, nw;
    bool leaf_lds;
    __device__ int* wm() const { return reinterpret_cast<int*>(smem + o_wm); }  // work list: partner / bead
    __device__ int* wx() const { return reinterpret_cast<int*>(smem + o_wx); }  // work list: owner / op tag
    __device__ double* wt() const { return reinterpret_cast<double*>(smem + o_wt); }  // predicted times
    __device__ int* wy() const { return reinterpret_cast<int*>(smem + o_wy); }  // (type + 1) << 16 | partner
    __device__ int* blist() const { return reinterpret_cast<int*>(smem + o_blist); }  // blocks to rescan
    __device__ MinSlot* slot() const { return reinterpret_cast<MinSlot*>(smem + o_slot); }
    __device__ SpecInfo* spec() const { return reinterpret_cast<SpecInfo*>(smem + o_spec); }
    __device__ DownInfo* down() const { return reinterpret_cast<DownInfo*>(smem + o_down); }
    __device__ Pair* pair() const { return reinterpret_cast<Pair*>(smem + o_pair); }
    __device__ Sc* sc() const { return reinterpret_cast<Sc*>(smem + o_sc); }
    __device__ Sc* msc() const { return reinterpret_cast<Sc*>(smem + o_msc); }
    __device__ Batch* batch() const { return reinterpret_cast<Batch*>(smem + o_batch); }
    __device__ Leaf* lleaf() const { return reinterpret_cast<Leaf*>(smem + o_leaf); }
};
// the Lds views themselves (one per wavefront), after the SysDev copy
constexpr int kLdOff = kSdOff + (int)((sizeof(SysDev) + 15) / 16 * 16);
constexpr int kLdStride = (int)((sizeof(Lds) + 15) / 16 * 16);
__device__ inline const Lds& ldsv() { return *reinterpret_cast<const Lds*>(smem + kLdOff + wave_id() * kLdStride); }
// the shared blocks that make_lds lays out after the views
constexpr int kMscOff = kLdOff + kLdStride * kMaxWaves;
constexpr int kBatchOff = kMscOff + (int)((sizeof(Sc) + 15) / 16 * 16);
__device__ inline Sc& master() { return *reinterpret_cast<Sc*>(smem + kMscOff); }
__device__ inline Batch& round_rec() { return *reinterpret_cast<Batch*>(smem + kBatchOff); }
template <class T>
__device__ inline T* sgpr_ptr(T* p) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (T*)(((unsigned long long)hi << 32) | lo);
}
// The wavefront's views as a value in scalar registers, for functions with
// many wave fences (after each one the compiler would read a view's offset
// from LDS again before using it).
__device__ inline Lds lds_regs() {
    const Lds& m = ldsv();
    Lds r;
    r.o_blk = __builtin_amdgcn_readfirstlane(m.o_blk);
    r.o_wm = __builtin_amdgcn_readfirstlane(m.o_wm);
    r.o_wx = __builtin_amdgcn_readfirstlane(m.o_wx);
    r.o_blist = __builtin_amdgcn_readfirstlane(m.o_blist);
    r.o_pair = __builtin_amdgcn_readfirstlane(m.o_pair);
    r.o_sc = __builtin_amdgcn_readfirstlane(m.o_sc);
    r.o_leaf = __builtin_amdgcn_readfirstlane(m.o_leaf);
    r.o_wd = __builtin_amdgcn_readfirstlane(m.o_wd);
    r.o_wt = __builtin_amdgcn_readfirstlane(m.o_wt);
    r.o_wy = __builtin_amdgcn_readfirstlane(m.o_wy);
    r.o_slot = __builtin_amdgcn_readfirstlane(m.o_slot);
    r.o_spec = __builtin_amdgcn_readfirstlane(m.o_spec);
    r.o_down = __builtin_amdgcn_readfirstlane(m.o_down);
    r.o_msc = __builtin_amdgcn_readfirstlane(m.o_msc);
    r.o_batch = __builtin_amdgcn_readfirstlane(m.o_batch);
    r.o_mark = __builtin_amdgcn_readfirstlane(m.o_mark);
    r.o_one = __builtin_amdgcn_readfirstlane(m.o_one);
    r.o_pool = __builtin_amdgcn_readfirstlane(m.o_pool);
    r.nwr = __builtin_amdgcn_readfirstlane(m.nwr);
    r.leaf = sgpr_ptr(m.leaf);
    r.nblk = __builtin_amdgcn_readfirstlane(m.nblk);
    r.nsup = __builtin_amdgcn_readfirstlane(m.nsup);
    r.maxw = __builtin_amdgcn_readfirstlane(m.maxw);
    r.nw = __builtin_amdgcn_readfirstlane(m.nw);
    r.leaf_lds = __builtin_amdgcn_readfirstlane(m.leaf_lds ? 1 : 0) != 0;
    r.mark_mask = (unsigned)__builtin_amdgcn_readfirstlane((int)m.mark_mask);
    return r;
}
// a leaf another wavefront of the workgroup has just written (its HBM copy
// read past the vector L1)
__device__ inline Leaf leaf_get_fresh(const Lds& L, int k) {
    if (L.leaf_lds) return L.lleaf()[k];
    unsigned long long* q = reinterpret_cast<unsigned long long*>(L.leaf + k);
    const unsigned long long a = __hip_atomic_load((GLB unsigned long long*)q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long b = __hip_atomic_load((GLB unsigned long long*)(q + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    Leaf r;
    r.tim = __longlong_as_double((long long)a);
    r.nptnr = (int)(unsigned)b;
    r.meta = (int)(unsigned)(b >> 32);
    return r;
}
__device__ inline unsigned* lds_words(int off) { return (unsigned*)__builtin_assume_aligned(smem + off, 16); }
// What the event loop reads of its system and of the LDS plan, as values
// that stay in scalar registers for the whole launch.
struct Hot {
    Rec* rec;
    double2* bw;
    int4* extra;
    int4* ovr;
    int* nb_up;
    int* nb_dn;
    int* nup;
    int* ndn;
    Leaf* leaf;
    unsigned long long* stamp;
    unsigned mark_mask;
    int N, cap, nblk, nsup, o_blk, o_leaf, o_mark, o_w;
    bool leaf_lds;
};
__device__ inline Hot load_hot(const SysDev& S, const Lds& L) {
    Hot H;
    H.rec = sgpr_ptr(S.rec);
    H.bw = sgpr_ptr(S.bw);
    H.extra = sgpr_ptr(S.extra);
    H.ovr = sgpr_ptr(S.ovr);
    H.nb_up = sgpr_ptr(S.nb_up);
    H.nb_dn = sgpr_ptr(S.nb_dn);
    H.nup = sgpr_ptr(S.nup);
    H.ndn = sgpr_ptr(S.ndn);
    H.leaf = sgpr_ptr(S.leaf);
    H.mark_mask = (unsigned)uni((int)L.mark_mask);
    H.stamp = sgpr_ptr(S.stamp);
    H.N = uni(S.N);
    H.cap = uni(S.cap);
    H.nblk = uni(L.nblk);
    H.nsup = uni(L.nsup);
    H.o_blk = uni(L.o_blk);
    H.o_leaf = uni(L.o_leaf);
    H.o_mark = uni(L.o_mark);
    H.o_w = uni(L.o_one);
    H.leaf_lds = uni(L.leaf_lds ? 1 : 0) != 0;
    return H;
}
// element i of a buffer: scalar base, 32-bit byte offset
template <class T>
__device__ inline T ld_at(const T* base, int i) {
    const GLB char* q = (const GLB char*)base + (unsigned)i * (unsigned)sizeof(T);
    if constexpr (sizeof(T) % 16 == 0) {
        u32x4 t[sizeof(T) / 16];
#pragma unroll
        for (int k = 0; k < (int)(sizeof(T) / 16); ++k) t[k] = ((const GLB u32x4*)q)[k];
        T r;
        __builtin_memcpy(&r, t, sizeof(T));
        return r;
    } else
        return *(const GLB T*)q;
}
template <class T>
__device__ inline void st_at(T* base, int i, const T& v) {
    GLB char* q = (GLB char*)base + (unsigned)i * (unsigned)sizeof(T);
    u32x4 t[sizeof(T) / 16];
    __builtin_memcpy(t, &v, sizeof(T));
#pragma unroll
    for (int k = 0; k < (int)(sizeof(T) / 16); ++k) ((GLB u32x4*)q)[k] = t[k];
}
// calendar entry k, V: Lds or Hot
template <class V>
__device__ inline Leaf leaf_ld(const V& H, int k) {
    return H.leaf_lds ? reinterpret_cast<const Leaf*>(smem + H.o_leaf)[k] : ld_at(H.leaf, k);
}
template <class V>
__device__ inline void leaf_st(const V& H, int k, const Leaf& v) {
    if (H.leaf_lds)
        reinterpret_cast<Leaf*>(smem + H.o_leaf)[k] = v;
    else
        st_at(H.leaf, k, v);
}
__device__ inline void stamp_st(const Hot& H, int k, unsigned long long v) {
    __hip_atomic_store((GLB unsigned long long*)((GLB char*)H.stamp + (unsigned)k * 8u), v, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline void dirty_or(int par, int blk) {
    __hip_atomic_fetch_or(&round_rec().dirty[par][blk / kSup], 1ull << (blk & (kSup - 1)), __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_WORKGROUP);
}
// A calendar entry's time as the block minima hold it: the bits of the
// nearest float (negative times as 0), in the order of the times except that
// near ones may share a value; +infinity for no entry.  The minima only say
// which blocks can hold an entry below a time, so four bytes per block and
// one instruction per reduction step do: the exact keys are compared where
// entries are taken.
constexpr unsigned kNoTime = 0x7F800000u;
__device__ inline unsigned leaf_time(const Leaf& lf) {
    const float f = (float)lf.tim;
    const unsigned u = (unsigned)max(__float_as_int(f), 0);
    return leaf_bin(lf.meta) < 0 ? kNoTime : u;
}
template <int CTRL>
__device__ inline unsigned ror_min(unsigned v) {
    return min(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true));
}
// U entries of the calendar per lane (index -1: none), all loads in flight
// together: a branch on where the leaves are around each one waited for it
template <int U>
__device__ inline void leaves_ld(const Hot& H, const int (&idx)[U], Leaf (&lf)[U]) {
    if (H.leaf_lds) {
#pragma unroll
        for (int u = 0; u < U; ++u) lf[u] = reinterpret_cast<const Leaf*>(smem + H.o_leaf)[max(idx[u], 0)];
    } else {
#pragma unroll
        for (int u = 0; u < U; ++u) lf[u] = ld_at(H.leaf, max(idx[u], 0));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) lf[u].meta = idx[u] >= 0 ? lf[u].meta : 0;
}
// minima of the blocks in the list: one row of 16 lanes per block, 32 blocks
// per step so that eight independent reductions overlap
__device__ inline void rescan_listed(const Hot& H, const int* list, int nb) {
    const int lane = lane_id(), N3 = H.N + 3;
    unsigned* const blk = lds_words(H.o_blk);
    for (int base = 0; base < nb; base += 32) {
        unsigned v[8];
        int bq[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int q = base + 4 * u + (lane >> 4);
            bq[u] = q < nb ? list[q] : -1;
        }
        Leaf lf[8];
        int idx[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int k = bq[u] * kBlk + (lane & 15);
            idx[u] = bq[u] >= 0 && k < N3 ? k : -1;
        }
        leaves_ld(H, idx, lf);
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = leaf_time(lf[u]);
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = ror_min<0x121>(v[u]);
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = ror_min<0x122>(v[u]);
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = ror_min<0x124>(v[u]);
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = ror_min<0x128>(v[u]);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if ((lane & 15) == 0 && bq[u] >= 0) blk[bq[u]] = v[u];
    }
}
constexpr int kListMax = 512;  // blocks of a work list (one wavefront's one-pass area, OnePass)
// Adds the blocks 64 s + bit of mask to the list.
__device__ inline int list_blocks(int* list, int n, int s, unsigned long long mask) {
    const int lane = lane_id();
    if ((mask >> lane) & 1ull) list[n + before_me(mask)] = s * kSup + lane;
    return n + __popcll(mask);
}
// The block minima after the entries of the blocks in Batch::dirty[par]
// changed (one wavefront; the mask is cleared).
__device__ inline void tree_update(const Hot& H, int par, int* list) {
    const int lane = lane_id();
    Batch& B = round_rec();
    unsigned long long d = 0;
    if (lane < H.nsup) {
        d = B.dirty[par][lane];
        B.dirty[par][lane] = 0;
    }
    unsigned long long sm = __ballot(d != 0);
    int n = 0;
    while (sm) {
        const int s = __ffsll((long long)sm) - 1;
        sm &= sm - 1;
        n = list_blocks(list, n, s, readlane_u64(d, s));
        if (n > kListMax - kSup || !sm) {
            wave_sync();
            rescan_listed(H, list, n);
            wave_sync();
            n = 0;
        }
    }
}
// The pool of the next selection from the up-to-date block minima (one
// wavefront): every entry whose proxy lies below an edge, the K entries
// popped by the round in flight left out.  The edge lies Batch::width after
// t0; the width follows the density of events so that the pool holds a few
// more entries than a round takes (`want`), tried again up to `tries` times.
// Left with too many entries for the pool, it is empty (edge 0: nothing lies
// below it).
// meet: the wavefront owes the round's first barrier, where the others
// exchange footprint marks; it meets them once it has looked over the block
// minima, which with tree_update takes about as long as they need to get
// there.  With the barrier before that they waited at their second one for
// the collection's end: 1 700 cycles of each round at 6144 beads, 4 000 at
// 23 424.
__device__ inline void collect_pool(const Hot& H, int K, double t0, int want, int tries, int* list, bool meet) {
    const int lane = lane_id(), N3 = H.N + 3;
    Batch& B = round_rec();
    const Sc& c = master();
    const unsigned* const blk = lds_words(H.o_blk);
    const double off = c.tbin_off, sortsize = c.sortsize, imax = c.interval_max;
    double w = B.width;
    // the popped entries are the calendar's least: all proxies below the
    // last one's, and those that share its proxy by index
    const Key kl = B.key[K > 0 ? K - 1 : 0];
    const double pl = K > 0 ? key_proxy(kl) : -1.0;
    const int il = K > 0 ? key_idx(kl) : -1;
    int count = 0;
    double edge = 0.0;
    for (int tr = 0; tr < tries; ++tr) {
        Key ek;
        ek.t = t0 + w;
        const int bin = (int)min((ek.t + off) / sortsize, (double)kNumbin) + 1;
        ek.bc = min(max(bin, 1), kNumbin) << 8;
        ek.ip = 0;
        edge = key_proxy(ek);
        // blocks that can hold an entry below the edge (its time rounded up:
        // bins and times agree to far less than a float's spacing)
        const unsigned te = (unsigned)max(__float_as_int((float)ek.t), 0) + 2u;
        int n = 0;
        bool many = false;
        for (int s0 = 0; s0 < H.nsup && !many; s0 += 8) {
            unsigned v[8], least = kNoTime;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int b = (s0 + u) * kSup + lane;
                v[u] = blk[min(b, H.nblk - 1)];
                v[u] = b < H.nblk ? v[u] : kNoTime;
                least = min(least, v[u]);
            }
            if (__ballot(least < te) == 0) continue;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const unsigned long long m = __ballot(v[u] < te);
                if (m) n = list_blocks(list, n, s0 + u, m);
                many = many || n > kListMax - kSup;
                if (many) break;
            }
        }
        wave_sync();
        if (meet) __syncthreads();
        meet = false;
        // their entries below it
        count = 0;
        for (int base = 0; base < n && !many; base += 16) {
            Leaf lf[4];
            int idx[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int q = base + 4 * u + (lane >> 4), k = (q < n ? list[q] : H.nblk) * kBlk + (lane & 15);
                idx[u] = k < N3 ? k : -1;
            }
            leaves_ld(H, idx, lf);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (base + 4 * u >= n) continue;
                const Key e = leaf_key(lf[u], idx[u]);
                const double p = key_proxy(e);
                bool in = p < edge && p >= pl && idx[u] != il;
                if (__ballot(in && p == pl)) {
                    for (int q = 0; q < K; ++q) in = in && uni(key_idx(B.key[q])) != idx[u];
                }
                const unsigned long long m = __ballot(in);
                const int pos = count + before_me(m);
                if (in && pos < kCandMax) B.cand[pos] = e;
                count += __popcll(m);
            }
            many = count > kCandMax;
        }
        if (many) {
            w *= 0.5;
            count = kCandMax + 1;
        } else if (count < want && ek.t < imax) {
            w *= count == 0 ? 4.0 : 1.6;
        } else {
            if (count > want + 6) w *= 0.9;
            break;
        }
    }
    if (lane == 0) {
        B.width = w;
        B.ncand = count > kCandMax ? 0 : count;
        B.edge = count > kCandMax ? 0.0 : edge;
    }
    wave_sync();
}

// every block minimum; all wavefronts of the system take part
__device__ inline void rescan_all(const Hot& H, int wave, int nw) {
    const int lane = lane_id(), N3 = H.N + 3;
    unsigned* const blk = lds_words(H.o_blk);
    for (int base = 4 * wave; base < H.nblk; base += 4 * nw) {
        const int b = base + (lane >> 4), idx = b * kBlk + (lane & 15);
        unsigned v = kNoTime;
        if (idx < N3) v = leaf_time(leaf_ld(H, idx));
        v = ror_min<0x121>(v);
        v = ror_min<0x122>(v);
        v = ror_min<0x124>(v);
        v = ror_min<0x128>(v);
        if ((lane & 15) == 0 && b < H.nblk) blk[b] = v;
    }
}

// ------------------------------------------------------------------------
// multi-wavefront rounds: footprint marks and the accepted prefix
// ------------------------------------------------------------------------
// shoulder beads of an H-bond pair (repuls_add.f:16-25): N bead i, C bead j
__device__ inline void shoulder_idx(int i, int Li, int j, int Lj, int& ncim1, int& ncai, int& ncaj, int& nnjp1) {
    ncim1 = i + Li - 1;
    ncai = i - Li;
    ncaj = j - 2 * Lj;
    nnjp1 = j - Lj + 1;
}

// Lane's bead of the shoulder set an event on (i, j) may read or rewrite
// (main.F90:1487-1634 via repuls_check/_3, repuls_add/_del_a/_del_b and the
// H-bond partner's identity): the H-bond partners of i and j (lanes 0, 1)
// and the shoulder beads of (i,j), (j,i), (i,hbp(i)), (hbp(i),i),
// (j,hbp(j)), (hbp(j),j) (lanes 2..25); -1 where there is none
__device__ inline int shoulder_bead(const SysDev&, const Pair& P, int lane) {
    const SysDev& S = sdev();
    const int hi = P.xi.w, hj = P.j >= 0 ? P.xj.w : -1;
    if (lane == 0) return hi;
    if (lane == 1) return hj;
    if (lane >= 26 || P.j < 0) return -1;
    const int g = (lane - 2) >> 2, q = (lane - 2) & 3;
    const int x = g < 2 ? P.i : (g < 4 ? P.i : P.j);
    const int y = g < 2 ? P.j : (g < 4 ? hi : hj);
    if (y < 0) return -1;
    const int tx = x == P.i ? P.ri.topo : P.rj.topo;
    const int ty = y == P.i ? P.ri.topo : (y == P.j ? P.rj.topo : gl1(&S.rec[y].topo));
    const bool swap = (g & 1) != 0;
    const int n = swap ? y : x, cb = swap ? x : y;
    const int Ln = topo_len(swap ? ty : tx), Lc = topo_len(swap ? tx : ty);
    int a[4];
    shoulder_idx(n, Ln, cb, Lc, a[0], a[1], a[2], a[3]);
    const int v = q == 0 ? a[0] : (q == 1 ? a[1] : (q == 2 ? a[2] : a[3]));
    return (v >= 0 && v < S.N) ? v : -1;
}
// Footprint marks of bead b, in LDS (V: Lds or Hot).  Where a word per bead
// does not fit, the words are shared (b & mark_mask): a shared word can only
// end a round earlier or replay an update on an entry that nobody rewrote.
template <class V>
__device__ inline unsigned* mark_word(const V& L, int b) {
    return lds_words(L.o_mark) + ((unsigned)b & L.mark_mask);
}
template <class V>
__device__ inline void mark_or(const V& L, int b, unsigned bits) {
    __hip_atomic_fetch_or(mark_word(L, b), bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline unsigned mark_get(const Hot& L, int b) {
    return __hip_atomic_load(mark_word(L, b), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <class V>
__device__ inline void mark_clear(const V& L, int b) {
    __hip_atomic_store(mark_word(L, b), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// A wavefront's place in a multi-wavefront round: -1 alone; 0 the round's
// first event (always committed, writes as it goes); k >= 1 a speculative
// event whose writes wait for the round's checks.  In a round every
// wavefront passes the kRoundBars round barriers once (footprints marked,
// new calendar keys known), whichever way it leaves.
constexpr int kRoundBars = 2;
__device__ inline void bar_to(int& nb, int n) {
    while (nb < n) {
        __syncthreads();
        ++nb;
    }
}
__device__ inline void spec_abort_at(int bk, int& nb) {
    if (lane_id() == 0) atomicMin(&round_rec().cut, bk);
    bar_to(nb, kRoundBars);
}

__device__ inline void round_clear_marks(const Lds& L, const SysDev& S, int dent, int i, int j, int sp) {
    const int lane = lane_id();
    if (dent >= 0) mark_clear(L, dent);
    if (lane == 0) mark_clear(L, i);
    if (lane == 1 && j >= 0) mark_clear(L, j);
    if (sp >= 0) mark_clear(L, sp);
}
// Events of a round committed: the prefix before the first cut-off event,
// before the first event after an error, and before the first event whose
// key is not below every new calendar key of the events before it (the
// serial order would have run one of those first).
__device__ __noinline__ int batch_accepted() {
    const Batch& B = round_rec();
    int A = min(B.K, B.cut);
    Key lo = B.knew[0];
    unsigned long long lo_st = B.knew_st[0];
    if (B.st[0] != 0) A = min(A, 1);
    for (int k = 1; k < A; ++k) {
        const Key kk = B.key[k];
        // kk was added before the round began, lo during it: on equal bin
        // and time lo comes first (stamp 0 is older than every add)
        if (!key_less_st(kk, 0ull, lo, lo_st)) return k;
        if (B.st[k] != 0) return k + 1;
        if (key_less_st(B.knew[k], B.knew_st[k], lo, lo_st)) {
            lo = B.knew[k];
            lo_st = B.knew_st[k];
        }
    }
    return A;
}

// The same, one round entry per lane: an exclusive prefix minimum of the new
// keys' proxies against the popped keys' proxies; a shared proxy goes to the
// exact form above.  Uniform over the wavefront.
__device__ inline int accepted(const Batch& B) {
    const int lane = lane_id();
    const int top = uni(min(B.K, B.cut));
    const int q = lane & (kMaxWaves - 1);
    const bool in = lane < top;
    const int st = in ? B.st[q] : 0;
    const unsigned long long sm = __ballot(st != 0);
    if (__ballot(in && B.knew[q].bc != kEmptyBc) == 0) return sm ? min(top, (int)__ffsll((long long)sm)) : top;
    const double pk = key_proxy(B.key[q]);
    const double pn = in ? key_proxy(B.knew[q]) : __hiloint2double(kInfHi, 0);
    auto shr = [](double v, auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        return __hiloint2double(__builtin_amdgcn_update_dpp(kInfHi, __double2hiint(v), C, 0xf, 0xf, false),
                                __builtin_amdgcn_update_dpp(0, __double2loint(v), C, 0xf, 0xf, false));
    };
    double lo = shr(pn, std::integral_constant<int, 0x111>{});
    lo = min_raw(lo, shr(lo, std::integral_constant<int, 0x111>{}));
    lo = min_raw(lo, shr(lo, std::integral_constant<int, 0x112>{}));
    lo = min_raw(lo, shr(lo, std::integral_constant<int, 0x114>{}));
    const bool live = in && lane >= 1;
    if (__ballot(live && pk == lo)) return uni(batch_accepted());
    const unsigned long long fail = __ballot(live && pk > lo);
    int A = top;
    if (fail) A = min(A, __ffsll((long long)fail) - 1);
    if (sm) A = min(A, (int)__ffsll((long long)sm));
    return A;
}

// ------------------------------------------------------------------------
// rescheduling after an event: partial_events.f:16-201
// ------------------------------------------------------------------------
__device__ __noinline__ void shoulders_clear(int n, int Ln, int cb, int Lc);

// The list rows of i and j (lane k: slot k) with their lengths; they do not
// change between list rebuilds, so a pair event loads them before it
// resolves its outcome
struct Rows {
    int eui, edi, euj, edj;
    int nui, ndi, nuj, ndj;
};
__device__ inline Rows load_rows(const SysDev& S, int i, int j) {
    const int lane = lane_id(), cap = S.cap;
    const int jr = j >= 0 ? j : i;
    Rows r;
    r.nui = gl1(S.nup + (i));
    r.ndi = gl1(S.ndn + (i));
    r.nuj = j >= 0 ? gl1(S.nup + (j)) : 0;
    r.ndj = j >= 0 ? gl1(S.ndn + (j)) : 0;
    r.eui = lane < cap ? gl1(S.nb_up + ((size_t)i * cap + lane)) : 0;
    r.edi = lane < cap ? gl1(S.nb_dn + ((size_t)i * cap + lane)) : 0;
    r.euj = lane < cap ? gl1(S.nb_up + ((size_t)jr * cap + lane)) : 0;
    r.edj = lane < cap ? gl1(S.nb_dn + ((size_t)jr * cap + lane)) : 0;
    return r;
}
__device__ inline Rec load_rec(const SysDev&, const Pair& P, int m) {
    const SysDev& S = sdev();

    if (m == P.i) return P.ri;
    if (m == P.j) return P.rj;
    return gld(S.rec + (m));
}

// Cooperative full recompute of bead l (rl, bwl, xl wave-uniform): min over
// l's up list and upper shoulder partners (partial_events.f:121-139).
__device__ void full_one(const SysDev&, const Lds&, int l, const Rec& rl, double2 bwl, int4 xl, double tf,
                         double T0, double& tim, int& np, int& ct, int& status) {
    const Lds L = lds_regs();

    const SysDev& S = sdev();

    const DevTables& T = tabs();
    const Pair& P = *L.pair();
    const int lane = lane_id(), cap = S.cap;
    const int nu = gl1(S.nup + (l));
    const int nx = (xl.x > l ? 1 : 0) + (xl.y > l ? 1 : 0) + (xl.z > l ? 1 : 0);
    const int tot = nu + nx;
    double bt = 1e300;
    int bp = INT_MAX, bm = -1, bty = -1;
    for (int base = 0; base < tot; base += kW) {
        const int p = base + lane;
        if (p < tot) {
            int m, stat;
            if (p < nu) {
                const int ent = gl1(S.nb_up + ((size_t)l * cap + p));
                m = ent & 0xFFFFFF;
                stat = ent >> 24;
            } else {
                const int k = p - nu;
                int cnt = 0;
                m = -1;
                if (xl.x > l) {
                    if (cnt == k) m = xl.x;
                    ++cnt;
                }
                if (xl.y > l) {
                    if (cnt == k) m = xl.y;
                    ++cnt;
                }
                if (xl.z > l) {
                    if (cnt == k) m = xl.z;
                    ++cnt;
                }
                stat = -1;
            }
            const Rec rm = load_rec(S, P, m);
            const int4 om = gld(S.ovr + (m));
            if (stat < 0) stat = static_t(T, rm.topo, rl.topo);
            const int code = dyn_code(om, l, stat);  // ev_code(m, l), eventredo_up.f:28
            double tij = 1000000000.0;
            int ty = 0;
            predict(T, code, rl, rm, dyn_bptnr(rl.dyn) == m, bwl, tf, tij, ty);
            if (ty == -99) status = kErrBadCode;
            if (tij < 0.0 && fabs(tij) > 1.0e-10) status = kErrNegativeTime;
            if (tij < bt) {
                bt = tij;
                bp = p;
                bm = m;
                bty = ty;
            }
        }
    }
    wave_min_pred(bt, bp, bm, bty);
    if (bt < T0) {
        tim = bt + tf;
        np = bm;
        ct = bty;
    } else {
        tim = T0 + tf;
        np = -1;
        ct = -1;
    }
}

// eventredo_down.f: single-pair update of (st_t, st_p, st_c) of bead l
__device__ inline void single_update(const DevTables& T, const Rec& rl, int4 ol, double2 bwl, int p, const Rec& rp,
                                     double tf, double& st_t, int& st_p, int& st_c, bool& modified, int& status) {
    const int code = dyn_code(ol, p, static_t(T, rl.topo, rp.topo));  // ev_code(l, p)
    double tij = 1000000000.0;
    int ty = 0;
    predict(T, code, rl, rp, dyn_bptnr(rl.dyn) == p, bwl, tf, tij, ty);
    if (ty == -99) status = kErrBadCode;
    if (tij < 0.0 && fabs(tij) > 1.0e-10) status = kErrNegativeTime;
    tij = tij + tf;
    if (tij < st_t) {
        st_t = tij;
        st_p = p;
        st_c = ty;
        modified = true;
    }
}

// Generic form for any down-set size: full recomputes one at a time.
// extra_blk: a further calendar block to rescan (the ghost entry), or -1
__device__ void reschedule_generic(const SysDev&, const DevTables&, const Lds&, Sc&, const Pair&,
                                   int extra_blk, bool xpulse_del) {
    const Lds& L = ldsv();

    const SysDev& S = sdev();

    const DevTables& T = tabs();
    Sc& c = *L.sc();
    const Pair& P = *L.pair();

    const int lane = lane_id(), cap = S.cap;
    const int i = P.i, j = P.j;
    const double tf = c.tfalse;
    const double T0 = c.interval_max + kLt - tf;
    int status = 0;
    PH_BEGIN(tph);
    // ---- list rows of i and j, one entry per lane (cap <= 64)
    const int nui = gl1(S.nup + (i)), ndi = gl1(S.ndn + (i));
    const int nuj = j >= 0 ? gl1(S.nup + (j)) : 0, ndj = j >= 0 ? gl1(S.ndn + (j)) : 0;
    const int eui = lane < nui ? gl1(S.nb_up + ((size_t)i * cap + lane)) : 0;
    const int edi = lane < ndi ? gl1(S.nb_dn + ((size_t)i * cap + lane)) : 0;
    const int euj = lane < nuj ? gl1(S.nb_up + ((size_t)j * cap + lane)) : 0;
    const int edj = lane < ndj ? gl1(S.nb_dn + ((size_t)j * cap + lane)) : 0;
    // ---- work list: candidates of i (tag 0) and j (tag 1), then the down
    //      set with its op partner (tag 2: i, tag 3: j), in reference order
    const int xi0 = P.xi.x, xi1 = P.xi.y, xi2 = P.xi.z;
    const int xj0 = P.xj.x, xj1 = P.xj.y, xj2 = P.xj.z;
    int w = 0;
    if (lane < nui) {
        L.wm()[lane] = eui;
        L.wx()[lane] = 0;
    }
    w = nui;
    const int kNoStat = 0xFF << 24;
    if (xi0 > i) { if (lane == 0) { L.wm()[w] = xi0 | kNoStat; L.wx()[w] = 0; } ++w; }
    if (xi1 > i) { if (lane == 0) { L.wm()[w] = xi1 | kNoStat; L.wx()[w] = 0; } ++w; }
    if (xi2 > i) { if (lane == 0) { L.wm()[w] = xi2 | kNoStat; L.wx()[w] = 0; } ++w; }
    if (j >= 0) {
        if (lane < nuj) {
            L.wm()[w + lane] = euj;
            L.wx()[w + lane] = 1;
        }
        w += nuj;
        if (xj0 > j) { if (lane == 0) { L.wm()[w] = xj0 | kNoStat; L.wx()[w] = 1; } ++w; }
        if (xj1 > j) { if (lane == 0) { L.wm()[w] = xj1 | kNoStat; L.wx()[w] = 1; } ++w; }
        if (xj2 > j) { if (lane == 0) { L.wm()[w] = xj2 | kNoStat; L.wx()[w] = 1; } ++w; }
    }
    const int ncand = w;
    if (lane < ndi) {
        L.wm()[w + lane] = edi & 0xFFFF;
        L.wx()[w + lane] = 2;
    }
    w += ndi;
    if (xi0 >= 0 && xi0 < i) { if (lane == 0) { L.wm()[w] = xi0; L.wx()[w] = 2; } ++w; }
    if (xi1 >= 0 && xi1 < i) { if (lane == 0) { L.wm()[w] = xi1; L.wx()[w] = 2; } ++w; }
    if (xi2 >= 0 && xi2 < i) { if (lane == 0) { L.wm()[w] = xi2; L.wx()[w] = 2; } ++w; }
    if (j >= 0) {
        const int l = edj & 0xFFFF;
        const bool keep = lane < ndj && l != i;
        const unsigned long long bal = __ballot(keep);
        const int pre = before_me(bal);
        if (keep) {
            L.wm()[w + pre] = l;
            L.wx()[w + pre] = 3;
        }
        w += __popcll(bal);
        if (xj0 >= 0 && xj0 < j) { if (lane == 0) { L.wm()[w] = xj0; L.wx()[w] = 3; } ++w; }
        if (xj1 >= 0 && xj1 < j) { if (lane == 0) { L.wm()[w] = xj1; L.wx()[w] = 3; } ++w; }
        if (xj2 >= 0 && xj2 < j) { if (lane == 0) { L.wm()[w] = xj2; L.wx()[w] = 3; } ++w; }
    }
    const int nD = w - ncand;
    if (w > L.maxw) status = kErrListCapacity;
    wave_sync_mem();
    PH_END(S, kPhLoads, tph);
    // ---- candidate predictions of the full recomputes of i and j
    PH_ADDN(S, kPhNPred, min(ncand, L.maxw));
    PH_ADDN(S, kPhNPredPass, (ncand + kW - 1) / kW);
    double bt0 = 1e300, bt1 = 1e300;
    int bp0 = INT_MAX, bp1 = INT_MAX, bm0 = -1, bm1 = -1, bty0 = -1, bty1 = -1;
    for (int base = 0; base < ncand; base += kW) {
        const int q = base + lane;
        if (q < ncand && q < L.maxw) {
            const int ent = L.wm()[q];
            const int owner = L.wx()[q];
            const int m = ent & 0xFFFFFF;
            int stat = (ent >> 24) & 0xFF;
            const Rec rx = owner == 0 ? P.ri : P.rj;
            const int x = owner == 0 ? i : j;
            const Rec rm = load_rec(S, P, m);
            const int4 om = gld(S.ovr + (m));
            if (stat == 0xFF) stat = static_t(T, rm.topo, rx.topo);
            const int code = dyn_code(om, x, stat);  // ev_code(m, x)
            double tij = 1000000000.0;
            int ty = 0;
            predict(T, code, rx, rm, dyn_bptnr(rx.dyn) == m, owner == 0 ? P.bwi : P.bwj, tf, tij, ty);
            if (ty == -99) status = kErrBadCode;
            if (tij < 0.0 && fabs(tij) > 1.0e-10) status = kErrNegativeTime;
            if (owner == 0) {
                if (tij < bt0) {
                    bt0 = tij;
                    bp0 = q;
                    bm0 = m;
                    bty0 = ty;
                }
            } else if (tij < bt1) {
                bt1 = tij;
                bp1 = q;
                bm1 = m;
                bty1 = ty;
            }
        }
    }
    wave_min_pred(bt0, bp0, bm0, bty0);
    wave_min_pred(bt1, bp1, bm1, bty1);
    double ti = T0 + tf, tj = T0 + tf;
    int pi = -1, ci = -1, pj = -1, cj = -1;
    if (bt0 < T0) {
        ti = bt0 + tf;
        pi = bm0;
        ci = bty0;
    }
    if (bt1 < T0) {
        tj = bt1 + tf;
        pj = bm1;
        cj = bty1;
    }
    PH_END(S, kPhPred, tph);
    // ---- the down set: per unique bead, its I-ops then its J-ops
    if (lane == 0) {
        L.blist()[0] = i / kBlk;
        L.blist()[1] = j >= 0 ? j / kBlk : i / kBlk;
        L.blist()[2] = extra_blk >= 0 ? extra_blk : i / kBlk;
    }
    int nbl = 3;
    for (int base = 0; base < nD; base += kW) {
        const int q = base + lane;
        bool first = false, is_i = false;
        int l = -1, cI = 0, cJ = 0;
        if (q < nD && ncand + q < L.maxw) {
            l = L.wm()[ncand + q];
            first = true;
            for (int r = 0; r < q; ++r)
                if (L.wm()[ncand + r] == l) {
                    first = false;
                    break;
                }
            if (first)
                for (int r = 0; r < nD && ncand + r < L.maxw; ++r)
                    if (L.wm()[ncand + r] == l) {
                        if (L.wx()[ncand + r] == 2) ++cI;
                        else ++cJ;
                    }
            is_i = (l == i);
        }
        Rec rl = P.ri;
        int4 ol = make_int4(-1, -1, -1, -1), xl = make_int4(-1, -1, -1, -1);
        double2 bwl = make_double2(0.0, 0.0);
        double st_t = 0.0;
        int st_p = -1, st_c = -1;
        if (first) {
            rl = load_rec(S, P, l);
            ol = gld(S.ovr + (l));
            bwl = gld(S.bw + (l));
            xl = gld(S.extra + (l));
            if (is_i) {  // bead i, reached through extra(j,:): its fresh result
                st_t = ti;
                st_p = pi;
                st_c = ci;
            } else {
                const Leaf lf = leaf_ld(L, l);
                st_t = lf.tim;
                st_p = lf.nptnr;
                st_c = leaf_ct(lf.meta);
            }
        }
        bool modified = false, pending = false;
        int rem = first ? cI + cJ : 0;
        for (int guard = 0; guard < 64 * 9; ++guard) {
            while (rem > 0 && !pending) {
                const bool opi = rem > cJ;
                const int p = opi ? i : j;
                --rem;
                if (st_p != p)
                    single_update(T, rl, ol, bwl, p, opi ? P.ri : P.rj, tf, st_t, st_p, st_c, modified, status);
                else
                    pending = true;
            }
            const unsigned long long pm = __ballot(pending);
            if (pm == 0) break;
            const int leader = __ffsll((long long)pm) - 1;
            const int lf_l = __shfl(l, leader, kW);
            const Rec rlf = shfl_rec(rl, leader);
            const double2 bwlf = make_double2(__shfl(bwl.x, leader, kW), __shfl(bwl.y, leader, kW));
            const int4 xlf = make_int4(__shfl(xl.x, leader, kW), __shfl(xl.y, leader, kW), __shfl(xl.z, leader, kW),
                                       __shfl(xl.w, leader, kW));
            double ft;
            int fp, fc;
            full_one(S, L, lf_l, rlf, bwlf, xlf, tf, T0, ft, fp, fc, status);
            if (lane == leader) {
                st_t = ft;
                st_p = fp;
                st_c = fc;
                modified = true;
                pending = false;
            }
        }
        // bead i's state lives in (ti, pi, ci) and is written with i's leaf
        const unsigned long long im = __ballot(first && is_i);
        if (im) {
            const int src = __ffsll((long long)im) - 1;
            ti = __shfl(st_t, src, kW);
            pi = __shfl(st_p, src, kW);
            ci = __shfl(st_c, src, kW);
        }
        if (is_i) modified = false;
        if (modified) {
            Leaf lf;
            lf.tim = st_t;
            lf.nptnr = st_p;
            lf.meta = make_meta(calc_bin(c, st_t, false, status), st_c);
            leaf_st(L, l, lf);
            stamp_set(l, mk_stamp(c.coll, (j >= 0 ? 3 : 4) + q));
        }
        const unsigned long long mm = __ballot(modified);
        const int pre = before_me(mm);
        if (modified && nbl + pre < kMaxBlist) L.blist()[nbl + pre] = l / kBlk;
        nbl += __popcll(mm);
        if (nbl > kMaxBlist) nbl = kMaxBlist;
    }
    PH_END(S, kPhDown, tph);
    if (lane == 0) {
        // adds in partial_events.f order: i, j, then the down set (a ghost
        // event's own entry came first)
        Leaf a;
        a.tim = ti;
        a.nptnr = pi;
        a.meta = make_meta(calc_bin(c, ti, false, status), ci);
        leaf_st(L, i, a);
        stamp_set(i, mk_stamp(c.coll, j >= 0 ? 1 : 2));
        if (j >= 0) {
            Leaf b;
            b.tim = tj;
            b.nptnr = pj;
            b.meta = make_meta(calc_bin(c, tj, false, status), cj);
            leaf_st(L, j, b);
            stamp_set(j, mk_stamp(c.coll, 2));
        }
    }
    // repuls_del_b.f once the rescheduling is done
    if (xpulse_del && lane == 0) {
        const bool iN = dyn_ident(P.ri.dyn) < dyn_ident(P.rj.dyn);
        const int Li = topo_len(P.ri.topo), Lj = topo_len(P.rj.topo);
        if (iN)
            shoulders_clear(i, Li, j, Lj);
        else
            shoulders_clear(j, Lj, i, Li);
    }
    status = wave_status(status);
    if (status && !c.status) c.status = status;
    if (!L.leaf_lds)
        wave_sync_mem();
    else
        wave_sync();
    if (lane == 0) L.batch()->nbl = nbl;
    PH_END(S, kPhLeaf, tph);
}

// partial_events.f:16-201 after an event of pair (i, j) (j < 0: ghost of i).
// One batch of predictions covers the full recomputes of i and j and of the
// down-set beads whose calendar partner is i or j (speculatively: the
// recompute happens only if their op sequence reaches it, and is then the
// same value); each owner's minimum over (time, list position) comes out of
// LDS atomics.  The remaining single-pair updates run one down bead per
// lane.  Three dependent rounds of global loads: the rows of i and j; the
// down beads, the rows of the batched beads and the candidates of i and j;
// the partners of the batched beads.  Down sets above one wavefront take
// the generic path.  extra_blk: a further calendar block to rescan (the
// ghost entry), or -1
__device__ __noinline__ void reschedule(const SysDev&, const DevTables&, const Lds&, Sc&, const Pair&, int extra_blk,
                           bool xpulse_del, int bk) {
    const Lds L = lds_regs();

    const SysDev& S = sdev();

    const DevTables& T = tabs();
    Sc& c = *L.sc();
    const Pair& P = *L.pair();
    // the wavefront's work-area views, held in scalar registers: the wave
    // fences below would make the compiler read them from LDS again
    int* const v_wm = reinterpret_cast<int*>(smem + __builtin_amdgcn_readfirstlane(L.o_wm));
    int* const v_wx = reinterpret_cast<int*>(smem + __builtin_amdgcn_readfirstlane(L.o_wx));
    int* const v_wd = reinterpret_cast<int*>(smem + __builtin_amdgcn_readfirstlane(L.o_wd));
    int* const v_wy = reinterpret_cast<int*>(smem + __builtin_amdgcn_readfirstlane(L.o_wy));
    double* const v_wt = reinterpret_cast<double*>(smem + __builtin_amdgcn_readfirstlane(L.o_wt));
    MinSlot* const v_slot = reinterpret_cast<MinSlot*>(smem + __builtin_amdgcn_readfirstlane(L.o_slot));
    SpecInfo* const v_spec = reinterpret_cast<SpecInfo*>(smem + __builtin_amdgcn_readfirstlane(L.o_spec));
    DownInfo* const v_down = reinterpret_cast<DownInfo*>(smem + __builtin_amdgcn_readfirstlane(L.o_down));
    const int maxw = __builtin_amdgcn_readfirstlane(L.maxw);

    const int lane = lane_id(), cap = S.cap;
    const int i = P.i, j = P.j;
    const double tf = c.tfalse;
    const double T0 = c.interval_max + kLt - tf;
    const int dbase = maxw - (2 * cap + 8);  // down-set region of the work list
    const bool batch = bk >= 0;
    // place of i's add among this event's calendar adds (a ghost event adds
    // its own entry first); j follows, then the down set in list order
    const int sub0 = j >= 0 ? 1 : 2;
    int status = 0, nb = 0;
    PH_BEGIN(tph);
    // ---- first loads: list rows of i and j, whole rows with their lengths
    const Rows rw = load_rows(S, i, j);
    const int nui = rw.nui, ndi = rw.ndi, nuj = rw.nuj, ndj = rw.ndj;
    const int eui = rw.eui, edi = rw.edi, euj = rw.euj, edj = rw.edj;
    const int xi0 = P.xi.x, xi1 = P.xi.y, xi2 = P.xi.z;
    const int xj0 = P.xj.x, xj1 = P.xj.y, xj2 = P.xj.z;
    const int kNoStat = 0xFF << 24;
    // ---- work list: candidates of i (owner 0) and j (owner 1) at 0..
    int w = 0;
    if (lane < nui) {
        v_wm[lane] = eui;
        v_wx[lane] = 0;
    }
    w = nui;
    if (xi0 > i) { if (lane == 0) { v_wm[w] = xi0 | kNoStat; v_wx[w] = 0; } ++w; }
    if (xi1 > i) { if (lane == 0) { v_wm[w] = xi1 | kNoStat; v_wx[w] = 0; } ++w; }
    if (xi2 > i) { if (lane == 0) { v_wm[w] = xi2 | kNoStat; v_wx[w] = 0; } ++w; }
    if (j >= 0) {
        if (lane < nuj) {
            v_wm[w + lane] = euj;
            v_wx[w + lane] = 1;
        }
        w += nuj;
        if (xj0 > j) { if (lane == 0) { v_wm[w] = xj0 | kNoStat; v_wx[w] = 1; } ++w; }
        if (xj1 > j) { if (lane == 0) { v_wm[w] = xj1 | kNoStat; v_wx[w] = 1; } ++w; }
        if (xj2 > j) { if (lane == 0) { v_wm[w] = xj2 | kNoStat; v_wx[w] = 1; } ++w; }
    }
    const int ncand = w;
    // ---- the down set at dbase.., tag 2 (op with i) / 3 (op with j), in
    //      reference order: i's down list and lower shoulder partners, then j's
    int d = 0;
    if (lane < ndi) {
        v_wm[dbase + lane] = edi & 0xFFFF;
        v_wx[dbase + lane] = 2;
    }
    d = ndi;
    if (xi0 >= 0 && xi0 < i) { if (lane == 0) { v_wm[dbase + d] = xi0; v_wx[dbase + d] = 2; } ++d; }
    if (xi1 >= 0 && xi1 < i) { if (lane == 0) { v_wm[dbase + d] = xi1; v_wx[dbase + d] = 2; } ++d; }
    if (xi2 >= 0 && xi2 < i) { if (lane == 0) { v_wm[dbase + d] = xi2; v_wx[dbase + d] = 2; } ++d; }
    if (j >= 0) {
        const int l = edj & 0xFFFF;
        const bool keep = lane < ndj && l != i;
        const unsigned long long bal = __ballot(keep);
        const int pre = before_me(bal);
        if (keep) {
            v_wm[dbase + d + pre] = l;
            v_wx[dbase + d + pre] = 3;
        }
        d += __popcll(bal);
        if (xj0 >= 0 && xj0 < j) { if (lane == 0) { v_wm[dbase + d] = xj0; v_wx[dbase + d] = 3; } ++d; }
        if (xj1 >= 0 && xj1 < j) { if (lane == 0) { v_wm[dbase + d] = xj1; v_wx[dbase + d] = 3; } ++d; }
        if (xj2 >= 0 && xj2 < j) { if (lane == 0) { v_wm[dbase + d] = xj2; v_wx[dbase + d] = 3; } ++d; }
    }
    const int nD = d;
    if (nD > kW) {
        // the generic form writes as it goes: no other event of the round
        // is committed
        if (batch && lane == 0) atomicMin(&L.batch()->cut, 1);
        wave_sync_mem();
        PH_COUNT(S, kPhNGeneric);
        reschedule_generic(S, T, L, c, P, extra_blk, xpulse_del);
        if (batch) bar_to(nb, kRoundBars);
        return;
    }
    if (lane < 2 + kMaxSpec) {
        v_slot[lane].tkey = ~0ull;
        v_slot[lane].packed = ~0u;
    }
    wave_sync();
    PH_END(S, kPhRows, tph);
    // ---- one lane per down-set entry: first occurrence of its bead, the
    //      bead's op counts, and whether its full recompute is batched
    int l = -1, cI = 0, cJ = 0;
    bool first = false;
    const int dent = lane < nD ? v_wm[dbase + lane] : -1;
    {
        // every lane compares its bead with each entry, read from lanes
        const int lv = dent;
        const int tv = lane < nD ? v_wx[dbase + lane] : 0;
        l = lv;
        first = lane < nD;
        for (int r = 0; r < nD; ++r) {
            const int lr = __builtin_amdgcn_readlane(lv, r);
            const int tr = __builtin_amdgcn_readlane(tv, r);
            if (lr == lv) {
                if (r < lane) first = false;
                if (tr == 2) ++cI;
                else ++cJ;
            }
        }
        if (!first) {
            cI = 0;
            cJ = 0;
        }
    }
    const bool is_i = first && l == i;
    Leaf lf0;
    lf0.tim = 0.0;
    lf0.nptnr = -1;
    lf0.meta = 0;
    if (first && !is_i) lf0 = leaf_ld(L, l);
    bool spec = first && !is_i && ((lf0.nptnr == i && cI > 0) || (lf0.nptnr == j && cJ > 0));
    const unsigned long long smask = __ballot(spec);
    const int myslot = spec ? before_me(smask) : -1;
    if (myslot >= kMaxSpec) spec = false;
    const int nspec = min(__popcll(smask), kMaxSpec);
    if (spec) v_spec[myslot].l = l;
    wave_sync();
    PH_END(S, kPhScan, tph);
    // ---- second loads: the down beads' own data, the rows of the batched beads
    //      and the candidates of i and j, all in flight together
    Rec rl = P.ri;
    int4 ol = make_int4(-1, -1, -1, -1), xl = make_int4(-1, -1, -1, -1);
    double2 bwl = make_double2(0.0, 0.0);
    int nul = 0;
    if (first) {
        rl = load_rec(S, P, l);
        ol = gld(S.ovr + (l));
        bwl = gld(S.bw + (l));
        xl = gld(S.extra + (l));
    }
    if (spec) nul = gl1(S.nup + (l));
    int sent[kMaxSpec];
#pragma unroll
    for (int s2 = 0; s2 < kMaxSpec; ++s2) {
        sent[s2] = 0;
        if (s2 < nspec && lane < cap) sent[s2] = gl1(S.nb_up + ((size_t)v_spec[s2].l * cap + lane));
    }
    const int cent = lane < ncand ? v_wm[lane] : 0;
    const int cm = cent & 0xFFFFFF;
    Rec crm = P.ri;
    int4 com = make_int4(-1, -1, -1, -1);
    if (lane < ncand) {
        crm = load_rec(S, P, cm);
        com = gld(S.ovr + (cm));
    }
    // the down beads' own data for their single-pair predictions
    if (first && cI + cJ > 0) {
        DownInfo& di = v_down[lane];
        di.r = rl;
        di.o = ol;
        di.bw = bwl;
    }
    // the batched beads' pair entries, after the candidates
    if (spec) {
        SpecInfo& si = v_spec[myslot];
        si.r = rl;
        si.bw = bwl;
        si.x = xl;
        si.nu = nul;
        si.nx = (xl.x > l ? 1 : 0) + (xl.y > l ? 1 : 0) + (xl.z > l ? 1 : 0);
    }
    wave_sync();
    if (lane == 0) {
        int off = ncand;
        for (int s2 = 0; s2 < nspec; ++s2) {
            SpecInfo& si = v_spec[s2];
            const int n = si.nu + si.nx;
            if (off + n <= dbase) {
                si.off = off;
                off += n;
            } else
                si.off = -1;  // no room: this bead's recompute runs on its own
        }
        v_wd[0] = off;
    }
    wave_sync();
    const int npairs = v_wd[0];
#pragma unroll
    for (int s2 = 0; s2 < kMaxSpec; ++s2) {
        if (s2 < nspec) {
            const int off = v_spec[s2].off, nu = v_spec[s2].nu;
            if (off >= 0) {
                if (lane < nu) {
                    v_wm[off + lane] = sent[s2];
                    v_wx[off + lane] = 2 + s2;
                }
                if (lane == 0) {
                    const int4 x = v_spec[s2].x;
                    const int ls = v_spec[s2].l;
                    int k = off + nu;
                    if (x.x > ls) { v_wm[k] = x.x | kNoStat; v_wx[k] = 2 + s2; ++k; }
                    if (x.y > ls) { v_wm[k] = x.y | kNoStat; v_wx[k] = 2 + s2; ++k; }
                    if (x.z > ls) { v_wm[k] = x.z | kNoStat; v_wx[k] = 2 + s2; ++k; }
                }
            }
        }
    }
    int sp = -1;  // the wavefront's bead of the shoulder set, marked in a round
    bool sp_w = false;
    // the down bead's updates may take a full recompute (a pending op)
    const bool mfull = first && !is_i && ((lf0.nptnr == i && cI > 0) || (lf0.nptnr == j && cJ > 0) || cI >= 2 || cJ >= 2);
    // single-pair predictions of the down beads (placed after the pairs)
    const bool wantI = first && cI > 0, wantJ = first && cJ > 0;
    const unsigned long long mI = __ballot(wantI), mJ = __ballot(wantJ);
    const int nI = __popcll(mI), nsing = nI + __popcll(mJ);
    const bool sing_fit = npairs + nsing <= maxw;
    // ---- the round's footprint marks (run_event): this event leads the
    //      round, so it checks nothing and is always committed
    if (batch) {
        PH_RESET(tph);
        Batch& B = *L.batch();
        const unsigned sbit = 1u, lbit = 1u << 8, fbit = 1u << 16;
        sp = shoulder_bead(S, P, lane);
        if (lane == 0) B.wdone[0] = 0;
        if (dent >= 0) mark_or(L, dent, lbit | (mfull ? fbit : 0u));
        if (lane == 0) mark_or(L, i, sbit | lbit | fbit);
        if (lane == 1 && j >= 0) mark_or(L, j, sbit | lbit | fbit);
        sp_w = (P.flags & kPairWroteSp) != 0;
        if (sp_w && sp >= 0) mark_or(L, sp, sbit);
        bar_to(nb, 1);
        PH_END(S, kPhBMark, tph);
    }
    // ---- the single-pair predictions (l, i) and (l, j) of each down bead,
    //      after the pair entries: each is the same for every op of l with
    //      that bead, so one per (bead, partner) serves the whole op sequence
    int sqI = -1, sqJ = -1;
    if (sing_fit) {
        if (wantI) {
            sqI = npairs + before_me(mI);
            v_wm[sqI] = lane;
        }
        if (wantJ) {
            sqJ = npairs + nI + before_me(mJ);
            v_wm[sqJ] = lane | 0x100;
        }
    }
    const int ntot = sing_fit ? npairs + nsing : npairs;
    wave_sync();
    PH_END(S, kPhLoads, tph);
    // ---- the prediction batch: the candidates of i and j, the batched
    //      beads' partners, then the single-pair predictions
    PH_ADDN(S, kPhNPred, ntot);
    PH_ADDN(S, kPhNPredPass, (ntot + kW - 1) / kW);
    for (int base = 0; base < ntot; base += kW) {
        const int q = base + lane;
        if (q < ntot) {
            const bool single = q >= npairs;
            const int ent = base == 0 && q < ncand ? cent : v_wm[q];
            const int owner = single ? 0 : v_wx[q];
            int m, stat, xc;
            Rec ra, rb;
            int4 oc;
            double2 bwa;
            if (single) {
                // eventredo_down.f: ev_code(l, p) with l's record first
                const DownInfo& di = v_down[ent & 0xFF];
                const bool oj = (ent & 0x100) != 0;
                m = oj ? j : i;
                ra = di.r;
                rb = oj ? P.rj : P.ri;
                oc = di.o;
                bwa = di.bw;
                xc = m;
                stat = static_t(T, ra.topo, rb.topo);
            } else {
                m = ent & 0xFFFFFF;
                stat = (ent >> 24) & 0xFF;
                if (owner == 0) {
                    xc = i;
                    ra = P.ri;
                    bwa = P.bwi;
                } else if (owner == 1) {
                    xc = j;
                    ra = P.rj;
                    bwa = P.bwj;
                } else {
                    const SpecInfo& si = v_spec[owner - 2];
                    xc = si.l;
                    ra = si.r;
                    bwa = si.bw;
                }
                if (base == 0 && q < ncand) {
                    rb = crm;
                    oc = com;
                } else {
                    rb = load_rec(S, P, m);
                    oc = gld(S.ovr + (m));
                }
                if (stat == 0xFF) stat = static_t(T, rb.topo, ra.topo);
            }
            const int code = dyn_code(oc, xc, stat);  // ev_code(m, x), or ev_code(l, p) for a single
            double tij = 1000000000.0;
            int ty = 0;
            predict(T, code, ra, rb, dyn_bptnr(ra.dyn) == m, bwa, tf, tij, ty);
            v_wt[q] = tij;
            if (single) {
                v_wy[q] = ty;  // checked where the op sequence uses it
            } else {
                if (ty == -99) status = kErrBadCode;
                if (tij < 0.0 && fabs(tij) > 1.0e-10) status = kErrNegativeTime;
                v_wy[q] = (((ty + 1) & 31) << 16) | (m & 0xFFFF);  // fields masked: position stays in bits 21..31
                atomicMin(&v_slot[owner].tkey, t_order(tij));
            }
        }
    }
    wave_sync();
    for (int base = 0; base < npairs; base += kW) {
        const int q = base + lane;
        if (q < npairs) {
            const int owner = v_wx[q];
            if (t_order(v_wt[q]) == v_slot[owner].tkey) atomicMin(&v_slot[owner].packed, ((unsigned)q << 21) | (unsigned)v_wy[q]);
        }
    }
    wave_sync();
    PH_END(S, kPhPred, tph);
    // owner results (full recompute rule: an event only below T0)
    double ti = T0 + tf, tj = T0 + tf;
    int pi = -1, ci = -1, pj = -1, cj = -1;
    {
        const unsigned a = v_slot[0].packed;
        if (a != ~0u) {
            const double bt = v_wt[a >> 21];
            if (bt < T0) {
                ti = bt + tf;
                pi = (int)(a & 0xFFFF);
                ci = (int)((a >> 16) & 31) - 1;
            }
        }
        const unsigned b = v_slot[1].packed;
        if (j >= 0 && b != ~0u) {
            const double bt = v_wt[b >> 21];
            if (bt < T0) {
                tj = bt + tf;
                pj = (int)(b & 0xFFFF);
                cj = (int)((b >> 16) & 31) - 1;
            }
        }
    }
    const double ti0 = ti;
    const int pi0 = pi, ci0 = ci;
    double st_t = lf0.tim;
    int st_p = lf0.nptnr, st_c = leaf_ct(lf0.meta);
    bool modified = false, pending = false;
    int rem = first ? cI + cJ : 0;
    if (is_i) {
        st_t = ti;
        st_p = pi;
        st_c = ci;
    }
    // ---- the rest of each down bead's ops; full recomputes from the batch,
    //      others (not foreseen) cooperatively one at a time
    const bool have_full = spec && v_spec[myslot].off >= 0;
    PH_LANE_DECL(ph_single);
    for (int guard = 0; guard < 64 * 9; ++guard) {
        while (first && (rem > 0 || pending)) {
            if (pending) {
                if (is_i) {
                    st_t = ti0;
                    st_p = pi0;
                    st_c = ci0;
                } else if (have_full) {
                    const unsigned a = v_slot[2 + myslot].packed;
                    st_t = T0 + tf;
                    st_p = -1;
                    st_c = -1;
                    if (a != ~0u) {
                        const double bt = v_wt[a >> 21];
                        if (bt < T0) {
                            st_t = bt + tf;
                            st_p = (int)(a & 0xFFFF);
                            st_c = (int)((a >> 16) & 31) - 1;
                        }
                    }
                } else
                    break;
                modified = true;
                pending = false;
            } else {
                const bool opi = rem > cJ;
                const int p = opi ? i : j;
                const int sq = opi ? sqI : sqJ;
                --rem;
                if (st_p == p)
                    pending = true;
                else if (sq >= 0) {
                    // eventredo_down.f from the batch's prediction
                    double tij = v_wt[sq];
                    const int ty = v_wy[sq];
                    if (ty == -99) status = kErrBadCode;
                    if (tij < 0.0 && fabs(tij) > 1.0e-10) status = kErrNegativeTime;
                    tij = tij + tf;
                    if (tij < st_t) {
                        st_t = tij;
                        st_p = p;
                        st_c = ty;
                        modified = true;
                    }
                } else {
                    single_update(T, rl, ol, bwl, p, opi ? P.ri : P.rj, tf, st_t, st_p, st_c, modified, status);
                    PH_LANE_INC(ph_single);
                }
            }
        }
        const unsigned long long pm = __ballot(pending);
        if (pm == 0) break;
        PH_COUNT(S, kPhNFull);
        const int leader = __ffsll((long long)pm) - 1;
        const int lf_l = __shfl(l, leader, kW);
        const Rec rlf = shfl_rec(rl, leader);
        const double2 bwlf = make_double2(__shfl(bwl.x, leader, kW), __shfl(bwl.y, leader, kW));
        const int4 xlf = make_int4(__shfl(xl.x, leader, kW), __shfl(xl.y, leader, kW), __shfl(xl.z, leader, kW),
                                   __shfl(xl.w, leader, kW));
        double ft;
        int fp, fc;
        full_one(S, L, lf_l, rlf, bwlf, xlf, tf, T0, ft, fp, fc, status);
        if (lane == leader) {
            st_t = ft;
            st_p = fp;
            st_c = fc;
            modified = true;
            pending = false;
        }
    }
    PH_LANE_ADD(S, kPhNSingle, ph_single);
    // bead i's state lives in (ti, pi, ci) and is written with i's leaf
    const unsigned long long im = __ballot(is_i);
    if (im) {
        const int src = __ffsll((long long)im) - 1;
        ti = __shfl(st_t, src, kW);
        pi = __shfl(st_p, src, kW);
        ci = __shfl(st_c, src, kW);
    }
    const bool wr = modified && !is_i;
    Leaf lf, la, lb;
    if (wr) {
        lf.tim = st_t;
        lf.nptnr = st_p;
        lf.meta = make_meta(calc_bin(c, st_t, false, status), st_c);
    }
    if (lane == 0) {
        la.tim = ti;
        la.nptnr = pi;
        la.meta = make_meta(calc_bin(c, ti, false, status), ci);
        if (j >= 0) {
            lb.tim = tj;
            lb.nptnr = pj;
            lb.meta = make_meta(calc_bin(c, tj, false, status), cj);
        }
    }
    status = wave_status(status);
    if (status && !c.status) c.status = status;
    if (batch) {
        // report the least new calendar key and the status, then commit
        // only within the round's accepted prefix
        Batch& B = *L.batch();
        PH_END(S, kPhDown, tph);
        Key kn = wr ? leaf_key(lf, l) : empty_key();
        unsigned long long ks = wr ? mk_stamp(c.coll, sub0 + 2 + lane) : 0ull;
        if (lane == 0) {
            const Key ka = leaf_key(la, i);
            const unsigned long long sa = mk_stamp(c.coll, sub0);
            if (key_less_st(ka, sa, kn, ks)) {
                kn = ka;
                ks = sa;
            }
            if (j >= 0) {
                const Key kb = leaf_key(lb, j);
                const unsigned long long sb = mk_stamp(c.coll, sub0 + 1);
                if (key_less_st(kb, sb, kn, ks)) {
                    kn = kb;
                    ks = sb;
                }
            } else {
                // a ghost event leading the round: its next ghost time
                const Key kg = leaf_key(leaf_ld(L, S.N), S.N);
                const unsigned long long sg = mk_stamp(c.coll, 1);  // re-added by this ghost event
                if (key_less_st(kg, sg, kn, ks)) {
                    kn = kg;
                    ks = sg;
                }
            }
        }
        unsigned long long kns = 0;
        kn = key_min_wave_st(kn, ks, kns);
        if (lane == 0) {
            B.knew[0] = kn;
            B.knew_st[0] = kns;
            B.st[0] = c.status;
        }
        bar_to(nb, kRoundBars);
        PH_END(S, kPhBKeys, tph);
        // every wavefront has checked: clear this one's marks
        round_clear_marks(L, S, dent, i, j, sp_w ? sp : -1);
    }
    if (wr) {
        leaf_st(L, l, lf);
        stamp_set(l, mk_stamp(c.coll, sub0 + 2 + lane));
    }
    if (lane == 0) {
        L.blist()[0] = i / kBlk;
        L.blist()[1] = j >= 0 ? j / kBlk : i / kBlk;
        L.blist()[2] = extra_blk >= 0 ? extra_blk : i / kBlk;
    }
    const unsigned long long mm = __ballot(wr);
    const int pre = before_me(mm);
    if (wr) L.blist()[3 + pre] = l / kBlk;
    const int nbl = 3 + __popcll(mm);
    PH_END(S, kPhDown, tph);
    if (lane == 0) {
        leaf_st(L, i, la);
        stamp_set(i, mk_stamp(c.coll, sub0));
        if (j >= 0) {
            leaf_st(L, j, lb);
            stamp_set(j, mk_stamp(c.coll, sub0 + 1));
        }
    }
    // repuls_del_b.f once the rescheduling is done
    if (xpulse_del && lane == 0) {
        const bool iN = dyn_ident(P.ri.dyn) < dyn_ident(P.rj.dyn);
        const int Li = topo_len(P.ri.topo), Lj = topo_len(P.rj.topo);
        if (iN)
            shoulders_clear(i, Li, j, Lj);
        else
            shoulders_clear(j, Lj, i, Li);
    }
    if (batch) {
        // the round's block rescans run after every committed event's
        // writes; a later event that replays on these entries waits for
        // the flag
        wave_sync_mem();
        if (lane == 0) {
            L.batch()->nbl = nbl;
            __hip_atomic_store(&L.batch()->wdone[0], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        return;
    }
    if (!L.leaf_lds || xpulse_del) {
        wave_sync_mem();
    } else
        wave_sync();
    if (lane == 0) L.batch()->nbl = nbl;
    PH_END(S, kPhLeaf, tph);
}

// ------------------------------------------------------------------------
// event dynamics: eventdyn.f, bumped.f, repuls_*.f (uniform over lanes)
// ------------------------------------------------------------------------
// Outcome of eventdyn.f for event type ct (in: predicted or resolved by the
// caller, out: resolved): the impulse ratio along the pair vector, and the
// nudge bumped.f's callers give the pair off the discontinuity, bd along the
// pair vector (sgn +1: apart, -1: together, 0: none).  g: the pair's
// geometry; a, c: identities; bwi: bead i's own bond window.
__device__ __forceinline__ void impulse(const DevTables& T, const Geo& g, double bmi, double bmj, int a, int c, double2 bwi,
                                        bool bonded_ij, int evcode, int& ct, double& ratio, double& bd, int& sgn,
                                        int& status) {
    const double rmass = 2 * bmi * bmj / (bmi + bmj);
    const double b = g.b;
    ratio = 0.0;
    sgn = 0;
    bd = 0.0;
    if (ct <= 3) {
        double sq;
        if (ct == 1) {
            const double pe = T.ev_param[1][evcode], ssq = T.sigma_sq[a][c];
            if (evcode == 15 && !bonded_ij)
                sq = ssq;
            else {
                sq = ssq * (pe * pe);
                if (evcode >= 22 && evcode <= 26) {
                    const double q = T.sqz610[evcode - 21][a > c ? a : c];
                    sq = sq * (q * q);
                }
            }
        } else {
            double blmin, blmax;
            bond_window(T, evcode, bwi, blmin, blmax);
            sq = ct == 2 ? blmin * blmin : blmax * blmax;
        }
        ratio = rmass * b / sq;
        if (ct < 1) status = kErrDyn;
        return;
    }
    const bool shl = ct == 5 || ct == 6 || ct == 13;
    if (!shl && ct != 4 && ct != 8 && ct != 9) {
        status = kErrDyn;
        return;
    }
    const double wellsq = shl ? T.shlddia_sq[a][c] : T.welldia_sq[a][c];
    const double epsave = shl ? -T.epsilon1 : T.ep_sqrt[a][c];
    const double del_pe = 4.0 * wellsq * epsave / rmass;
    bd = kSm * sqrt(wellsq);
    bool bounce = false;
    double root = 0.0;
    switch (ct) {
        case 4:
            bounce = !(b * b + del_pe > 0.0);
            root = sqrt(del_pe + b * b);
            ct = bounce ? 22 : 20;
            sgn = bounce ? 1 : -1;
            break;
        case 8:
            bounce = !(b * b > del_pe);
            root = -sqrt(-del_pe + b * b);
            ct = bounce ? 22 : 21;
            sgn = bounce ? -1 : 1;
            break;
        case 5:
            root = -sqrt(-del_pe + b * b);
            ct = 24;
            sgn = 1;
            break;
        case 6:
            bounce = !(b * b > -del_pe);
            root = sqrt(del_pe + b * b);
            ct = bounce ? 26 : 25;
            sgn = bounce ? 1 : -1;
            break;
        default:  // 9, 13
            bounce = true;
            ct = shl ? 27 : 23;
            sgn = 1;
            break;
    }
    ratio = bounce ? rmass * b / wellsq : rmass * (root + b) / (2.0 * wellsq);
}

__device__ inline double dist_rec(const Rec& a, const Rec& b, double tf) {
    Geo g;
    geo(a, b, tf, g);
    return sqrt(g.rx * g.rx + g.ry * g.ry + g.rz * g.rz);
}
// An index taken from an event's H-bond partner or identities, brought into
// the system.  A speculative event may read those while the round's first
// event writes them: identities of before and after an H-bond formed or broke
// order N and C bead the wrong way round, and a cleared shoulder code points
// at a partner of -1; shoulder_idx then gives beads up to a chain's length
// before the first.  Such an event shares a bead with the first one and is
// discarded at the footprint check, whatever it reads; it must only read
// inside the system.
__device__ inline int in_system(int m, int N) { return (unsigned)m < (unsigned)N ? m : 0; }
// a bead's record as the event sees it: the colliding pair's own from the
// wavefront's Pair in LDS, any other from memory
__device__ inline Rec pair_rec(int m) {
    const Pair& P = *ldsv().pair();
    return load_rec(sdev(), P, in_system(m, sdev().N));
}
// repuls_check.f:16-81 (n = the N bead, cb = the C bead), the colliding pair
// read from LDS; these run in few events and stay out of line, so that the
// event's own registers and code stay small
__device__ __noinline__ bool shoulders_far(int n, int cb, double tf) {
    const DevTables& T = tabs();
    const Rec rn = pair_rec(n), rc = pair_rec(cb);
    int ncim1, ncai, ncaj, nnjp1;
    shoulder_idx(n, topo_len(rn.topo), cb, topo_len(rc.topo), ncim1, ncai, ncaj, nnjp1);
    const double d1 = dist_rec(rn, pair_rec(ncaj), tf), d2 = dist_rec(rn, pair_rec(nnjp1), tf);
    const double d3 = dist_rec(rc, pair_rec(ncai), tf), d4 = dist_rec(rc, pair_rec(ncim1), tf);
    return d1 > T.shder[1] && d2 > T.shder[2] && d3 > T.shder[3] && d4 > T.shder[4];
}
// repuls_check_3.f:16-102: the three shoulders other than k
__device__ __noinline__ bool shoulders_far_3(int n, int cb, int k, double tf) {
    const DevTables& T = tabs();
    const Rec rn = pair_rec(n), rc = pair_rec(cb);
    int ncim1, ncai, ncaj, nnjp1;
    shoulder_idx(n, topo_len(rn.topo), cb, topo_len(rc.topo), ncim1, ncai, ncaj, nnjp1);
    int m = 0;
    if (ncaj != k && dist_rec(rn, pair_rec(ncaj), tf) > T.shder[1]) ++m;
    if (nnjp1 != k && dist_rec(rn, pair_rec(nnjp1), tf) > T.shder[2]) ++m;
    if (ncai != k && dist_rec(rc, pair_rec(ncai), tf) > T.shder[3]) ++m;
    if (ncim1 != k && dist_rec(rc, pair_rec(ncim1), tf) > T.shder[4]) ++m;
    return m == 3;
}
// squared distance of two beads, the colliding pair read from LDS
__device__ __noinline__ double pair_r2(int a, int b, double tf) {
    Geo g;
    geo(pair_rec(a), pair_rec(b), tf, g);
    return g.r2;
}
// repuls_del_b.f (single lane; n = N bead, cb = C bead)
__device__ __noinline__ void shoulders_clear(int n, int Ln, int cb, int Lc) {
    const SysDev& S = sdev();
    int ncim1, ncai, ncaj, nnjp1;
    shoulder_idx(n, Ln, cb, Lc, ncim1, ncai, ncaj, nnjp1);
    int4 en = gld(S.extra + (n)), ec = gld(S.extra + (cb));
    en.x = -1;
    en.y = -1;
    en.w = -1;
    ec.x = -1;
    ec.y = -1;
    ec.w = -1;
    gst(S.extra + (n), en);
    gst(S.extra + (cb), ec);
    gs1(&S.extra[ncaj].z, -1);
    gs1(&S.extra[nnjp1].z, -1);
    gs1(&S.extra[ncai].z, -1);
    gs1(&S.extra[ncim1].z, -1);
}
// repuls_add.f:14-47 / repuls_del_a.f:14-37 (single lane; n = N bead, cb = C bead)
__device__ __noinline__ int repuls_add(int n, int Ln, int cb, int Lc) {
    const SysDev& S = sdev();
    int status = 0;

    int ncim1, ncai, ncaj, nnjp1;
    shoulder_idx(n, Ln, cb, Lc, ncim1, ncai, ncaj, nnjp1);
    set_code(S, ncaj, n, 50, status);
    set_code(S, n, ncaj, 40, status);
    set_code(S, n, nnjp1, 40, status);
    set_code(S, nnjp1, n, 50, status);
    set_code(S, ncai, cb, 50, status);
    set_code(S, cb, ncai, 40, status);
    set_code(S, cb, ncim1, 40, status);
    set_code(S, ncim1, cb, 50, status);
    int4 en = gld(S.extra + (n)), ec = gld(S.extra + (cb));
    en.x = ncaj;
    en.y = nnjp1;
    en.w = cb;
    ec.x = ncai;
    ec.y = ncim1;
    ec.w = n;
    gst(S.extra + (n), en);
    gst(S.extra + (cb), ec);
    gs1(&S.extra[ncaj].z, n);
    gs1(&S.extra[nnjp1].z, n);
    gs1(&S.extra[ncai].z, cb);
    gs1(&S.extra[ncim1].z, cb);
    return status;
}
__device__ __noinline__ int repuls_del_a(int n, int Ln, int cb, int Lc) {
    const SysDev& S = sdev();
    int status = 0;

    int ncim1, ncai, ncaj, nnjp1;
    shoulder_idx(n, Ln, cb, Lc, ncim1, ncai, ncaj, nnjp1);
    set_code(S, ncaj, n, 1, status);
    set_code(S, n, ncaj, 1, status);
    set_code(S, n, nnjp1, 1, status);
    set_code(S, nnjp1, n, 1, status);
    set_code(S, ncai, cb, 1, status);
    set_code(S, cb, ncai, 1, status);
    set_code(S, ncim1, cb, 1, status);
    set_code(S, cb, ncim1, 1, status);
    return status;
}
__device__ inline bool terminal_t(int t) {
    const int k = topo_kind(t), r = topo_res(t), L = topo_len(t);
    return (k == 1 && r == 1) || (k == 2 && r == L);
}

// The wavefront's work area while an event is rescheduled in one pass.
struct __attribute__((aligned(16))) BaseRec {
    Rec r;
    double2 bw;
    int idx, pad[3];
};
constexpr int kOwners = 2 + kMaxSpec;
struct OnePass {
    BaseRec base[kOwners];  // 0: bead i, 1: bead j, then the beads recomputed in full
    double wt[kW];
    unsigned long long tkey[kOwners];  // least time
    int win[kOwners];                  // its lane, the first of equal ones
    int wy[kW];
    int lst[kW];
};
static_assert(sizeof(OnePass) >= sizeof(int) * kListMax, "the calendar wavefront's block list lies over its work area");
static_assert(sizeof(OnePass) >= sizeof(double) * kW, "so do the selection's proxies over wavefront 0's");
// result lanes of beads i and j: entries take the lanes below
constexpr int kLaneI = kW - 2, kLaneJ = kW - 1;

// A lane's part of one gather that fetches everything an event needs of its
// two beads, 8 bytes per lane: lanes 0-7 and 8-15 the records of i and j,
// 16-17 the overrides of i, 18-21 the shoulder partners, 22-25 the bond
// windows, 26-29 the list lengths (up and down of i, then of j).  As
// wave-uniform 16-byte loads the same data took thirteen instructions of
// 1 KB each through the CU's 64 B/cycle path.
struct Gather {
    const GLB char* base;
    int sh;  // log2 of the buffer's element size
};
constexpr unsigned kGatherJ = 0x3330FF00u;  // lanes of bead j
constexpr int kGatherLanes = 30;
__device__ inline Gather load_gather(const SysDev& S) {
    const int lane = lane_id();
    // (addresses as numbers: a select between pointer fields keeps its
    // struct in memory)
    const unsigned long long rec = (unsigned long long)S.rec, ovr = (unsigned long long)S.ovr,
                             ext = (unsigned long long)S.extra, bw = (unsigned long long)S.bw,
                             nup = (unsigned long long)S.nup, ndn = (unsigned long long)S.ndn;
    unsigned long long p = rec + (unsigned)(lane & 7) * 8u;
    Gather G;
    G.sh = 6;
    if (lane >= 16) {
        p = (lane < 18 ? ovr : (lane < 22 ? ext : bw)) + (unsigned)(lane & 1) * 8u;
        G.sh = 4;
    }
    if (lane >= 26) {
        p = (lane & 1) == 0 ? nup : ndn;
        G.sh = 2;
    }
    G.base = (const GLB char*)p;
    return G;
}
// lane l takes lane l + 3 of its row of 16
__device__ inline double up3(double v) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), 0x103, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), 0x103, 0xf, 0xf, true));
}

// The draws of an Andersen ghost collision (main.F90:1000-1041) from counter
// rc on: bead, two accepted polar pairs and the next ghost time's uniform.
struct GhostDraw {
    int i, guard;
    double v1, v2, r, w1, wr, tg;
    unsigned long long rc;
};
// one draw after the other, for draws that a single sweep of 64 does not hold
__device__ __noinline__ GhostDraw ghost_draw_serial(unsigned long long seed, unsigned long long rc, int N) {
    GhostDraw d;
    d.guard = 0;
    do {
        d.i = (int)(rng_u01(seed, 0, rc++) * N);
    } while (d.i == N && ++d.guard < 1000);
    do {
        d.v1 = 2.0 * rng_u01(seed, 0, rc++) - 1.0;
        d.v2 = 2.0 * rng_u01(seed, 0, rc++) - 1.0;
        d.r = d.v1 * d.v1 + d.v2 * d.v2;
    } while ((d.r == 0.0 || d.r >= 1.0) && ++d.guard < 1000);
    do {
        d.w1 = 2.0 * rng_u01(seed, 0, rc++) - 1.0;
        const double w2 = 2.0 * rng_u01(seed, 0, rc++) - 1.0;
        d.wr = d.w1 * d.w1 + w2 * w2;
    } while ((d.wr == 0.0 || d.wr >= 1.0) && ++d.guard < 2000);
    do {
        d.tg = rng_u01(seed, 0, rc++);
    } while ((d.tg < 1.e-18 || d.tg == 1.0) && ++d.guard < 3000);
    d.rc = rc;
    return d;
}
// the same draws, lane l holding the uniform of counter rc + l
__device__ inline GhostDraw ghost_draw(unsigned long long seed, unsigned long long rc, int N) {
    const int lane = lane_id();
    const double u = rng_u01(seed, 0, rc + (unsigned long long)lane);
    GhostDraw d;
    d.guard = 0;
    d.i = uni((int)(u * N));
    // polar pairs start at the odd lanes
    const double v1 = 2.0 * u - 1.0, v2 = 2.0 * __shfl_down(u, 1, kW) - 1.0;
    const double r = v1 * v1 + v2 * v2;
    const unsigned long long m = __ballot((lane & 1) && lane < kW - 2 && !(r == 0.0 || r >= 1.0));
    const unsigned long long m2 = m & (m - 1);
    if (d.i < N && m2 != 0) {
        const int p1 = __ffsll((long long)m) - 1, p2 = __ffsll((long long)m2) - 1;
        d.v1 = readlane_d(v1, p1);
        d.v2 = readlane_d(v2, p1);
        d.r = readlane_d(r, p1);
        d.w1 = readlane_d(v1, p2);
        d.wr = readlane_d(r, p2);
        d.tg = readlane_d(u, p2 + 2);
        d.rc = rc + (unsigned long long)(p2 + 3);
        if (!(d.tg < 1.e-18 || d.tg == 1.0)) return d;
    }
    return ghost_draw_serial(seed, rc, N);
}

// One event of a round on one wavefront: a bead-pair event (outcome
// resolution main.F90:1487-1634, dynamics, H-bond and shoulder bookkeeping
// main.F90:641-921) or an Andersen ghost collision (main.F90:997-1049),
// then partial_events.f:16-201 for it.
// e: the calendar entry; jp, ct: its partner and type; tf, nbin, coll: the
// false time, bin and number of the event; bk: its place in the round.
// Returns the round's accepted events if this one is committed, else 0.
// K: the round's entries; a single one needs no footprint marks and no
// acceptance.  The new calendar entries below the pool's edge go to the
// wavefront's share of Batch::fresh and the rewritten blocks to
// Batch::dirty[par].
//
// The pair's records stay spread over lanes 0 to 15 as the gather brings
// them (one component per lane): the impulse, the nudge and the ghost's
// velocity draw update them with one division for all components, and they
// go to LDS and back to memory as they lie.  What decides control flow or is
// shared by all lanes is read from the lanes into scalar registers.
//
// The rescheduling takes one pass of 64 lanes: a lane per candidate of i
// and j (tags 0 and 1), per down-set entry (tags 2 and 3: its op partner i
// or j), and per candidate of a down bead that may be recomputed in full
// (tag 4 + s).  Each lane gathers its own entry's bead and predicts it
// against its base bead (i, j or the recomputed bead, staged in LDS), so
// every prediction costs one gather and the event three dependent rounds of
// loads: the pair and its rows; the entries' beads and the rows of the
// beads recomputed; those rows' beads.  An event of more than 62 entries (two lanes
// take the results of i and j) or of more than kMaxSpec full recomputes
// runs the multi-pass form, which holds any number.  What bounds an event
// is the length of its dependent chain, so the code keeps wave-uniform
// values in scalar registers and replaces divergent branches by selects.
// Measured at four wavefronts, 5000 entries of 128 / 512 beads: 45.3 / 37.1 ms
// with the multi-pass form for every event, 29.7 / 24.8 with one pass; 27.9 /
// 22.0 with the pair's records as wave-uniform structs, 21.8 / 17.5 spread
// over lanes; 20.4 / 15.5 with each owner's result taken from ballots, 19.6 /
// 14.8 with the LDS minimum of lanes.  Listing and loading the entries before
// the outcome, to cover the loads' latency, is 2 to 6 % slower: it takes 145
// more instructions per entry.
__device__ __forceinline__ int run_event(const Hot& H, const Gather& G, int e, int jp, int ct, double tf, int nbin,
                                         long long coll, int bk, int K, int par, int fsh) {
    const int lane = lane_id();
    const DevTables& T = tabs();
    Sc& mc = master();
    Batch& B = round_rec();
    OnePass& W = *reinterpret_cast<OnePass*>(smem + H.o_w);
    const double interval_max = mc.interval_max, tbin_off = mc.tbin_off, sortsize = mc.sortsize;
    const bool solo = K == 1, batch = !solo;
    int flags = 0, st0 = 0, nb = 0, extra_blk = -1;
    bool xdel = false;
    const int cap = H.cap, sl = min(lane, cap - 1);
    const bool jside = (lane & 8) != 0;        // lanes 8 to 15: bead j
    const int comp = lane & 7;                 // component of a record's lane
    const bool ispos = lane < 16 && comp < 3, isvel = lane < 16 && comp >= 3 && comp < 6;
    PH_BEGIN(tph);
    GhostDraw gd;
    const bool ghost = e >= H.N;
    int bead = e;
    if (ghost) {
        gd = ghost_draw(sdev().seed, mc.rc0, H.N);
        bead = uni(gd.i);
    }
    // (selects below take plain values: one between captured variables or
    // fields would be made on their addresses and keep them in memory)
    const int i = bead, j = ghost ? -1 : jp;
    const int lane_bead = jside ? j : i;
    // ---- the pair's data and its list rows
    const int jx = ghost ? i : j;
    double val = 0.0;
    if (lane < kGatherLanes)
        val = *(const GLB double*)(G.base + ((unsigned)(((kGatherJ >> (lane & 31)) & 1u) ? jx : i) << G.sh));
    const int eui = ld_at(H.nb_up, i * cap + sl), edi = ld_at(H.nb_dn, i * cap + sl);
    const int euj = ld_at(H.nb_up, jx * cap + sl), edj = ld_at(H.nb_dn, jx * cap + sl);
    auto lane_lo = [&](int l) __attribute__((always_inline)) { return __builtin_amdgcn_readlane(__double2loint(val), l); };
    auto lane_hi = [&](int l) __attribute__((always_inline)) { return __builtin_amdgcn_readlane(__double2hiint(val), l); };
    auto lane_int4 = [&](int l) __attribute__((always_inline)) { return make_int4(lane_lo(l), lane_hi(l), lane_lo(l + 1), lane_hi(l + 1)); };
    const int topoi = lane_lo(7), topoj = lane_lo(15);
    int dyni = lane_hi(7), dynj = lane_hi(15);
    int4 xi = lane_int4(18), xj = lane_int4(20);
    const int nui = lane_lo(26), ndi = lane_lo(27);
    const int nuj = ghost ? 0 : lane_lo(28), ndj = ghost ? 0 : lane_lo(29);
    const double bmi = readlane_d(val, 6);
    auto store_pair = [&]() __attribute__((always_inline)) {  // the records of i and j to memory
        if (lane < 16 && !(ghost && jside))
            *(GLB double*)(G.base + ((unsigned)lane_bead << 6)) = val;
    };
    auto stage_pair = [&]() __attribute__((always_inline)) {  // ... to the wavefront's Pair in LDS
        Pair& P = *ldsv().pair();
        if (lane < 16) reinterpret_cast<double*>(jside ? &P.rj : &P.ri)[comp] = val;
        if (lane == 0) {
            P.i = i;
            P.j = j;
            P.xi = xi;
            P.xj = xj;
        }
        wave_sync();
    };
    if (!ghost) {
        const int evcode = dyn_code(lane_int4(16), j, uni(static_t(T, topoi, topoj)));  // ev_code(i, j)
        const bool ok = !terminal_t(topoi) && !terminal_t(topoj);
        const int idi = dyn_ident(dyni), idj = dyn_ident(dynj);
        const int Li = topo_len(topoi), Lj = topo_len(topoj);
        // the pair vectors: lane k < 6 of i minus lane k of j
        const double df = val - __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(val), 0x128, 0xf, 0xf, true),
                                                 __builtin_amdgcn_mov_dpp(__double2loint(val), 0x128, 0xf, 0xf, true));
        Geo g;
        {
            const double vx = readlane_d(df, 3), vy = readlane_d(df, 4), vz = readlane_d(df, 5);
            g.rx = min_image(readlane_d(df, 0) + vx * tf);
            g.ry = min_image(readlane_d(df, 1) + vy * tf);
            g.rz = min_image(readlane_d(df, 2) + vz * tf);
            g.b = g.rx * vx + g.ry * vy + g.rz * vz;
            g.r2 = 0.0;
            g.v2 = 0.0;
        }
        bool fence = false;
        auto dyn_of = [&](int m) __attribute__((always_inline)) { return m == i ? dyni : (m == j ? dynj : uni(gl1(&H.rec[in_system(m, H.N)].dyn))); };
        if (ct == 7) {
            flags |= kPairReadsSp;
            if (xi.w < 0 && xj.w < 0) {
                if (ok) {
                    stage_pair();
                    ct = uni((idi < idj ? shoulders_far(i, j, tf) : shoulders_far(j, i, tf)) ? 4 : 14);
                } else {
                    // a random draw: its counter value is known only in order
                    if (bk >= 1) {
                        spec_abort_at(bk, nb);
                        return 0;
                    }
                    const unsigned long long rc = mc.rc1;
                    ct = uni(rng_u01(sdev().seed, 1, rc) <= 0.2 ? 4 : 9);
                    if (lane == 0) mc.rc1 = rc + 1;
                }
            } else
                ct = 9;
        } else if (ct == 10) {
            flags |= kPairReadsSp;
            const bool own = evcode < 45;
            const int hbp = own ? xi.w : xj.w, idh = dyn_ident(dyn_of(hbp));
            stage_pair();
            bool far;
            if (own)
                far = idi < idh ? shoulders_far_3(i, hbp, j, tf) : shoulders_far_3(hbp, i, j, tf);
            else
                far = idj < idh ? shoulders_far_3(j, hbp, i, tf) : shoulders_far_3(hbp, j, i, tf);
            ct = uni(far ? 5 : 15);
        } else if (ct == 12) {
            flags |= kPairReadsSp;
            const bool own = evcode < 45;
            const int hbp = own ? xi.w : xj.w;
            const int xd = own ? dyni : dynj;
            if (dyn_bptnr(xd) == hbp) {
                stage_pair();
                const double d2 = pair_r2(own ? i : j, hbp, tf);
                ct = uni((d2 - T.sigma_sq[dyn_ident(xd)][dyn_ident(dyn_of(hbp))]) < 0.0 ? 13 : 6);
            } else
                ct = 15;
        }
        int status = 0;
        double bd = 0.0;
        int sgn = 0;
        const double gx = g.rx, gy = g.ry, gz = g.rz;
        const double rk = comp == 0 || comp == 3 ? gx : (comp == 1 || comp == 4 ? gy : gz);
        const bool hit = ct < 14;
        double ratio = 0.0;
        const double bmj = readlane_d(val, 14);
        if (hit) {
            const double2 bwi = make_double2(readlane_d(val, 22), readlane_d(val, 23));
            impulse(T, g, bmi, bmj, idi, idj, bwi, dyn_bptnr(dyni) == j, evcode, ct, ratio, bd, sgn, status);
            ct = uni(ct);
            sgn = uni(sgn);
        } else {
            // bumped.f: push the pair off the discontinuity
            bd = evcode >= 40 ? kSm * sqrt(T.shlddia_sq[idi][idj]) : kSm * sqrt(T.welldia_sq[idi][idj]);
            sgn = uni(g.b < 0.0 ? -1 : 1);
        }
        if (sgn != 0) {
            const double nd = bd * rk;
            val = ispos ? ((sgn < 0) != jside ? val - nd : val + nd) : val;
        }
        if (hit) {
            // v -+ dv / m, x +- dv tf / m: one division per component lane
            const double dv = ratio * rk;
            const double q = (ispos ? dv * tf : dv) / (jside ? bmj : bmi);
            const bool neg = isvel ? !jside : jside;
            val = ispos || isvel ? (neg ? val - q : val + q) : val;
        }
        if (ct >= 20) {
            if (ct == 20) {
                if (idi + idj == 5) {
                    dyni = make_dyn(idi + 4, j);
                    dynj = make_dyn(idj + 4, i);
                    if (ok) {
                        if (bk >= 1) {
                            spec_abort_at(bk, nb);
                            return 0;
                        }
                        if (lane == 0) status |= idi < idj ? repuls_add(i, Li, j, Lj) : repuls_add(j, Lj, i, Li);
                        fence = true;
                    }
                }
            } else if (ct == 21) {
                if (idi <= 8) {
                    if (ok) {
                        if (bk >= 1) {
                            spec_abort_at(bk, nb);
                            return 0;
                        }
                        if (lane == 0) status |= idi < idj ? repuls_del_a(i, Li, j, Lj) : repuls_del_a(j, Lj, i, Li);
                        xdel = true;
                        fence = true;
                    }
                    if (dyn_bptnr(dyni) == j) {
                        dyni = make_dyn(idi - 4, -1);
                        dynj = make_dyn(idj - 4, -1);
                    }
                }
            } else if (ct == 24 || ct == 25) {
                flags |= kPairReadsSp;
                const bool own = evcode < 45;
                const int hbp = own ? xi.w : xj.w, x = own ? i : j;
                int xdyn = own ? dyni : dynj, hdyn = dyn_of(hbp);
                const int idx = dyn_ident(xdyn), idh = dyn_ident(hdyn);
                bool changed = false;
                if (ct == 24 && idx + idh == 5) {
                    xdyn = make_dyn(idx + 4, hbp);
                    hdyn = make_dyn(idh + 4, x);
                    changed = true;
                } else if (ct == 25 && idx >= 5) {
                    xdyn = make_dyn(idx - 4, -1);
                    hdyn = make_dyn(idh - 4, -1);
                    changed = true;
                }
                if (changed) {
                    if (own) dyni = xdyn;
                    else dynj = xdyn;
                    if (hbp == i) dyni = hdyn;
                    else if (hbp == j) dynj = hdyn;
                    else {
                        if (bk >= 1) {
                            spec_abort_at(bk, nb);
                            return 0;
                        }
                        if (lane == 0) gs1(&H.rec[hbp].dyn, hdyn);
                        fence = true;
                    }
                }
            }
            const int di = dyni, dj = dynj;
            const int dd = jside ? dj : di;
            val = lane < 16 && comp == 7 ? __hiloint2double(dd, __double2loint(val)) : val;
        } else if ((ct == 14 || ct == 16) && ok) {
            if (bk >= 1) {
                spec_abort_at(bk, nb);
                return 0;
            }
            if (lane == 0) {
                if (ct == 14)
                    status |= idi < idj ? repuls_add(i, Li, j, Lj) : repuls_add(j, Lj, i, Li);
                else
                    status |= idi < idj ? repuls_del_a(i, Li, j, Lj) : repuls_del_a(j, Lj, i, Li);
            }
            xdel = ct == 16;
            fence = true;
        }
        if (bk < 1) store_pair();  // a speculative event writes its pair once committed
        if (fence) {
            flags |= kPairWroteSp;
            // shoulder tables changed: make them visible before the predictions
            wave_sync_mem();
            xi = uni(ld_at(H.extra, i));
            xj = uni(ld_at(H.extra, j));
        }
        st0 = wave_status(status);
        PH_END(sdev(), kPhPair, tph);
    } else {
        const SysDev& S = sdev();
        const int N = H.N;
        // the three logarithms in lanes 0 to 2, the velocity scales in lanes 0 and 1
        const double d1 = gd.r, d2 = gd.wr, d3 = gd.tg, p1 = gd.v1, p2 = gd.v2, p3 = gd.w1;
        const double lr = lane == 0 ? d1 : (lane == 1 ? d2 : d3);
        const double lg = dlog(lr);
        const double fact = sqrt(-2.0 * S.setemp * bmi * lg / lr);
        const double f0 = readlane_d(fact, 0), f1 = readlane_d(fact, 1);
        const double v_old = up3(val);  // (lane moves need every lane: not inside a select)
        val = lane < 3 ? val + v_old * tf : val;
        const double nv = (lane == 3 ? p1 * f0 : (lane == 4 ? p2 * f0 : p3 * f1)) / bmi;
        val = lane >= 3 && lane < 6 ? nv : val;
        const double v_new = up3(val);
        val = lane < 3 ? val - v_new * tf : val;
        if (gd.guard >= 1000) st0 = kErrRng;
        const double tg = -1.0 * readlane_d(lg, 2) * S.avegtime + tf;
        int status = 0;
        Leaf g;
        g.tim = tg;
        g.nptnr = -2;
        g.meta = make_meta(bin_of(interval_max, tbin_off, sortsize, nbin, tg, status), -2);
        store_pair();
        if (lane == 0) {
            leaf_st(H, N, g);
            stamp_st(H, N, mk_stamp(coll, 1));  // added before partial_events' adds (main.F90:1041-1049)
            mc.rc0 = gd.rc;
            mc.numghosts++;
            B.gbead = i;
        }
        if (status && !st0) st0 = status;
        const double tf_old = uni(mc.old_tfalse);
        if (tf < tf_old) {
            tf = tf_old;
            if (lane == 0) mc.tfalse = tf;
        }
        xj = make_int4(-1, -1, -1, -1);
        extra_blk = N / kBlk;
        ct = 0;
        PH_END(sdev(), kPhGhost, tph);
    }
    if (lane == 0) B.ty[bk] = ct;

    // place of i's add among this event's calendar adds (a ghost event adds
    // its own entry first); j follows, then the down set in list order
    const int sub0 = j >= 0 ? 1 : 2;
    const double T0 = interval_max + kLt - tf;
    // an entry of the list: bead | up-row length of a down bead << 16 (127:
    // not known) | static code << 24 (63: not known) | tag << 30
    const int kNoRow = (0x3F << 24) | (127 << 16);
    const bool has_x = (xi.x & xi.y & xi.z & xj.x & xj.y & xj.z) != -1;  // any shoulder partner
    bool multi = nui + ndi + nuj + ndj + (has_x ? 12 : 0) > kLaneI;
    int ncand = 0, n0 = 0, ntot = 0, m = 0, tag = 0, stat = 0, nspec = 0;
    int cI = 0, cJ = 0, pI = lane, pJ = lane;
    bool first = false, is_i = false, spec = false, dn = false, act = false, late = false;
    unsigned long long dups = 0;
    Rec mine;
    int4 om = make_int4(-1, -1, -1, -1);
    double2 bwm = make_double2(0.0, 0.0);
    Leaf lf0;
    lf0.tim = 0.0;
    lf0.nptnr = -1;
    lf0.meta = 0;
    unsigned long long specm = 0;
    if (!multi) {
        // ---- the entry list: candidates of i, candidates of j, the down set
        //      in reference order (i's down list and lower shoulder partners, then j's)
        const int kDnI = (int)0x80000000u, kDnJ = (int)0xC0000000u, kCaJ = 0x40000000;
        int nDi;
        if (!has_x) {
            const bool keep = lane < ndj && (edj & 0xFFFF) != i;
            const unsigned long long bal = __ballot(keep);
            ncand = nui + nuj;
            nDi = ndi;
            n0 = ncand + ndi + __popcll(bal);
            if (lane < nui) W.lst[lane] = eui;
            if (lane < nuj) W.lst[nui + lane] = euj | kCaJ;
            if (lane < ndi) W.lst[ncand + lane] = edi | kDnI;
            if (keep) W.lst[ncand + ndi + before_me(bal)] = edj | kDnJ;
        } else {
            int w = nui;
            if (lane < nui) W.lst[lane] = eui;
            auto one = [&](int b, int tg) __attribute__((always_inline)) {
                if (lane == 0) W.lst[w] = b | tg | kNoRow;
                ++w;
            };
            auto uppers = [&](const int4& x, int b, int tg) __attribute__((always_inline)) {
                if (x.x > b) one(x.x, tg);
                if (x.y > b) one(x.y, tg);
                if (x.z > b) one(x.z, tg);
            };
            auto lowers = [&](const int4& x, int b, int tg) __attribute__((always_inline)) {
                if (x.x >= 0 && x.x < b) one(x.x, tg);
                if (x.y >= 0 && x.y < b) one(x.y, tg);
                if (x.z >= 0 && x.z < b) one(x.z, tg);
            };
            uppers(xi, i, 0);
            if (lane < nuj) W.lst[w + lane] = euj | kCaJ;
            w += nuj;
            if (j >= 0) uppers(xj, j, kCaJ);
            ncand = w;
            if (lane < ndi) W.lst[w + lane] = edi | kDnI;
            w += ndi;
            lowers(xi, i, kDnI);
            nDi = w - ncand;
            if (j >= 0) {
                const bool keep = lane < ndj && (edj & 0xFFFF) != i;
                const unsigned long long bal = __ballot(keep);
                if (keep) W.lst[w + before_me(bal)] = edj | kDnJ;
                w += __popcll(bal);
                lowers(xj, j, kDnJ);
            }
            n0 = w;
        }
        // the base beads i and j
        if (lane < 16) reinterpret_cast<double*>(&W.base[jside ? 1 : 0].r)[comp] = val;
        if (lane >= 22 && lane < 26) reinterpret_cast<double*>(&W.base[(lane - 22) >> 1].bw)[lane & 1] = val;
        if (lane < 2) W.base[lane].idx = lane == 0 ? i : j;
        if (lane < kOwners) {
            W.tkey[lane] = ~0ull;
            W.win[lane] = kW;
        }
        wave_sync();
        PH_END(sdev(), kPhRows, tph);
        // ---- every entry's bead; a down entry's own calendar entry and bond window
        act = lane < n0;
        const int ent = act ? W.lst[lane] : 0;
        m = ent & 0xFFFF;
        tag = (int)((unsigned)ent >> 30);
        stat = (ent >> 24) & 0x3F;
        dn = act && lane >= ncand;
        if (dn) lf0 = leaf_ld(H, m);
        if (act) {
            mine = ld_at(H.rec, m);
            om = ld_at(H.ovr, m);
        }
        if (dn) bwm = ld_at(H.bw, m);
        // ---- down entries of one bead: its ops with i and with j, and the
        //      lane of an op of each kind (equal predictions)
        const int rj0 = ncand + nDi, key = dn ? m : -1 - lane;
        if (!has_x) {
            // a row holds a bead once: only an entry of i and one of j can be
            // of one bead.  An entry of i looks for its mate, and tells it.
            int mate = -1;
            for (int r = rj0; r < n0; ++r) mate = key == __builtin_amdgcn_readlane(key, r) ? r : mate;
            const bool of_i = dn && lane < rj0, both = of_i && mate >= 0;
            cI = of_i ? 1 : 0;
            cJ = mate >= 0 ? 1 : 0;
            pJ = mate >= 0 ? mate : lane;
            const int told = __builtin_amdgcn_ds_permute((both ? mate : kLaneJ) << 2, both ? 1 : 0);
            dups = __ballot(dn && told != 0);
        } else {
            int r = ncand;
            unsigned long long above = ~((2ull << r) - 1ull);
            for (; r < rj0; ++r, above <<= 1) {
                const bool eq = key == __builtin_amdgcn_readlane(key, r);
                cI += eq ? 1 : 0;
                pI = eq ? r : pI;
                dups |= __ballot(eq) & above;
            }
            for (; r < n0; ++r, above <<= 1) {
                const bool eq = key == __builtin_amdgcn_readlane(key, r);
                cJ += eq ? 1 : 0;
                pJ = eq ? r : pJ;
                dups |= __ballot(eq) & above;
            }
        }
        first = dn && !((dups >> lane) & 1ull);
        is_i = first && m == i;
        // a bead whose updates may take a full recompute
        spec = first && !is_i && ((lf0.nptnr == i && cI > 0) || (lf0.nptnr == j && cJ > 0) || cI >= 2 || cJ >= 2);
        specm = __ballot(spec);
        nspec = __popcll(specm);
        multi = nspec > kMaxSpec;
        if (!multi) {
            // ---- their candidates: up rows (the entry carries the length)
            //      and upper shoulder partners, a lane each from n0 on
            int4 xl = make_int4(-1, -1, -1, -1);
            if (spec) xl = ld_at(H.extra, m);
            int w2 = n0, rowat = -1, q = 0;
            for (unsigned long long sm = specm; sm; sm &= sm - 1, ++q) {
                const int src = __ffsll((long long)sm) - 1;
                const int l = __builtin_amdgcn_readlane(m, src);
                int nu = (__builtin_amdgcn_readlane(ent, src) >> 16) & 127;
                if (nu == 127) nu = uni(gl1(H.nup + l));
                const int k = lane - w2;
                if (k >= 0 && k < nu) {
                    rowat = l * cap + k;
                    tag = 4 + q;
                }
                w2 += nu;
            }
            late = lane >= n0 && lane < w2;
            int ent2 = 0;
            if (late) ent2 = ld_at(H.nb_up, rowat);
            const unsigned long long xm = __ballot(spec && (xl.x > m || xl.y > m || xl.z > m));
            // (a load's unused word would free its register at once, and the
            // next value there wait for every load in flight)
            asm volatile("" ::"v"(xl.w));
            if (xm) {
                // shoulder partners follow their rows' order within an owner
                // because the owner's least position wins only among equal times
                q = 0;
                for (unsigned long long sm = specm; sm; sm &= sm - 1, ++q) {
                    const int src = __ffsll((long long)sm) - 1;
                    if (!((xm >> src) & 1ull)) continue;
                    const int l = __builtin_amdgcn_readlane(m, src);
#pragma unroll
                    for (int u = 0; u < 3; ++u) {
                        const int x = __builtin_amdgcn_readlane(u == 0 ? xl.x : (u == 1 ? xl.y : xl.z), src);
                        if (x > l) {
                            if (lane == w2) {
                                ent2 = x | kNoRow;
                                tag = 4 + q;
                                late = true;
                            }
                            ++w2;
                        }
                    }
                }
            }
            multi = w2 > kLaneI;
            ntot = w2;
            PH_END(sdev(), kPhScan, tph);
            // the pair's own beads take their new states
            if (act && (m == i || m == j)) mine = W.base[m == i ? 0 : 1].r;
            if (spec) {
                BaseRec& b = W.base[2 + before_me(specm)];
                b.r = mine;
                b.bw = bwm;
                b.idx = m;
            }
            if (late && !multi) {
                m = ent2 & 0xFFFF;
                stat = (ent2 >> 24) & 0x3F;
                om = ld_at(H.ovr, m);
                mine = ld_at(H.rec, m);
            }
        }
    }
    if (multi) {
        // only the first wavefront has the multi-pass form's work lists: a
        // speculative event that needs them waits to lead a round
        if (bk >= 1) {
            spec_abort_at(bk, nb);
            return 0;
        }
        const Lds& L = ldsv();
        stage_pair();
        {
            Pair& P = *L.pair();
            if (lane >= 22 && lane < 26) reinterpret_cast<double*>(lane < 24 || ghost ? &P.bwi : &P.bwj)[lane & 1] = val;
            if (ghost && lane >= 22 && lane < 24) reinterpret_cast<double*>(&P.bwj)[lane & 1] = val;
            if (ghost && lane < 8) reinterpret_cast<double*>(&P.rj)[comp] = val;
            if (lane == 0) {
                P.flags = flags;
                P.pad = 0;
                if (st0 && !mc.status) mc.status = st0;
            }
        }
        wave_sync();
        reschedule(sdev(), T, L, *L.sc(), *L.pair(), extra_blk, xdel, batch ? 0 : -1);
        if (solo) bar_to(nb, 1);
        // its new entries are not offered to the pool
        for (int q = lane; q < B.nbl; q += kW) dirty_or(par, L.blist()[q]);
        if (lane == 0) {
            B.full = 1;
            if (solo) B.st[0] = 0;
            B.st_rep[0] = 0;
        }
        return batch ? accepted(B) : 1;
    }
    PH_END(sdev(), kPhLoads, tph);
    const int own = lane == kLaneI ? i : (lane == kLaneJ ? j : -1);  // the result lanes' beads
    int rep = -1;   // earlier event whose calendar-entry write this bead's updates replay on
    int sp = -1;    // the lane's bead of the shoulder set
    const bool sp_w = (flags & kPairWroteSp) != 0, sp_r = (flags & kPairReadsSp) != 0;
    // ---- a round's footprint check.  Marks per bead: bit k = wavefront k
    //      rewrites the bead's state, bit 8+k = it rewrites the bead's
    //      calendar entry, bit 16+k = that rewrite may be a full recompute.
    //      Event k commits only if no earlier event of the round rewrites a
    //      state it reads or an entry it rewrites; a later event reads the
    //      state before this one's writes (they wait for the round's last
    //      barrier), as in the serial order.  One exception: a down bead
    //      whose entry exactly one earlier event rewrote by single-pair
    //      updates only, and whose own updates here are single-pair ones,
    //      replays those updates on that event's entry once it is written.
    auto clear_marks = [&]() __attribute__((always_inline)) {
        if (dn) mark_clear(H, m);
        if (own >= 0) mark_clear(H, own);
        if (bk == 0 && sp_w && sp >= 0) mark_clear(H, sp);
    };
    if (batch) {
        const unsigned sbit = 1u << bk, lbit = 1u << (8 + bk), fbit = 1u << (16 + bk);
        if ((bk == 0 && sp_w) || (bk >= 1 && sp_r)) {
            stage_pair();
            sp = shoulder_bead(sdev(), *ldsv().pair(), lane);
        }
        if (lane == 0) B.wdone[bk] = 0;
        if (dn || own >= 0) mark_or(H, dn ? m : own, dn ? lbit | (spec ? fbit : 0u) : sbit | lbit | fbit);
        if (bk == 0 && sp_w && sp >= 0) mark_or(H, sp, sbit);
        bar_to(nb, 1);
        PH_END(sdev(), kPhBMark, tph);
        if (bk >= 1) {
            const unsigned lowS = sbit - 1u, lowL = lowS << 8;
            const bool look = lane < ntot || own >= 0;
            bool bad = false;
            if (look) {
                const unsigned mk = mark_get(H, own >= 0 ? own : m);
                bad = (mk & lowS) != 0u;
                if (own >= 0) bad = (mk & (lowS | lowL)) != 0u;
                if (!bad && first && (mk & lowL)) {
                    // (other lanes of the same bead leave it to its first)
                    const unsigned wl = (mk & lowL) >> 8;
                    const int q = __ffs(wl) - 1;
                    if (!is_i && (wl & (wl - 1u)) == 0u && !(mk & (1u << (16 + q))) && !spec)
                        rep = q;
                    else
                        bad = true;
                }
            }
            if (sp_r && sp >= 0 && (mark_get(H, sp) & lowS)) bad = true;
            if (__ballot(bad) && lane == 0) atomicMin(&B.cut, bk);
            PH_END(sdev(), kPhBCheck, tph);
            // the cut only moves down: a wavefront already past it stops here
            // (the others learn theirs at the next barrier)
            wave_sync();
            if (bk >= uni(B.cut)) {
                bar_to(nb, kRoundBars);
                clear_marks();
                return 0;
            }
        }
    }
    // ---- the predictions: the entry's bead against its base bead
    PH_ADDN(sdev(), kPhNPred, ntot);
    PH_ADDN(sdev(), kPhNPredPass, 1);
    act = lane < ntot;
    wave_sync();
    double tij = 1000000000.0;
    int ty = 0, status = 0;
    const int slot = tag < 4 ? (tag & 1) : tag - 2;
    if (act) {
        const BaseRec& b = W.base[slot];
        const Rec rb = b.r;
        const int bidx = b.idx;
        const double2 bwb = b.bw;
        if (late && (m == i || m == j)) mine = W.base[m == i ? 0 : 1].r;
        Geo g;
        geo(rb, mine, tf, g);  // the order of the two only flips the signs of vectors
        if (stat == 0x3F) stat = static_t(T, mine.topo, rb.topo);  // symmetric in its beads
        const int code = dyn_code(om, bidx, stat);  // ev_code(m, x) of a candidate, ev_code(l, p) of a down bead
        const int adyn = dn ? mine.dyn : rb.dyn, cdyn = dn ? rb.dyn : mine.dyn;  // the lower bead's first
        const double2 bwa = make_double2(dn ? bwm.x : bwb.x, dn ? bwm.y : bwb.y);
        predict_geo(T, code, dyn_ident(adyn), dyn_ident(cdyn), dyn_bptnr(adyn) == (dn ? bidx : m), bwa, g, tij, ty);
    }
    // a down bead's prediction is checked where its op uses it
    const bool err_c = ty == -99, err_t = tij < 0.0 && fabs(tij) > 1.0e-10;
    if (act && !dn) status = err_t ? kErrNegativeTime : (err_c ? kErrBadCode : 0);
    // ---- each owner's least (time, list position)
    const unsigned long long tk = t_order(tij);
    const bool cnd = act && !dn;
    if (cnd) atomicMin(&W.tkey[slot], tk);
    if (dups) {
        W.wt[lane] = tij;
        W.wy[lane] = ty;
    }
    wave_sync();
    if (cnd && tk == W.tkey[slot]) atomicMin(&W.win[slot], lane);
    PH_END(sdev(), kPhPred, tph);
    // an owner's result, on its lane: those of i and j, and the lanes of the
    // beads recomputed (full recompute rule: an event only below T0)
    double ft = T0 + tf;
    int fp = -1, fc = -1;
    {
        const int rslot = lane == kLaneI || is_i ? 0 : (lane == kLaneJ ? 1 : 2 + before_me(specm));
        wave_sync();
        const int src = own >= 0 || is_i || spec ? W.win[rslot] : kW;
        const double bt = __shfl(tij, src & (kW - 1), kW);
        const int bp = __shfl(m, src & (kW - 1), kW), bc = __shfl(ty, src & (kW - 1), kW);
        if (src < kW && bt < T0) {
            ft = bt + tf;
            fp = bp;
            fc = bc;
        }
    }
    // ---- each down bead's ops, those with i first
    const bool whole = is_i || own >= 0;
    double st_t = whole ? ft : lf0.tim;
    int st_p = whole ? fp : lf0.nptnr, st_c = whole ? fc : leaf_ct(lf0.meta);
    bool modified = false;
    double sI = tij, sJ = tij;
    int yI = ty, yJ = ty;
    if (dups) {
        sI = W.wt[pI];
        yI = W.wy[pI];
        sJ = W.wt[pJ];
        yJ = W.wy[pJ];
    }
    auto op = [&](bool on, int p, double t, int y) __attribute__((always_inline)) {
        const bool full = on && st_p == p;
        const bool single = on && !full;
        if (single && y == -99) status = kErrBadCode;
        if (single && t < 0.0 && fabs(t) > 1.0e-10) status = kErrNegativeTime;
        const double tt = t + tf;
        const bool less = single && tt < st_t;
        st_t = full ? ft : (less ? tt : st_t);
        st_p = full ? fp : (less ? p : st_p);
        st_c = full ? fc : (less ? y : st_c);
        modified |= full || less;
    };
    op(first && cI >= 1, i, sI, yI);
    if (has_x && __ballot(first && cI >= 2)) {
        for (int k = 2; k <= 4; ++k) op(first && cI >= k, i, sI, yI);
    }
    op(first && cJ >= 1, j, sJ, yJ);
    if (has_x && __ballot(first && cJ >= 2)) {
        for (int k = 2; k <= 4; ++k) op(first && cJ >= k, j, sJ, yJ);
    }
    // bead i's state, with the updates of the entry that names it among j's
    // down set, is written by i's lane
    const unsigned long long im = __ballot(is_i);
    if (im) {
        const int src = __ffsll((long long)im) - 1;
        const double t = readlane_d(st_t, src);
        const int p = __builtin_amdgcn_readlane(st_p, src), y = __builtin_amdgcn_readlane(st_c, src);
        st_t = lane == kLaneI ? t : st_t;
        st_p = lane == kLaneI ? p : st_p;
        st_c = lane == kLaneI ? y : st_c;
    }
    // ---- the new calendar entries, one per lane: the modified down beads',
    //      i's and j's
    const bool wr = (modified && !is_i) || own >= 0;
    const int rb = own >= 0 ? own : m;
    const unsigned long long stp = mk_stamp(coll, own >= 0 ? sub0 + (lane - kLaneI) : sub0 + 2 + (lane - ncand));
    Leaf lf;
    lf.tim = st_t;
    lf.nptnr = st_p;
    lf.meta = 0;
    if (wr) lf.meta = make_meta(bin_of(interval_max, tbin_off, sortsize, nbin, st_t, status), st_c);
    status = wave_status(status);
    if (status && !st0) st0 = status;
    // the keys they will have; a ghost event's own new entry takes the idle lane of j
    Key kn = wr ? leaf_key(lf, rb) : empty_key();
    unsigned long long ks = stp;
    if (ghost && lane == kLaneJ) {
        kn = leaf_key(leaf_ld(H, H.N), H.N);
        ks = mk_stamp(coll, 1);  // re-added by this ghost event
    }
    PH_END(sdev(), kPhDown, tph);
    int A = 1;
    if (batch) {
        // report the least new calendar key and the status, then commit
        // only within the round's accepted prefix
        // (only one ahead of the round's last entry can end the prefix)
        unsigned long long kns = 0;
        Key kl = empty_key();
        if (__ballot(key_proxy(kn) <= key_proxy(B.key[K - 1]))) kl = key_min_wave_st(kn, ks, kns);
        if (lane == 0) {
            B.knew[bk] = kl;
            B.knew_st[bk] = kns;
            B.st[bk] = st0;
            B.st_rep[bk] = 0;
        }
        bar_to(nb, kRoundBars);
        PH_END(sdev(), kPhBKeys, tph);
        // every wavefront has checked: clear this one's marks
        clear_marks();
        A = accepted(B);
        if (bk >= A) return 0;
        if (bk >= 1) store_pair();
        if (bk == 0 && st0 && lane == 0 && !mc.status) mc.status = st0;
    } else {
        if (lane == 0) {
            B.st[0] = 0;
            B.st_rep[0] = 0;
            if (st0 && !mc.status) mc.status = st0;
        }
        bar_to(nb, 1);  // the pool's edge is known
    }
    bool wb = wr;  // the lane's bead takes a new entry (its block is rescanned)
    if (__ballot(rep >= 0)) {
        int st2 = 0;
        if (rep >= 0) {
            // the earlier event's entry first, then this event's single-pair
            // updates on it (i before j, eventredo_down.f), as the serial order
            // would have applied them
            while (__hip_atomic_load(&B.wdone[rep], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) == 0)
                __builtin_amdgcn_s_sleep(1);
            const Leaf cur = leaf_get_fresh(ldsv(), m);
            lf = cur;
            int rc = leaf_ct(cur.meta);
            wb = false;
            if (cI > 0 && sI + tf < lf.tim) {
                lf.tim = sI + tf;
                lf.nptnr = i;
                rc = yI;
                wb = true;
            }
            if (cJ > 0 && sJ + tf < lf.tim) {
                lf.tim = sJ + tf;
                lf.nptnr = j;
                rc = yJ;
                wb = true;
            }
            if (wb) lf.meta = make_meta(bin_of(interval_max, tbin_off, sortsize, nbin, lf.tim, st2), rc);
            kn = wb ? leaf_key(lf, rb) : empty_key();
        }
        st2 = wave_status(st2);
        if (st2 && lane == 0) B.st_rep[bk] = st2;
    }
    if (wb) {
        leaf_st(H, rb, lf);
        stamp_st(H, rb, stp);
    }
    {
        const bool gl = ghost && lane == kLaneJ;
        if (wb || gl) dirty_or(par, gl ? extra_blk : rb / kBlk);
        const bool near = key_proxy(kn) < B.edge;
        const unsigned long long nm = __ballot(near);
        const int n = __popcll(nm), cap_f = 1 << fsh, pos = before_me(nm);
        if (near && pos < cap_f) B.fresh[(bk << fsh) + pos] = kn;
        if (lane == 0) {
            B.nfresh[bk] = min(n, cap_f);
            if (n > cap_f) B.full = 1;
        }
    }
    // repuls_del_b.f once the rescheduling is done
    if (xdel && lane == 0) {
        const bool iN = dyn_ident(dyni) < dyn_ident(dynj);
        const int a = iN ? i : j, b = iN ? j : i;
        const int La = topo_len(iN ? topoi : topoj), Lb = topo_len(iN ? topoj : topoi);
        shoulders_clear(a, La, b, Lb);
    }
    if (batch) {
        // the round's tree update runs after every committed event's
        // writes; a later event that replays on these entries waits for
        // the flag
        wave_sync_mem();
        if (lane == 0) __hip_atomic_store(&B.wdone[bk], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    PH_END(sdev(), kPhLeaf, tph);
    return A;
}

// ------------------------------------------------------------------------
// neighbour lists: nbor.f membership restated for a coarse-cell search
// ------------------------------------------------------------------------
// Pair (i, j) is listed when its fine cells (cell_add.f binning) are within
// the n_wrap=2 stencil (|d| <= 2 per axis, periodic) and either its code is
// a bond/local one (4-12, 17-26) or r^2 <= rlsq(code) (nbor.f:63-128).
// Steps: the fine and coarse cell of every bead and its place in the coarse
// cell (the count's atomic returns it; places come in any order, the rows are
// sorted afterwards); the cells' starts; copies of position, topology and
// fine cell in cell order; then a wavefront per coarse cell tests the beads
// of the cells around it (list_search).
//
// A wavefront's LDS scratch of a small system's list rebuild (the staged
// beads).  It lies over the work areas, block minima and leaves, which a
// rebuild leaves free.
constexpr int kScratch = 15872;
// v mod m for v in [-1, m]
__device__ inline int wrap1(int v, int m) { return v < 0 ? v + m : (v >= m ? v - m : v); }
// fine cell of a bead (cell_add.f), 10 bits per axis
__device__ inline int fine_cell(const SysDev& S, double x, double y, double z) {
    const int M = S.M;
    int cx = (int)((x + S.half) / S.width);
    int cy = (int)((y + S.half) / S.width);
    int cz = (int)((z + S.half) / S.width);
    cx = ((cx % M) + M) % M;
    cy = ((cy % M) + M) % M;
    cz = ((cz % M) + M) % M;
    return cx | (cy << 10) | (cz << 20);
}
// The coarse cell of a fine one: cq >= 2 fine cells each, the last one takes
// the remainder, so every fine cell within the n_wrap = 2 stencil of a bead's
// lies in the 27 coarse cells around the bead's own.
__device__ inline void coarse_of(int f, int cq, int Mq, int& qx, int& qy, int& qz) {
    qx = min((f & 1023) / cq, Mq - 1);
    qy = min(((f >> 10) & 1023) / cq, Mq - 1);
    qz = min((f >> 20) / cq, Mq - 1);
}
// bead k: fine cell (cfp), coarse cell and place in it
__device__ inline void list_cell(const SysDev& S, int Mq, int k, const Rec& b) {
    const int f = fine_cell(S, b.x, b.y, b.z);
    int qx, qy, qz;
    coarse_of(f, S.cq, Mq, qx, qy, qz);
    const int key = qx + Mq * (qy + Mq * qz);
    gs1(&S.cfp[k].x, f);
    gs1(S.ckey + (k), key);
    gs1(S.crank + (k), atomicAdd(&S.ccnt[key], 1));
}
// the same for beads [tid, N) by nthr
__device__ inline void list_cells(const SysDev& S, int tid, int nthr) {
    const int N = S.N, Mq = S.M / S.cq;
#pragma unroll 2
    for (int k = tid; k < N; k += nthr) list_cell(S, Mq, k, gld(S.rec + (k)));
}
// wave-inclusive sum
__device__ inline int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return v;
}
// Exclusive scan of the NC cell counts into the cells' starts on the
// workgroup's nw wavefronts, a contiguous part each: its sum, then (after the
// others' sums) its starts.  The counts, made by atomics and read at the L2,
// are zero again afterwards.  part: nw words of LDS.
__device__ inline void list_scan(int* cnt, int* start, int NC, int* part, int wave, int nw) {
    const int lane = lane_id();
    const int seg = ((NC + nw - 1) / nw + 255) / 256 * 256, lo = min(wave * seg, NC), hi = min(lo + seg, NC);
    auto at = [&](int q) { return q < hi ? __hip_atomic_load((GLB int*)cnt + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0; };
    int sum = 0;
#pragma unroll 4
    for (int q = lo + lane; q < hi; q += kW) sum += at(q);
    sum = __builtin_amdgcn_readlane(wave_scan(sum), kW - 1);
    if (lane == 0) part[wave] = sum;
    wg_sync(nw);
    int carry = 0, all = 0;
    for (int w = 0; w < nw; ++w) {
        carry += w < wave ? part[w] : 0;
        all += part[w];
    }
    for (int base = lo; base < hi; base += 4 * kW) {
        int v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = at(base + u * kW + lane);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int q = base + u * kW + lane, incl = wave_scan(v[u]);
            if (q < hi) {
                gs1(start + q, carry + incl - v[u]);
                gs1(cnt + q, 0);
            }
            carry += __builtin_amdgcn_readlane(incl, kW - 1);
        }
    }
    if (wave == 0 && lane == 0) gs1(start + NC, all);
}
// beads [tid, N) by nthr to their sorted places
__device__ inline void list_copy(const SysDev& S, int tid, int nthr) {
#pragma unroll 2
    for (int k = tid; k < S.N; k += nthr) {
        const Rec b = gld(S.rec + (k));
        const int p = gl1(S.cstart + (gl1(S.ckey + (k)))) + gl1(S.crank + (k));
        gst(S.spos + (p), make_double4(b.x, b.y, b.z, 0.0));
        gst(S.sinfo + (p), make_int4(k, b.topo, gl1(&S.cfp[k].x), 0));
    }
}
// The next `step` items of a list rebuild's step k for this wavefront.  Five
// wavefronts stand on four SIMDs, where two share one: even shares let the
// three others wait for them.
__device__ inline int next_share(int k, int step) {
    int v = 0;
    if (lane_id() == 0) v = atomicAdd(&round_rec().share[k], step);
    return uni(v);
}
// A wavefront's scratch of list_search: a window of candidates, the queue of
// pairs (bead of the cell << 16 | place in the window) and, per bead of the
// cell, its up and down entries and the later beads of its fine cell.
constexpr int kWindow = 2 * kW;  // candidates staged at a time
struct SearchLds {
    double x[kWindow], y[kWindow], z[kWindow];
    int bead[kWindow], topo[kWindow], fine[kWindow];
    int q[2 * kW];
    int cnt[3][kW];
};
constexpr int kSearchStride = kScratch / 2;
static_assert(sizeof(SearchLds) <= kSearchStride && kSearchStride % 16 == 0, "two wavefronts search in one's rebuild scratch");
constexpr int kCells = 16;  // sorted places whose cells a wavefront takes at a time
// The lists of the coarse cells whose first sorted bead lies in the kCells
// places from i0 on (one wavefront): rows, their lengths, and each bead's
// place in its fine cell's list as cell_add.f builds it (head first: the
// highest index at 1) with the up-row length in cfp.  mx: longest row met.
// A cell of four beads has some 35 candidates in the 27 cells around it at
// 6144 beads, 29 of them inside the stencil.  What bounds a cell is its chain:
// its rows' starts and beads (loaded while the cell before is searched), its
// candidates (staged in LDS), the pairs.  A bead is first tested against 64
// candidates by the stencil alone, a dozen instructions on packed bytes; the
// pairs that pass are queued, and batches of 64 of them take the exact test,
// ninety instructions on full lanes.  Testing each of a cell's beads exactly
// against every 64 candidates, with even shares of the cells, a list update
// (with its sort) took 412 K cycles at 512 beads, 1 820 K with 1920 at ten
// times the density, 3 850 K at 6144, on five wavefronts; so 317 K, 1 590 K
// and 3 680 K, and on eight 220 K at 512 beads and 2 420 K at 6144.
__device__ inline void list_search(const SysDev& S, const DevTables& T, int i0, SearchLds& W, int& mx, int& status) {
    const int lane = lane_id();
    const int N = uni(S.N), M = uni(S.M), cq = uni(S.cq), Mq = M / cq, cap = uni(S.cap);
    const int4* const sinfo = sgpr_ptr(S.sinfo);
    const double4* const spos = sgpr_ptr(S.spos);
    const int4* const ovr = sgpr_ptr(S.ovr);
    const int* const cstart = sgpr_ptr(S.cstart);
    int* const nb_up = sgpr_ptr(S.nb_up);
    int* const nb_dn = sgpr_ptr(S.nb_dn);
    const int ps = i0 + lane;
    int c0 = -1, c1 = -1, q = 0;
    if (lane < kCells && ps < N) {
        const int4 si = ld_at(sinfo, ps);
        int qx, qy, qz;
        coarse_of(si.z, cq, Mq, qx, qy, qz);
        q = qx | (qy << 10) | (qz << 20);
        const int key = qx + Mq * (qy + Mq * qz);
        c0 = ld_at(cstart, key);
        c1 = ld_at(cstart, key + 1);
    }
    // lane t < 9: the cells of one (y, z) neighbour row, consecutive along x;
    // lane 9 + t: the one across the box's face where there is one
    const int noff = Mq > 2 ? 3 : Mq;  // distinct offsets {0, +1, -1}
    const int t9 = lane < 9 ? lane : lane - 9, oy = t9 / 3, oz = t9 - 3 * oy;
    const bool rowl = lane < 18 && oy < noff && oz < noff;
    // a cell's rows and first 64 beads, loaded while the cell before is searched
    struct Cell {
        int b0, b1, qc, r0, len;
        int4 sb;
        double4 bp;
    };
    auto fetch = [&](int src) __attribute__((always_inline)) {
        Cell c;
        c.b0 = __builtin_amdgcn_readlane(c0, src);
        c.b1 = __builtin_amdgcn_readlane(c1, src);
        c.qc = __builtin_amdgcn_readlane(q, src);
        const int qx = c.qc & 1023, qy = (c.qc >> 10) & 1023, qz = c.qc >> 20;
        const bool wrap = Mq > 2 && (qx == 0 || qx == Mq - 1);
        const int ny = wrap1(qy + (oy == 2 ? -1 : oy), Mq), nz = wrap1(qz + (oz == 2 ? -1 : oz), Mq);
        const int row = Mq * (ny + Mq * nz), xw = qx == 0 ? Mq - 1 : 0;
        const bool on = rowl && (lane < 9 || wrap);
        c.r0 = ld_at(cstart, on ? row + (lane < 9 ? max(qx - 1, 0) : xw) : 0);
        c.len = ld_at(cstart, on ? row + (lane < 9 ? min(qx + 1, Mq - 1) : xw) + 1 : 0) - c.r0;
        const int me = min(c.b0 + lane, N - 1);
        c.sb = ld_at(sinfo, me);
        c.bp = ld_at(spos, me);
        return c;
    };
    unsigned long long heads = __ballot(c0 == ps);
    if (heads == 0) return;
    Cell next = fetch(__ffsll((long long)heads) - 1);
    while (heads) {
        const Cell cell = next;
        heads &= heads - 1;
        next = fetch(heads ? __ffsll((long long)heads) - 1 : 0);
        const int b0 = cell.b0, b1 = cell.b1, r0 = cell.r0, len = cell.len;
        const int qx = cell.qc & 1023, qy = (cell.qc >> 10) & 1023, qz = cell.qc >> 20;
        const int incl = wave_scan(len), excl = incl - len;
        const int C = __builtin_amdgcn_readlane(incl, kW - 1);
        const unsigned long long rows = __ballot(len > 0);
        // A fine cell relative to the cell's first, one byte per axis: from
        // the least of the cell before on, so the window of M cells holds
        // each residue once (the last coarse cell takes the remainder)
        const int last = M - (Mq - 1) * cq;
        auto rel = [&](int f, int o, int qc) {
            const int lo = qc > 0 ? -cq : -last;
            int d = f - o;
            d += d < lo ? M : 0;
            return d >= lo + M ? d - M : d;
        };
        auto packed = [&](int f) {
            return rel(f & 1023, qx * cq, qx) + (rel((f >> 10) & 1023, qy * cq, qy) << 8) +
                   (rel(f >> 20, qz * cq, qz) << 16);
        };
        for (int bb = b0; bb < b1; bb += kW) {
            // the cell's beads, one per lane
            const int nb = min(b1 - bb, kW);
            int4 sb = cell.sb;
            double4 bp = cell.bp;
            if (bb > b0) {
                sb = ld_at(sinfo, min(bb + lane, N - 1));
                bp = ld_at(spos, min(bb + lane, N - 1));
            }
            const int4 ob = ld_at(ovr, sb.x);
            const int brel = packed(sb.z);
            W.cnt[0][lane] = W.cnt[1][lane] = W.cnt[2][lane] = 0;
            int qh = 0, qn = 0;  // queue head and length
            const unsigned long long om = __ballot(lane < nb && (ob.x & ob.y & ob.z & ob.w) != -1);
            // the exact test of the next min(qn, 64) queued pairs
            auto drain = [&]() {
                wave_sync();
                const bool v = lane < min(qn, kW);
                const int e = v ? W.q[(qh + lane) & (2 * kW - 1)] : 0, b = e >> 16, at = e & 0xFFFF;
                const double xj = W.x[at], yj = W.y[at], zj = W.z[at];
                const int jb = W.bead[at], tj = W.topo[at], fj = W.fine[at];
                const int i = __shfl(sb.x, b, kW), ti = __shfl(sb.y, b, kW), fi = __shfl(sb.z, b, kW);
                const double xi = __shfl(bp.x, b, kW), yi = __shfl(bp.y, b, kW), zi = __shfl(bp.z, b, kW);
                // fine cells lie in [0, M): differences in (-M, M), taken mod M
                int dx = (fj & 1023) - (fi & 1023), dy = ((fj >> 10) & 1023) - ((fi >> 10) & 1023), dz = (fj >> 20) - (fi >> 20);
                dx += dx < 0 ? M : 0;
                dy += dy < 0 ? M : 0;
                dz += dz < 0 ? M : 0;
                const bool far = (dx > 2 && dx < M - 2) || (dy > 2 && dy < M - 2) || (dz > 2 && dz < M - 2);
                const bool in = v && jb != i && !far;
                const int stat = static_t(T, tj, ti);
                // ev_code(j,i), nbor.f:63: j's overrides exist only towards i's
                int code = stat;
                if (om && __ballot(in && ((om >> b) & 1ull))) {
                    const int ox = __shfl(ob.x, b, kW), oyv = __shfl(ob.y, b, kW);
                    const int ozv = __shfl(ob.z, b, kW), ow = __shfl(ob.w, b, kW);
                    if (in && ((ox >= 0 && (ox >> 8) == jb) || (oyv >= 0 && (oyv >> 8) == jb) ||
                               (ozv >= 0 && (ozv >> 8) == jb) || (ow >= 0 && (ow >> 8) == jb)))
                        code = dyn_code(ld_at(ovr, jb), i, stat);
                }
                const double rx = min_image(xi - xj), ry = min_image(yi - yj), rz = min_image(zi - zj);
                const double r2 = rx * rx + ry * ry + rz * rz;
                const bool local = (code >= 4 && code <= 12) || (code >= 17 && code < 27);
                const bool cut = code >= 1 && code <= 50 && r2 <= T.rlsq[min((unsigned)code, 50u)];
                const bool up = jb > i;
                if (in && (local || cut)) {
                    const int pos = atomicAdd(&W.cnt[up ? 0 : 1][b], 1);
                    if (pos < cap) gs1((up ? nb_up : nb_dn) + (i * cap + pos), jb | (stat << 24));
                }
                if (in && up && fj == fi) atomicAdd(&W.cnt[2][b], 1);
                qh += min(qn, kW);
                qn -= min(qn, kW);
            };
            for (int w0 = 0; w0 < C; w0 += kWindow) {
                // stage the window's candidates
                const int wn = min(C - w0, kWindow);
                int p0 = 0, p1 = 0;
                for (unsigned long long rm = rows; rm; rm &= rm - 1) {
                    const int t = __ffsll((long long)rm) - 1;
                    const int ex = __builtin_amdgcn_readlane(excl, t) - w0, st = __builtin_amdgcn_readlane(r0, t) - ex;
                    p0 = lane >= ex ? st + lane : p0;
                    p1 = lane + kW >= ex ? st + lane + kW : p1;
                }
                p0 = lane < wn ? p0 : 0;
                p1 = lane + kW < wn ? p1 : 0;
                const int4 i0_ = ld_at(sinfo, p0);
                const double4 x0 = ld_at(spos, p0);
                const int4 i1_ = ld_at(sinfo, p1);
                const double4 x1 = ld_at(spos, p1);
                wave_sync();
                W.x[lane] = x0.x;
                W.y[lane] = x0.y;
                W.z[lane] = x0.z;
                W.bead[lane] = i0_.x;
                W.topo[lane] = i0_.y;
                W.fine[lane] = i0_.z;
                W.x[lane + kW] = x1.x;
                W.y[lane + kW] = x1.y;
                W.z[lane + kW] = x1.z;
                W.bead[lane + kW] = i1_.x;
                W.topo[lane + kW] = i1_.y;
                W.fine[lane + kW] = i1_.z;
                for (int h = 0; h < wn; h += kW) {
                    const bool cand = h + lane < wn;
                    // per byte 64 + 2 + the difference to a bead of the cell:
                    // 64 to 68 inside the stencil
                    const int crel = packed(h == 0 ? i0_.z : i1_.z) + 0x424242;
                    for (int b = 0; b < nb; ++b) {
                        const int x = (crel - __builtin_amdgcn_readlane(brel, b)) ^ 0x404040;
                        const bool near = Mq <= 2 || ((x | (x + 0x030303)) & 0xF8F8F8) == 0;
                        const unsigned long long m = __ballot(cand && near);
                        if (cand && near) W.q[(qh + qn + before_me(m)) & (2 * kW - 1)] = (b << 16) | (h + lane);
                        qn += __popcll(m);
                        const bool end = h + kW >= wn && b == nb - 1;
                        while (qn >= kW || (end && qn > 0)) drain();
                    }
                }
            }
            wave_sync();
            if (lane < nb) {
                const int nu = W.cnt[0][lane], nd = W.cnt[1][lane];
                if (nu > cap || nd > cap) status = kErrListCapacity;
                mx = max(mx, max(nu, nd));
                gs1(S.nup + (sb.x), min(nu, cap));
                gs1(S.ndn + (sb.x), min(nd, cap));
                gs2(S.cfp + (sb.x), make_int2(sb.z, (1 + W.cnt[2][lane]) | (min(nu, cap) << 16)));
            }
            wave_sync();
        }
    }
}
__device__ void rebuild_lists(const SysDev&, const Lds&, Sc& c) {
    const Lds& L = ldsv();
    const SysDev& S = sdev();
    const DevTables& T = tabs();
    const int lane = lane_id(), wave = wave_id(), nw = L.nw;
    const int tid = (int)threadIdx.x, nthr = kW * nw;
    const int Mq = S.M / S.cq, NC = Mq * Mq * Mq;
    PH_BEGIN(trl);
    list_cells(S, tid, nthr);
    wg_sync(nw);
    PH_END(S, kPhLCells, trl);
    list_scan(S.ccnt, S.cstart, NC, reinterpret_cast<int*>(smem + L.o_pool), wave, nw);
    wg_sync(nw);
    PH_END(S, kPhLScan, trl);
    list_copy(S, tid, nthr);
    wg_sync(nw);
    PH_END(S, kPhLCopy, trl);
    int mx = 0, status = 0;
    if (wave < 2 * L.nwr) {  // wavefronts with scratch
        SearchLds& W = *reinterpret_cast<SearchLds*>(smem + L.o_pool + wave * kSearchStride);
        for (int i0; (i0 = next_share(0, kCells)) < S.N;) list_search(S, T, i0, W, mx, status);
    }
    PH_END(S, kPhLSearch, trl);
    status = wave_status(status);
    if (status && !c.status) c.status = status;
    mx = wave_imax(mx);
    if (lane == 0) atomicMax(&S.st->max_nb_seen, (long long)mx);
    wg_sync(nw);
}

// Neighbour lists of a small system (N <= kDenseN) without the cell sort.
// Positions, topology words, override slots and fine cells are staged in
// LDS (wavefront 0's rebuild scratch); each wavefront
// takes beads in turn, tests the fine-cell stencil of all candidates one per
// lane, and queues the (bead, candidate) pairs that pass; full 64-lane
// batches of the queue then take the pair-code and cutoff test.  Membership
// is rebuild_lists' own (the n_wrap = 2 stencil, then the bonded/local codes
// or the cutoff, nbor.f:63-128); rows come in bead-index order.
// The staging takes 60 bytes per bead of wavefront 0's scratch and its queue
// 512 bytes after it.
constexpr int kDenseN = 256;
constexpr int kDenseQ = 128;  // queue ring: under 64 entries + one pass of 64
static_assert(60 * kDenseN + 4 * kDenseQ <= kScratch, "dense list staging exceeds wavefront 0's scratch");
struct __attribute__((aligned(16))) Stage {
    double x, y, z;
    int topo, pad;
};
__device__ void rebuild_lists_dense(const SysDev&, const Lds&, Sc& c) {
    const Lds& L = ldsv();

    const SysDev& S = sdev();

    const DevTables& T = tabs();
    const int lane = lane_id(), wave = wave_id(), nw = L.nw;
    const int tid = (int)threadIdx.x, nthr = kW * nw;
    const int N = S.N, M = S.M, cap = S.cap;
    PH_BEGIN(trl);
    const int nr = L.nwr;
    unsigned char* const w0 = smem + L.o_pool;
    Stage* const stg = reinterpret_cast<Stage*>(w0);
    int4* const sovr = reinterpret_cast<int4*>(w0 + 32 * N);
    int2* const cnt = reinterpret_cast<int2*>(w0 + 48 * N);
    int* const sfine = reinterpret_cast<int*>(w0 + 56 * N);
    int* const q = wave == 0 ? reinterpret_cast<int*>(w0 + 60 * N) : reinterpret_cast<int*>(w0 + wave * kScratch);
    for (int k = tid; k < N; k += nthr) {
        const Rec b = gld(S.rec + (k));
        int cx = (int)((b.x + S.half) / S.width);
        int cy = (int)((b.y + S.half) / S.width);
        int cz = (int)((b.z + S.half) / S.width);
        cx = ((cx % M) + M) % M;
        cy = ((cy % M) + M) % M;
        cz = ((cz % M) + M) % M;
        Stage g;
        g.x = b.x;
        g.y = b.y;
        g.z = b.z;
        g.topo = b.topo;
        g.pad = 0;
        stg[k] = g;
        sovr[k] = gld(S.ovr + (k));
        sfine[k] = cx | (cy << 10) | (cz << 20);
    }
    for (int i = tid; i < N; i += nthr) cnt[i] = make_int2(0, 0);
    wg_sync(nw);
    // fine cells and each bead's place in its fine cell's list (cell_add.f:
    // head first, the highest index at 1), for the rows' nbor.f order: lane
    // k counts the later beads of its cell, 64 candidates per LDS read
    for (int k0 = wave * kW; k0 < N; k0 += nw * kW) {
        const int k = k0 + lane;
        const int f = k < N ? sfine[k] : -1;
        int pos = 1;
        for (int q0 = k0; q0 < N; q0 += kW) {
            const int v = q0 + lane < N ? sfine[q0 + lane] : -2;
#pragma unroll
            for (int m = 0; m < kW; ++m) pos += (__builtin_amdgcn_readlane(v, m) == f && q0 + m > k) ? 1 : 0;
        }
        if (k < N) {
            gs2(S.cfp + (k), make_int2(f, pos));
        }
    }
    PH_END(S, kPhLCells, trl);
    const unsigned long long below = (1ull << lane) - 1ull;
    int qh = 0, qn = 0;  // queue head and length (wavefront-uniform)
    // the pair test on the next min(qn, 64) queued pairs, in queue order
    auto drain = [&]() {
        const int nb = min(qn, kW);
        const bool v = lane < nb;
        const int e = v ? q[(qh + lane) & (kDenseQ - 1)] : 0;
        const int i = e >> 16, jb = e & 0xFFFF;
        bool take = false;
        int stat = 0;
        if (v) {
            const Stage si = stg[i], sj = stg[jb];
            const int4 oi = sovr[i];
            stat = static_t(T, sj.topo, si.topo);
            // ev_code(j,i), nbor.f:63: j's overrides exist only towards i's
            int code = stat;
            if ((oi.x >= 0 && (oi.x >> 8) == jb) || (oi.y >= 0 && (oi.y >> 8) == jb) ||
                (oi.z >= 0 && (oi.z >> 8) == jb) || (oi.w >= 0 && (oi.w >> 8) == jb))
                code = dyn_code(sovr[jb], i, stat);
            if ((code >= 4 && code <= 12) || (code >= 17 && code < 27)) {
                take = true;
            } else {
                double rx = si.x - sj.x, ry = si.y - sj.y, rz = si.z - sj.z;
                rx = rx - round(rx);
                ry = ry - round(ry);
                rz = rz - round(rz);
                const double r2 = rx * rx + ry * ry + rz * rz;
                take = code >= 1 && code <= 50 && r2 <= T.rlsq[code];
            }
        }
        const bool tu = take && jb > i, td = take && jb < i;
        const unsigned long long up = __ballot(tu), dn = __ballot(td);
        // a bead's pairs are contiguous in the queue: lanes [s, lane) of
        // this lane's segment precede it in its row
        const int ip = __shfl_up(i, 1);
        const unsigned long long hm = __ballot(v && (lane == 0 || ip != i));
        const unsigned long long hl = hm & ((2ull << lane) - 1ull);
        const int sh = hl ? 63 - __clzll(hl) : 0;
        const unsigned long long seg = below & ~((1ull << sh) - 1ull);
        const bool tail = v && (lane + 1 == nb || ((hm >> (lane + 1)) & 1ull));
        int2 b0 = make_int2(0, 0);
        if (v) b0 = cnt[i];
        if (tu) {
            const int p = b0.x + __popcll(up & seg);
            if (p < cap) gs1(S.nb_up + ((size_t)i * cap + p), jb | (stat << 24));
        }
        if (td) {
            const int p = b0.y + __popcll(dn & seg);
            if (p < cap) gs1(S.nb_dn + ((size_t)i * cap + p), jb | (stat << 24));
        }
        const unsigned long long segi = seg | (1ull << lane);
        if (tail) cnt[i] = make_int2(b0.x + __popcll(up & segi), b0.y + __popcll(dn & segi));
        qh = (qh + nb) & (kDenseQ - 1);
        qn -= nb;
    };
    for (int i = wave; wave < nr && i < N; i += nr) {
        const int fi = sfine[i];
        const int ix = fi & 1023, iy = (fi >> 10) & 1023, iz = fi >> 20;
        for (int base = 0; base < N; base += kW) {
            const int jb = base + lane;
            bool pass = false;
            if (jb < N && jb != i) {
                const int fj = sfine[jb];
                // fine cells lie in [0, M): differences in (-M, M), taken mod M
                int dx = (fj & 1023) - ix, dy = ((fj >> 10) & 1023) - iy, dz = (fj >> 20) - iz;
                dx += dx < 0 ? M : 0;
                dy += dy < 0 ? M : 0;
                dz += dz < 0 ? M : 0;
                pass = !((dx > 2 && dx < M - 2) || (dy > 2 && dy < M - 2) || (dz > 2 && dz < M - 2));
            }
            const unsigned long long m = __ballot(pass);
            if (pass) q[(qh + qn + before_me(m)) & (kDenseQ - 1)] = (i << 16) | jb;
            qn += __popcll(m);
            if (qn >= kW) drain();
        }
    }
    while (qn > 0) drain();
    wg_sync(nw);  // every bead's list place is written
    int mx = 0, status = 0;
    for (int i = wave + nr * lane; wave < nr && i < N; i += nr * kW) {
        const int2 n2 = cnt[i];
        gs1(S.nup + (i), min(n2.x, cap));
        gs1(S.ndn + (i), min(n2.y, cap));
        const int2 fp = gl2(S.cfp + (i));
        gs2(S.cfp + (i), make_int2(fp.x, fp.y | (min(n2.x, cap) << 16)));
        if (n2.x > cap || n2.y > cap) status = kErrListCapacity;
        mx = max(mx, max(n2.x, n2.y));
    }
    PH_END(S, kPhLSearch, trl);
    status = wave_status(status);
    if (status && !c.status) c.status = status;
    mx = wave_imax(mx);
    if (lane == 0) atomicMax(&S.st->max_nb_seen, (long long)mx);
    wg_sync(nw);
}

// events.f:19-103 for bead i at false time 0: its first event before `limit`
// over its up row and upper shoulder partners
__device__ inline void bead_event(const SysDev& S, const DevTables& T, int i, double limit, double& ti, int& pi, int& ci,
                                  int& status) {
    const int cap = S.cap;
    const Rec bi = gld(S.rec + (i));
    const double2 bwi = gld(S.bw + (i));
    ti = limit;
    pi = ci = -1;
    // the next partner's loads are in flight while one is predicted
    const int n = gl1(S.nup + (i));
    const int* const row = S.nb_up + (size_t)i * cap;
    int ent = n > 0 ? gl1(row) : 0, ent1 = n > 1 ? gl1(row + 1) : 0;
    Rec bm1 = bi;
    int4 om1 = make_int4(-1, -1, -1, -1);
    if (n > 0) {
        bm1 = gld(S.rec + (ent & 0xFFFF));
        om1 = gld(S.ovr + (ent & 0xFFFF));
    }
    for (int k = 0; k < n; ++k) {
        const Rec bm = bm1;
        const int4 om = om1;
        const int m = ent & 0xFFFF, stat = ent >> 24;
        ent = ent1;
        if (k + 1 < n) {
            bm1 = gld(S.rec + (ent & 0xFFFF));
            om1 = gld(S.ovr + (ent & 0xFFFF));
        }
        if (k + 2 < n) ent1 = gl1(row + (k + 2));
        const int code = dyn_code(om, i, stat);
        double tij = 1000000000.0;
        int ty = 0;
        predict(T, code, bi, bm, dyn_bptnr(bi.dyn) == m, bwi, 0.0, tij, ty);
        if (ty == -99) status = kErrBadCode;
        if (tij < ti) {
            ti = tij;
            pi = m;
            ci = ty;
        }
        if (tij < 0.0 && fabs(tij) > 1.0e-10) status = kErrNegativeTime;
    }
    const int4 e = gld(S.extra + (i));
    for (int k = 0; k < 3; ++k) {
        const int m = k == 0 ? e.x : (k == 1 ? e.y : e.z);
        if (m > i) {
            const Rec bm = gld(S.rec + (m));
            const int code = dyn_code(gld(S.ovr + (m)), i, static_t(T, bm.topo, bi.topo));
            double tij = 1000000000.0;
            int ty = 0;
            // events.f:79-83: code 1 -> core, anything else -> shoulder
            predict(T, code == 1 ? 1 : 40, bi, bm, dyn_bptnr(bi.dyn) == m, bwi, 0.0, tij, ty);
            if (tij < 0.0 && fabs(tij) > 1.0e-10) status = kErrNegativeTime;
            if (tij < ti) {
                pi = m;
                ci = ty;
                ti = tij;
            }
        }
    }
}
// events.f:11-127 with tfalse = 0: every bead's next event, then the
// calendar (the pseudo-events' entries from Batch::pseudo); all wavefronts of the system take part (the master scalars'
// scan position is at bin 1 already)
__device__ void events_all(const SysDev&, const DevTables&, const Lds&, Sc&) {
    const Lds& L = ldsv();

    const SysDev& S = sdev();

    const DevTables& T = tabs();
    Sc& c = *L.msc();

    const int tid = (int)threadIdx.x, nthr = kW * L.nw;
    const int N = S.N;
    int status = 0;
    for (int i0; (i0 = next_share(2, kW)) < N;) {
        const int i = i0 + lane_id();
        if (i >= N) break;
        double ti;
        int pi, ci;
        bead_event(S, T, i, c.interval_max + kLt, ti, pi, ci, status);
        Leaf lf;
        lf.tim = ti;
        lf.nptnr = pi;
        lf.meta = make_meta(calc_bin(c, ti, false, status), ci);
        leaf_st(L, i, lf);
        stamp_set(i, mk_stamp(c.coll, i + 1));  // events.f:111-122 adds in index order
    }
    for (int e = N + tid; e < N + 3; e += nthr) {
        Leaf lf = L.batch()->pseudo[e - N];
        lf.meta = make_meta(calc_bin(c, lf.tim, false, status), -2);
        leaf_st(L, e, lf);
        stamp_set(e, mk_stamp(c.coll, e + 1));
    }
    status = wave_status(status);
    if (status && !c.status) c.status = status;
    wg_sync(L.nw);
}

// Rows in nbor.f's order: every bead's up and down rows sorted by
// nbor_key, so that the lowest list position among partners tied in time
// is the one eventredo_up.f's strict < takes in nbor.f's row, and down
// rows are walked in partial_events.f's order.  One lane per row (row r:
// bead r / 2, its up row for even r, its down row for odd r): the row in
// registers (up to five 16-byte loads), its partners' cells and places in one
// round of loads, every entry written at its rank, the count of lower keys.
// The loops run to the longest row of the wavefront's 64.  A row of more than
// kSortMax entries is sorted by the whole wavefront, one lane per entry.
// Down-row entries take their bead's up-row length on the way (bits 16-22).
constexpr int kSortMax = 20;
__device__ inline void sort_rows(const SysDev& S, const DevTables& T, int r0) {
    const int lane = lane_id(), N = S.N, cap = S.cap, M = S.M;
    const bool vec = (cap & 3) == 0;  // rows of whole int4s (row bases are 16-byte aligned)
    const int r = r0 + lane;
    const bool act = r < 2 * N;
    const int x = act ? r >> 1 : 0;
    const bool dnr = (r & 1) != 0;
    int* const row = (dnr ? S.nb_dn : S.nb_up) + (size_t)x * cap;
    const int n = act ? min(gl1((dnr ? S.ndn : S.nup) + (x)), cap) : 0;
    const int2 cx = gl2(S.cfp + (x));
    const unsigned lx = fine_lin(cx.x, M + 4);
    const int ns = n <= kSortMax ? n : 0;
    const int nmax = wave_imax(ns);
    int e[kSortMax];
#pragma unroll
    for (int u = 0; u < kSortMax / 4; ++u) {
        e[4 * u] = e[4 * u + 1] = e[4 * u + 2] = e[4 * u + 3] = 0;
        if (4 * u < ns) {
            if (vec) {
                // reads up to the next multiple of 4 (<= kSortMax, <= cap)
                const int4 v = gld(reinterpret_cast<const int4*>(row) + u);
                e[4 * u] = v.x;
                e[4 * u + 1] = v.y;
                e[4 * u + 2] = v.z;
                e[4 * u + 3] = v.w;
            } else {
#pragma unroll
                for (int w = 0; w < 4; ++w)
                    if (4 * u + w < ns) e[4 * u + w] = gl1(row + (4 * u + w));
            }
        }
    }
    int2 cb[kSortMax];
#pragma unroll
    for (int u = 0; u < kSortMax; ++u) {
        cb[u] = make_int2(0, 0);
        if (u < ns) cb[u] = gl2(S.cfp + (e[u] & 0xFFFF));
    }
    unsigned long long key[kSortMax];
#pragma unroll
    for (int u = 0; u < kSortMax; ++u) {
        key[u] = ~0ull;
        if (u < nmax) {
            const unsigned long long k = nbor_key(M, T, cx, lx, cb[u]);
            key[u] = u < ns ? k : ~0ull;
        }
    }
#pragma unroll
    for (int u = 0; u < kSortMax; ++u) {
        if (u < nmax) {
            int rk = 0;
#pragma unroll
            for (int m = 0; m < 8; ++m) rk += key[m] < key[u] ? 1 : 0;
            if (nmax > 8) {
#pragma unroll
                for (int m = 8; m < 12; ++m) rk += key[m] < key[u] ? 1 : 0;
            }
            if (nmax > 12) {
#pragma unroll
                for (int m = 12; m < kSortMax; ++m) rk += key[m] < key[u] ? 1 : 0;
            }
            const int len = dnr ? cb[u].y >> 16 << 16 : 0;
            if (u < ns) gs1(row + (rk), (int)((unsigned)e[u] & 0xFF00FFFFu) | len);
        }
    }
    // rows longer than that: the wavefront sorts each in turn
    unsigned long long big = __ballot(n > kSortMax);
    while (big) {
        const int src = __ffsll((long long)big) - 1;
        big &= big - 1;
        const int rb_ = r0 + src, xb = rb_ >> 1, nbig = __shfl(n, src, kW);
        int* const rb = ((rb_ & 1) == 0 ? S.nb_up : S.nb_dn) + (size_t)xb * cap;
        const int2 cxb = gl2(S.cfp + (xb));
        int e1 = lane < nbig ? gl1(rb + (lane)) : 0;
        const int2 ce = gl2(S.cfp + (e1 & 0xFFFF));
        const unsigned long long kk = lane < nbig ? nbor_key(M, T, cxb, fine_lin(cxb.x, M + 4), ce) : ~0ull;
        if ((rb_ & 1) != 0) e1 |= (ce.y >> 16) << 16;
        int rk = 0;
        for (int m = 0; m < nbig; ++m) rk += readlane_u64(kk, m) < kk ? 1 : 0;
        wave_sync_mem();  // every lane has read its entry before any is written
        if (lane < nbig) gs1(rb + (rk), e1);
        wave_sync_mem();
    }
}
__device__ inline void sort_all_rows(const SysDev& S, const DevTables& T, int nw) {
    for (int r0; (r0 = next_share(1, kW)) < 2 * S.N;) sort_rows(S, T, r0);
    wg_sync(nw);
}

// Wrap and lists; all wavefronts of the system take part.
__device__ void wrap_and_lists(const SysDev&, const Lds&, Sc&) {
    const Lds& L = ldsv();

    const SysDev& S = sdev();

    Sc& c = *L.msc();

    const int tid = (int)threadIdx.x, nthr = kW * L.nw;
    if (tid == 0) c.nbin = 1;
    if (tid < 3) L.batch()->share[tid] = 0;
    if (tid < 3) L.batch()->pseudo[tid] = leaf_ld(L, S.N + tid);
    for (int k = tid; k < S.N; k += nthr) {
        Rec b = gld(S.rec + (k));
        b.x = b.x - round(b.x);
        b.y = b.y - round(b.y);
        b.z = b.z - round(b.z);
        gst(S.rec + (k), b);
        gst(S.old_r + (k), make_double4(b.x, b.y, b.z, 0.0));
    }
    wg_sync(L.nw);
    if (S.N <= kDenseN)
        rebuild_lists_dense(S, L, c);
    else
        rebuild_lists(S, L, c);
    sort_all_rows(S, tabs(), L.nw);
}

// Wrap, lists and full reschedule; all wavefronts of the system take part.
__device__ void rebuild(const SysDev&, const DevTables&, const Lds&, Sc&) {
    const Lds& L = ldsv();
    const SysDev& S = sdev();
    const DevTables& T = tabs();
    Sc& c = *L.msc();
    PH_BEGIN(trb);
    wrap_and_lists(S, L, c);
    PH_END(S, kPhLists, trb);
    events_all(S, T, L, c);
    // the scratch lay over the round's footprint marks too
    const int nm = (int)min((unsigned)S.N, L.mark_mask) + 1;
    for (int b = (int)threadIdx.x; b < nm; b += kW * L.nw) lds_words(L.o_mark)[b] = 0u;
    PH_END(S, kPhEvents, trb);
    PH_COUNT(S, kPhNRebuild);
}

// sync pseudo-event, main.F90:1126-1187, on all wavefronts of the system:
// sync_move advances the free flight, shifts the calendar and takes the
// displacement test (displ.f); after a barrier sync_decide (one lane) moves
// the time origin and says whether the lists are rebuilt; sync_finish
// (wavefront 0) schedules the next sync.
__device__ inline void sync_move(const Hot& H, const SysDev& S, double tf, int nthr) {
    const int tid = (int)threadIdx.x, N = H.N;
    for (int e = tid; e < N + 3; e += nthr) {
        Leaf lf = leaf_ld(H, e);
        lf.tim = lf.tim - tf;
        leaf_st(H, e, lf);
    }
    double moved_far = 0.0;
#pragma unroll 2
    for (int k = tid; k < N; k += nthr) {
        Rec b = ld_at(H.rec, k);
        const double4 o = gld(S.old_r + (k));
        b.x = b.x + b.vx * tf;
        b.y = b.y + b.vy * tf;
        b.z = b.z + b.vz * tf;
        st_at(H.rec, k, b);
        const double a = o.x - b.x, bb = o.y - b.y, cc = o.z - b.z;
        const double dis = a * a + bb * bb + cc * cc;
        const double moved = dis / S.hdelr;
        if (moved > moved_far) moved_far = moved;
    }
    moved_far = wave_max(moved_far);
    if (lane_id() == 0) atomicMax(&round_rec().moved, (unsigned long long)__double_as_longlong(moved_far));
}
__device__ inline bool sync_decide(const SysDev& S, Sc& c, double tf) {
    const double moved_far = __longlong_as_double((long long)round_rec().moved);
    c.t = c.t + tf;
    c.interval_max = c.interval_max - tf;
    c.tbin_off = c.tbin_off + tf;
    c.tfalse = 0.0;
    bool update = false;
    if (moved_far >= 0.1) {  // displ.f:37-46
        update = true;
        if (moved_far >= 1.25 * 1.25) {
            c.t_fact = c.t_fact / 1.01;
            c.interval = c.t_fact / sqrt(S.setemp);
        }
    }
    if (!(update || c.interval > c.interval_max)) return false;
    if (!update) {
        c.nforced++;
        c.n_forced = c.n_forced * 1.01;
    }
    c.interval_max = c.interval * c.n_forced;
    c.sortsize = c.interval_max / (double)kNumbin;
    c.tbin_off = 0.0;
    c.nupdates++;
    return true;
}
__device__ void sync_finish(const SysDev&, const Lds&, Sc&) {
    const Lds& L = ldsv();

    const SysDev& S = sdev();

    Sc& c = *L.sc();

    const int lane = lane_id();
    const int N = S.N;
    PH_BEGIN(tsy);
    int status = 0;
    const double t2 = c.interval * 0.999;
    if (lane == 0) {
        Leaf lf;
        lf.tim = t2;
        lf.nptnr = -2;
        lf.meta = make_meta(calc_bin(c, t2, true, status), -2);
        leaf_st(L, N + 1, lf);
        stamp_set(N + 1, mk_stamp(c.coll, N + 4));  // after a rebuild's events() adds
    }
    if (status && !c.status) c.status = status;
    wave_sync_mem();
    PH_END(S, kPhSync, tsy);
}

__device__ void output_event(const SysDev&, const Lds&, Sc&) {
    const Lds& L = ldsv();

    const SysDev& S = sdev();

    Sc& c = *L.sc();

    const int lane = lane_id();
    const int N = S.N;
    int status = 0;
    const double t3 = 3.3 / (sqrt(S.setemp)) + 5 + c.tfalse;
    if (lane == 0) {
        Leaf lf;
        lf.tim = t3;
        lf.nptnr = -2;
        lf.meta = make_meta(calc_bin(c, t3, false, status), -2);
        leaf_st(L, N + 2, lf);
        stamp_set(N + 2, mk_stamp(c.coll, 1));
    }
    if (status && !c.status) c.status = status;
    wave_sync_mem();
}

// LDS plan: tables, SysDev, the views, master scalars and round record; each wavefront's one-pass work area, block list
// and pair, wavefront 0's with the multi-pass form's work lists after them;
// then this system's block minima, its footprint marks and, if they fit the
// workgroup's lds_bytes, its calendar leaves: a small system in a launch
// sized for a large one keeps all its leaves in LDS.  Everything from the work areas on is
// also the scratch pool of a list rebuild.  One set of work lists (15 KB)
// instead of one per wavefront (25 KB each) leaves room for eight
// wavefronts at every size: only an event of more than 62 predictions needs
// them, and such an event runs as the first of its round.
__device__ __host__ inline int lds_wave_bytes() {
    return (int)((sizeof(OnePass) + 15) / 16 * 16 + sizeof(int) * kMaxBlist + (sizeof(Pair) + 15) / 16 * 16);
}
__device__ __host__ inline int lds_multi_bytes(int maxw) {
    return (4 * maxw + 15) / 16 * 16 * 3 + (8 * maxw + 15) / 16 * 16 + 64 +
           (int)(sizeof(MinSlot) * (2 + kMaxSpec) + sizeof(SpecInfo) * kMaxSpec + sizeof(DownInfo) * kW);
}
constexpr int kPoolOff = kBatchOff + (int)((sizeof(Batch) + 15) / 16 * 16);
static_assert(sizeof(MinSlot) % 16 == 0 && sizeof(SpecInfo) % 16 == 0 && sizeof(DownInfo) % 16 == 0 &&
                  sizeof(int) * kMaxBlist % 16 == 0,
              "work areas are whole 16-byte units");
__device__ Lds make_lds(const SysDev&, int maxw, int lds_bytes, int ne, int nw, int wave) {
    const SysDev& S = sdev();

    Lds L;
    const int N3 = S.N + 3;
    L.nblk = (N3 + kBlk - 1) / kBlk;
    L.nsup = (L.nblk + kSup - 1) / kSup;
    L.maxw = maxw;
    L.nw = nw;
    L.o_msc = kMscOff;
    L.o_batch = kBatchOff;
    L.o_pool = kPoolOff;
    int p = kPoolOff + wave * lds_wave_bytes();
    auto take = [&](int bytes) {
        const int o = p;
        p = (p + bytes + 15) / 16 * 16;
        return o;
    };
    L.o_one = take((int)sizeof(OnePass));
    L.o_blist = take((int)sizeof(int) * kMaxBlist);
    L.o_pair = take((int)sizeof(Pair));
    p = kPoolOff + (ne + 1) * lds_wave_bytes();
    L.o_wm = take((int)sizeof(int) * maxw);
    L.o_wx = take((int)sizeof(int) * maxw);
    L.o_wy = take((int)sizeof(int) * maxw);
    L.o_wt = take((int)sizeof(double) * maxw);
    L.o_wd = take(64);
    L.o_slot = take((int)sizeof(MinSlot) * (2 + kMaxSpec));
    L.o_spec = take((int)sizeof(SpecInfo) * kMaxSpec);
    L.o_down = take((int)sizeof(DownInfo) * kW);
    L.o_sc = kMscOff;
    L.o_blk = take((int)sizeof(unsigned) * L.nblk);
    // a footprint mark per bead, or as large a power of two as fits
    L.mark_mask = ~0u;
    const int words = (lds_bytes - p) / (int)sizeof(unsigned);
    int nm = S.N + 1;
    if (nm > words) {
        nm = 1024;
        while (2 * nm <= words) nm *= 2;
        L.mark_mask = (unsigned)nm - 1u;
    }
    L.o_mark = take((int)sizeof(unsigned) * nm);
    L.o_leaf = p;
    L.leaf_lds = N3 <= (lds_bytes - p) / (int)sizeof(Leaf);
    L.leaf = S.leaf;
    const int room = (lds_bytes - kPoolOff) / kScratch;
    L.nwr = room < nw ? room : nw;
    return L;
}

__device__ inline void load_sc(const SysState* st, Sc& c) {
    c.tfalse = st->tfalse;
    c.t = st->t;
    c.interval = st->interval;
    c.interval_max = st->interval_max;
    c.t_fact = st->t_fact;
    c.n_forced = st->n_forced;
    c.sortsize = st->sortsize;
    c.tbin_off = st->tbin_off;
    c.old_tfalse = st->old_tfalse;
    c.coll = st->coll;
    c.numghosts = st->numghosts;
    c.nupdates = st->nupdates;
    c.nforced = st->nforced;
    c.target = st->target;
    c.rc0 = st->rng_ctr[0];
    c.rc1 = st->rng_ctr[1];
    c.nbin = st->nbin;
    c.status = st->status;
    for (int k = 0; k < 32; ++k) c.nev[k] = st->nevents[k];
}
__device__ inline void store_sc(SysState* st, const Sc& c) {
    st->tfalse = c.tfalse;
    st->t = c.t;
    st->interval = c.interval;
    st->interval_max = c.interval_max;
    st->t_fact = c.t_fact;
    st->n_forced = c.n_forced;
    st->sortsize = c.sortsize;
    st->tbin_off = c.tbin_off;
    st->old_tfalse = c.old_tfalse;
    st->coll = c.coll;
    st->numghosts = c.numghosts;
    st->nupdates = c.nupdates;
    st->nforced = c.nforced;
    st->target = c.target;
    st->rng_ctr[0] = c.rc0;
    st->rng_ctr[1] = c.rc1;
    st->nbin = c.nbin;
    st->status = c.status;
    for (int k = 0; k < 32; ++k) st->nevents[k] = c.nev[k];
}
__device__ void copy_tables(const DevTables* src, DevTables* dst) {
    const double* s = (const double*)src;
    double* d = (double*)dst;
    const int n = (int)(sizeof(DevTables) / sizeof(double));
    for (int k = (int)threadIdx.x; k < n; k += (int)blockDim.x) d[k] = s[k];
}

}  // namespace

// ------------------------------------------------------------------------
// kernels
// ------------------------------------------------------------------------
// ---- start-up (main.F90:205-424 after the host-side H-bond restore) and a
// list update forced at the current time (pdmd_rebuild: the sync
// pseudo-event's shift of the time origin and its update branch,
// main.F90:1126-1187, without displacement test, rate adaptation or new sync
// entry): each step is one launch over the whole GPU, blockIdx.y the system.
// As a single workgroup per system the steps of 23 424 beads took 8.6 ms on
// one of 256 compute units, at 512 beads 205 us; the launches cost a few
// microseconds each, so small systems gain too.
constexpr int kGridT = 256;
constexpr int kStatsT = 1024;
__device__ inline void report(const SysDev& S, int status) {
    status = wave_status(status);
    if (status && lane_id() == 0) atomicCAS(&S.st->status, 0, status);  // the first error stays
}
// Beads to the new time origin (forced: advanced by the free flight) and
// into the box, and their cells (a launch of their own is 4 us more); the pseudo-events' entries seeded, or shifted.
__global__ __launch_bounds__(kGridT) void k_list_beads(const SysDev* __restrict__ sys, const int* ids, int forced) {
    const SysDev& S = sys[ids[blockIdx.y]];
    const int gid = (int)(blockIdx.x * kGridT + threadIdx.x), N = S.N;
    const double tf = forced ? S.st->tfalse : 0.0;
    if (gid < N) {
        Rec b = gld(S.rec + (gid));
        if (forced) {
            b.x = b.x + b.vx * tf;
            b.y = b.y + b.vy * tf;
            b.z = b.z + b.vz * tf;
        }
        b.x = b.x - round(b.x);
        b.y = b.y - round(b.y);
        b.z = b.z - round(b.z);
        gst(S.rec + (gid), b);
        gst(S.old_r + (gid), make_double4(b.x, b.y, b.z, 0.0));
        list_cell(S, S.M / S.cq, gid, b);
    } else if (gid < N + 3) {
        Leaf g;
        if (forced) {
            g = gld(S.leaf + (gid));
            g.tim = g.tim - tf;
        } else {
            if (gid == N) {
                g.tim = 1000000000.0;
                if (S.canon) {
                    double tgho = 0.0;
                    int guard = 0;
                    unsigned long long rc = S.st->rng_ctr[0];
                    do {
                        tgho = rng_u01(S.seed, 0, rc++);
                    } while ((tgho < 1.e-18 || tgho == 1.0) && ++guard < 1000);
                    S.st->rng_ctr[0] = rc;
                    g.tim = -1.0 * dlog(tgho) * S.avegtime * .0000001;
                }
            } else
                g.tim = gid == N + 1 ? S.st->interval : 3.3 / (sqrt(S.setemp)) + 5;
            g.nptnr = -2;
            g.meta = make_meta(-1, -2);
        }
        gst(S.leaf + (gid), g);
    }
}
// the cells' starts (one workgroup per system); the scalars of a forced update
constexpr int kScanT = 1024;
__global__ __launch_bounds__(kScanT) void k_list_scan(const SysDev* __restrict__ sys, const int* ids, int forced) {
    __shared__ int part[kScanT / kW];
    const SysDev& S = sys[ids[blockIdx.y]];
    if (threadIdx.x == 0) {
        SysState& st = *S.st;
        st.nbin = 1;
        if (forced) {
            st.t = st.t + st.tfalse;
            st.tfalse = 0.0;
            st.interval_max = st.interval * st.n_forced;
            st.sortsize = st.interval_max / (double)kNumbin;
            st.tbin_off = 0.0;
            st.nupdates++;
        }
    }
    const int Mq = S.M / S.cq;
    list_scan(S.ccnt, S.cstart, Mq * Mq * Mq, part, wave_id(), kScanT / kW);
}
__global__ __launch_bounds__(kGridT) void k_list_copy(const SysDev* __restrict__ sys, const int* ids) {
    list_copy(sys[ids[blockIdx.y]], (int)(blockIdx.x * kGridT + threadIdx.x), (int)(gridDim.x * kGridT));
}
// the tables in LDS
__device__ inline const DevTables& block_tables(const SysDev& S) {
    __shared__ __attribute__((aligned(16))) unsigned char mem[sizeof(DevTables)];
    DevTables& T = *reinterpret_cast<DevTables*>(mem);
    copy_tables(S.tab, &T);
    __syncthreads();
    return T;
}
__global__ __launch_bounds__(kGridT) void k_list_search(const SysDev* __restrict__ sys, const int* ids) {
    const SysDev& S = sys[ids[blockIdx.y]];
    constexpr int kPlaces = kCells * (kGridT / kW);  // of a workgroup
    if ((int)(blockIdx.x * kPlaces) >= S.N) return;
    const DevTables& T = block_tables(S);
    __shared__ SearchLds W[kGridT / kW];
    const int i0 = (int)(blockIdx.x * kPlaces) + wave_id() * kCells;
    int mx = 0, status = 0;
    if (i0 < S.N) list_search(S, T, i0, W[wave_id()], mx, status);
    report(S, status);
    mx = wave_imax(mx);
    if (lane_id() == 0) atomicMax(&S.st->max_nb_seen, (long long)mx);
}
__global__ __launch_bounds__(kGridT) void k_list_sort(const SysDev* __restrict__ sys, const int* ids) {
    const SysDev& S = sys[ids[blockIdx.y]];
    if ((int)(blockIdx.x * kGridT) >= 2 * S.N) return;
    const DevTables& T = block_tables(S);
    const int r0 = (int)(blockIdx.x * kGridT) + wave_id() * kW;
    if (r0 < 2 * S.N) sort_rows(S, T, r0);
}
// events() over the new lists (events.f), and the pseudo-events' bins
__global__ __launch_bounds__(kGridT) void k_list_events(const SysDev* __restrict__ sys, const int* ids) {
    const SysDev& S = sys[ids[blockIdx.y]];
    if ((int)(blockIdx.x * kGridT) >= S.N + 3) return;
    const DevTables& T = block_tables(S);
    const int i = (int)(blockIdx.x * kGridT + threadIdx.x), N = S.N;
    const SysState& st = *S.st;
    const double imax = st.interval_max;
    int status = 0;
    if (i < N + 3) {
        Leaf lf;
        int ci = -2;
        if (i < N)
            bead_event(S, T, i, imax + kLt, lf.tim, lf.nptnr, ci, status);
        else
            lf = gld(S.leaf + (i));
        lf.meta = make_meta(bin_of(imax, st.tbin_off, st.sortsize, 1, lf.tim, status), ci);
        gst(S.leaf + (i), lf);
        gs1(S.stamp + (i), mk_stamp(st.coll, i + 1));  // events.f:111-122 adds in index order
    }
    report(S, status);
}

// Takes up to kmax entries from the pool in key order (wavefront 0): the
// tree's candidates, the new entries of the last round's committed events
// and its popped entries that were not committed (B.key[A] to B.key[Kp - 1]).
// An entry whose key is no longer its leaf's was rewritten meanwhile and is
// dropped.  Pair events only after the first, since a pseudo-event runs
// alone; a ghost event may lead a round (its draws come first in the serial
// order).  Returns the number taken, 0 if the pool is empty.
//
// Every lane counts the proxies below its own, so one sweep over the
// entries (about a dozen, four per LDS access in flight) orders all of them; popping a round's entries one
// by one from a tree of minima took 2 200 cycles each.
__device__ __forceinline__ int select_pool(const Hot& H, int kmax, int A, int Kp, int ne, int fsh) {
    Batch& B = round_rec();
    const int lane = lane_id(), N = H.N;
    Key k = empty_key();
    bool have = false;
    const int f = lane - kCandMax, q = A + lane - (kCandMax + kFreshMax);
    if (lane < kCandMax) {
        have = lane < B.ncand;
        k = B.cand[lane];
    } else if (f < kFreshMax) {
        const int w = f >> fsh;
        have = w < ne && (f & ((1 << fsh) - 1)) < B.nfresh[min(w, kMaxWaves - 1)];
        k = B.fresh[f];
    } else {
        have = q < Kp;
        k = B.key[min(q, kMaxWaves - 1)];
    }
    const int idx = key_idx(k);
    const double pk = key_proxy(k);
    have = have && pk < B.edge;
    if (have) {
        const Key now = leaf_key(leaf_ld(H, idx), idx);
        have = now.t == k.t && now.bc == k.bc && now.ip == k.ip;
    }
    // The proxies side by side in LDS, every lane counts those below its own.
    // (An entry rewritten with an equal key stands in fresh and elsewhere: it
    // shows as a shared proxy.)
    unsigned long long vm = __ballot(have);
    int n = __popcll(vm);
    if (n == 0) return 0;
    double* const px = reinterpret_cast<double*>(smem + H.o_w);
    if (have) px[before_me(vm)] = pk;
    if (lane >= n) px[lane] = __hiloint2double(kInfHi, 0);
    wave_sync();
    int rank = 0;
    for (int q0 = 0; q0 < n; q0 += 4) {
        const double a = px[q0], b = px[q0 + 1], c = px[q0 + 2], d = px[q0 + 3];
        rank += (a < pk ? 1 : 0) + (b < pk ? 1 : 0) + (c < pk ? 1 : 0) + (d < pk ? 1 : 0);
    }
    const int last = kmax < kMaxWaves ? kmax : kMaxWaves - 1;
    if (have && rank <= last) B.order[rank] = lane;
    wave_sync();
    if (__ballot(have && rank <= last && B.order[rank] != lane)) {
        // shared proxies: one of each entry, in the exact order
        const bool isf = lane >= kCandMax && lane < kCandMax + kFreshMax;
        unsigned long long fm = __ballot(have && isf);
        while (fm) {
            const int s = __ffsll((long long)fm) - 1;
            fm &= fm - 1;
            if (idx == __builtin_amdgcn_readlane(idx, s) && lane != s) have = have && isf && lane < s;
        }
        vm = __ballot(have);
        n = __popcll(vm);
        rank = 0;
        unsigned long long sm = vm;
        while (sm) {
            const int s = __ffsll((long long)sm) - 1;
            sm &= sm - 1;
            rank += s != lane && key_less(readlane_key(k, s), k) ? 1 : 0;
        }
    }
    int K = min(kmax, n);
    unsigned long long special = __ballot(have && idx >= N);
    while (special) {
        const int s = __ffsll((long long)special) - 1;
        special &= special - 1;
        const int r = __builtin_amdgcn_readlane(rank, s), e = __builtin_amdgcn_readlane(idx, s);
        if (r > 0)
            K = min(K, r);
        else if (e > N)
            K = 1;
    }
    if (have && rank < K) B.key[rank] = k;
    wave_sync();
    return K;
}

// The round's entries (wavefront 0): from the pool, after collecting it
// again where it is incomplete or empty; the least entry of the calendar
// alone where no edge gives a pool (many entries of one time).  The master takes
// the first event's bin, time and number.  Returns 0 for an empty calendar.
__device__ __forceinline__ int select_round(const Hot& H, Sc& c, int kmax, int A, int Kp, int ne, int fsh, int want, int par) {
    PH_BEGIN(tsp);
    Batch& B = round_rec();
    const int lane = lane_id();
    int K = 0;
    for (int att = 0; att < 2; ++att) {
        if (att == 1 || !uni(B.full)) K = select_pool(H, kmax, A, Kp, ne, fsh);
        if (K > 0 || att == 1) break;
        PH_END(sdev(), kPhSelPop, tsp);
        int* const list = reinterpret_cast<int*>(smem + H.o_w);
        tree_update(H, par, list);
        collect_pool(H, 0, uni(c.tfalse), want, 24, list, false);
        if (lane < kMaxWaves) B.nfresh[lane] = 0;
        if (lane == 0) B.full = 0;
        wave_sync();
        A = Kp = 0;
        PH_END(sdev(), kPhSelCopy, tsp);
    }
    PH_END(sdev(), kPhSelPop, tsp);
    if (K == 0) {
        Key least = empty_key();
        for (int idx = lane; idx < H.N + 3; idx += kW) {
            const Key q = leaf_key(leaf_ld(H, idx), idx);
            if (q.bc != kEmptyBc && (least.bc == kEmptyBc || key_less(q, least))) least = q;
        }
        const Key k = key_min_wave(least);
        if (k.bc == kEmptyBc) {
            c.status = kErrBin;
            return 0;
        }
        if (lane == 0) B.key[0] = k;
        wave_sync();
        K = 1;
    }
    if (lane == 0) {
        const Key k0 = B.key[0];
        c.old_tfalse = c.tfalse;
        c.nbin = key_bin(k0);
        c.tfalse = k0.t;
        c.coll++;
    }
    wave_sync();
    return K;
}

__device__ inline void log_event(const SysDev& S, int& log_count, long long coll, int e, int jj, int ty, double t) {
    if (S.log && log_count < S.log_cap) {
        if (lane_id() == 0) {
            LogRec r;
            r.coll = coll;
            r.i = e + 1;
            r.j = jj + 1;
            r.type = ty;
            r.pad = 0;
            r.t = t;
            gst(S.log + (log_count), r);
        }
        ++log_count;
    }
}

// The event loop: each workgroup commits events of its system until the
// system's coll counter has advanced by inc[k].  With one event wavefront
// each round is one event.  With W of them a round takes up to
// W entries; pair events run side by side, one per wavefront, and the
// round commits the prefix of them that the serial order would have run
// the same way (disjoint footprints, no new entry ahead of a later one).
// A wall-clock budget (ticks of wall_clock64, 0 = none) stops a system early
// between rounds, so that one launch over systems of uneven speed ends
// evenly; flags & kStopAtOutput stops it right after its next output
// pseudo-event (where the reference writes observables and configurations).
// The registers (256 per lane) allow eight wavefronts on a compute unit.  A
// calendar wavefront that prepares the next selection while the events run,
// instead of wavefront 0 after them: 8000 entries of 6144 beads 33.2 -> 27.5
// ms at the step that brought it in; the whole loop 62.3 ms then, 14.3 now.
__global__ __launch_bounds__(64 * kMaxWaves) void k_run(const SysDev* __restrict__ sys, const int* ids, const long long* inc,
                                                       int maxw, int lds_bytes, int ne, long long budget, int flags,
                                                       unsigned long long* launch_t0) {
    // event wavefronts 0 to ne - 1, then the calendar wavefront; any others
    // only take part where all do (list updates, free flight)
    const int nw = (int)(blockDim.x >> 6), wave = wave_id(), lane = lane_id();
    if (threadIdx.x == 0) *reinterpret_cast<SysDev*>(smem + kSdOff) = sys[ids[blockIdx.x]];
    __syncthreads();
    const SysDev& S = sdev();
    if (lane == 0)
        *reinterpret_cast<Lds*>(smem + kLdOff + wave * kLdStride) = make_lds(S, maxw, lds_bytes, ne, nw, wave);
    __syncthreads();
    const Lds& L = ldsv();
    const int N = S.N, N3 = N + 3;
    copy_tables(S.tab, const_cast<DevTables*>(&tabs()));
    if (L.leaf_lds)
        for (int e = (int)threadIdx.x; e < N3; e += (int)blockDim.x) L.lleaf()[e] = gld(S.leaf + (e));
    for (int b = (int)threadIdx.x, nm = (int)min((unsigned)N, L.mark_mask) + 1; b < nm; b += (int)blockDim.x)
        lds_words(L.o_mark)[b] = 0u;
    __syncthreads();
    const DevTables& T = tabs();
    Sc& c = *L.sc();  // the master scalars
    Batch& B = *L.batch();
    if (threadIdx.x == 0) {
        load_sc(S.st, c);
        c.target = c.coll + inc[blockIdx.x];
    }
    __syncthreads();
    const Hot H = load_hot(S, L);
    const Gather G = load_gather(S);
    rescan_all(H, wave, nw);
    int log_count = S.st->log_count;
    // the budget runs from the launch's start: the earliest start among the
    // workgroups (launch_t0 is reset to all ones before a budgeted launch),
    // so that a workgroup dispatched late does not get a later deadline
    long long w0 = wall_clock64();
    const long long t_begin = w0;
    long long t_rebuild = 0, n_rebuild = 0;
    // the system's own limit on pair events per round (its tuned wavefronts)
    const int kcap = S.waves_cap > 0 && S.waves_cap < ne ? S.waves_cap : ne;
    if (budget > 0) {
        if (threadIdx.x == 0) {
            atomicMin(launch_t0, (unsigned long long)w0);
            B.t0 = (long long)__hip_atomic_load(launch_t0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        w0 = B.t0;
    }
    bool stop_out = false;
    // the pool holds a few entries more than a round takes; each event
    // wavefront has an equal share of the fresh entries' places
    const int want = kcap + 2, fsh = ne <= 1 ? 5 : (ne <= 2 ? 4 : (ne <= 4 ? 3 : 2));
    int par = 0, A = 0, Kp = 0;
    if (threadIdx.x < kSup) B.dirty[0][threadIdx.x] = B.dirty[1][threadIdx.x] = 0;
    if (threadIdx.x == 0) {
        B.full = 1;
        B.width = c.interval / 64.0;
    }
    __syncthreads();
    while (true) {
        if (wave == 0) {
            PH_BEGIN(tsel);
            int K = 0;
            if (uni(c.status) == 0 && !stop_out && !(budget > 0 && wall_clock64() - w0 > budget)) {
                const long long left = c.target - c.coll;
                const int room = uni((int)min((long long)kcap, left));
                if (room > 0) K = select_round(H, c, room, A, Kp, ne, fsh, want, par ^ 1);
            }
            if (lane == 0) {
                B.K = K;
                B.cut = K;
            }
            PH_END(S, kPhSelect, tsel);
        }
        __syncthreads();
        const int K = uni(B.K);
        if (K == 0) break;
        const Key k = B.key[wave < K ? wave : 0];
        const int e = uni(key_idx(k));
        int* const list = reinterpret_cast<int*>(smem + H.o_w);
        if (K == 1 && e > N) {
            // the sync or output event; the pool is collected again after it
            if (wave == ne) tree_update(H, par ^ 1, list);
            const double tf = uni(master().tfalse);
            if (threadIdx.x == 0) B.moved = 0;
            __syncthreads();
            if (e == N + 1) {
                PH_BEGIN(tsy);
                PH_COUNT(S, kPhNSync);
                sync_move(H, S, tf, kW * nw);
                __syncthreads();
                if (threadIdx.x == 0) B.rebuild = sync_decide(S, c, tf) ? 1 : 0;
                __syncthreads();
                PH_END(S, kPhSync, tsy);
                if (B.rebuild) {
                    const long long tr = wall_clock64();
                    rebuild(S, T, L, c);
                    t_rebuild += wall_clock64() - tr;
                    ++n_rebuild;
                    __syncthreads();
                }
                // every entry moved
                rescan_all(H, wave, nw);
                if (wave == 0) sync_finish(S, L, c);
            } else if (wave == 0) {
                output_event(S, L, c);
                stop_out = (flags & kStopAtOutput) != 0;
            }
            if (wave == 0) {
                log_event(S, log_count, c.coll, e, -1, 0, k.t);
                if (lane == 0) {
                    dirty_or(par ^ 1, e / kBlk);
                    B.full = 1;
                }
            }
            A = Kp = 0;
            __syncthreads();
            continue;
        }
        A = 0;
        Kp = K;
        if (wave == ne) {
            // the calendar wavefront: the minima after the last round's
            // events, then the pool the next round is taken from, while
            // this round's events run
            tree_update(H, par ^ 1, list);
            collect_pool(H, K, uni(B.key[K - 1].t), want, 2, list, K > 1);
            __syncthreads();
        } else {
            if (lane == 0 && wave < ne) B.nfresh[wave] = 0;
            if (wave < K) {
                // pair events (a ghost event may lead them), one per
                // wavefront; event k of a round is numbered and stamped as
                // the master will count it
                A = run_event(H, G, e, uni(key_p(k)), uni(key_ct(k)), k.t, uni(key_bin(k)), master().coll + wave, wave, K, par, fsh);
                if (A > 0 && lane == 0) {
                    const int ty = B.ty[wave];
                    if (ty >= 1 && ty <= 30)
                        __hip_atomic_fetch_add((unsigned long long*)&master().nev[ty], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            } else {
                int nb = 0;
                bar_to(nb, K > 1 ? kRoundBars : 1);
            }
        }
        par ^= 1;
        PH_BEGIN(ttail);
        if (wave == 0 && K > 1) {
            PH_COUNT(S, kPhNRound);
            PH_ADDN(S, kPhNPopped, K);
            PH_ADDN(S, kPhNCommit, A);
            PH_ADDN(S, kPhNCutMark, min(K, B.cut) < K ? 1 : 0);
            PH_ADDN(S, kPhNCutKey, A < min(K, B.cut) ? 1 : 0);
        }
        __syncthreads();
        if (wave == 0) {
            // the master takes the committed events in order
            if (S.log)
                for (int q = 0; q < A; ++q) {
                    const Key kk = B.key[q];
                    log_event(S, log_count, c.coll + q, key_idx(kk), key_idx(kk) == N ? B.gbead : key_p(kk), B.ty[q], kk.t);
                }
            {
                const int q = lane & (kMaxWaves - 1);
                int st = q > 0 ? B.st[q] : 0;
                st = st != 0 ? st : B.st_rep[q];
                st = wave_status(lane < A ? st : 0);
                if (st != 0 && lane == 0 && c.status == 0) c.status = st;
            }
            if (A >= 2 && lane == 0) {
                const Key kp = B.key[A - 2], kk = B.key[A - 1];
                c.coll += A - 1;
                c.old_tfalse = kp.t;
                c.tfalse = kk.t;
                c.nbin = key_bin(kk);
            }
            wave_sync();
        }
        PH_END(S, kPhBTail, ttail);
    }
    __syncthreads();
    if (L.leaf_lds)
        for (int e2 = (int)threadIdx.x; e2 < N3; e2 += (int)blockDim.x) gst(S.leaf + (e2), L.lleaf()[e2]);
    if (threadIdx.x == 0) {
        S.st->log_count = log_count;
        store_sc(S.st, c);
        S.st->run_ticks += wall_clock64() - t_begin;
        S.st->rebuild_ticks += t_rebuild;
        S.st->rebuilds += n_rebuild;
    }
}

// ------------------------------------------------------------------------
// debug checks of one system's state (one lane per bead i)
// ------------------------------------------------------------------------
// repuls_check.f:16-81 on a state array (n = the N bead, cb = the C bead);
// 11 when a shoulder bead falls outside the system
__device__ double check_rating(const DevTables& T, const Rec* rec, int N, int n, int cb, double tf) {
    const Rec rn = rec[n], rc = rec[cb];
    int ncim1, ncai, ncaj, nnjp1;
    shoulder_idx(n, topo_len(rn.topo), cb, topo_len(rc.topo), ncim1, ncai, ncaj, nnjp1);
    if (ncim1 < 0 || ncim1 >= N || ncai < 0 || ncai >= N || ncaj < 0 || ncaj >= N || nnjp1 < 0 || nnjp1 >= N)
        return 11.0;
    const double d1 = dist_rec(rn, rec[ncaj], tf), d2 = dist_rec(rn, rec[nnjp1], tf);
    const double d3 = dist_rec(rc, rec[ncai], tf), d4 = dist_rec(rc, rec[ncim1], tf);
    if (d1 > T.shder[1] && d2 > T.shder[2] && d3 > T.shder[3] && d4 > T.shder[4]) return 10.0;
    return 11.0;
}
// out[0..2]: checkover.f:21-131 over all pairs (i < j) at tfalse: cores
// closer than sigma (codes 1 and >= 15, squeezed for 22-26), bonds longer /
// shorter than their window (4-12); out[3]: least i*N + j among them;
// out[4..7]: check_nc_int.f:25-354 over i's listed code-15 partners:
// boundbad, unboundbad, n_ss, m_ss.  alt: positions and velocities to check
// in place of the resident ones (topology and codes stay the system's).
__global__ void k_check(const SysDev* sys, int id, const Rec* alt, unsigned long long* out) {
    const SysDev& S = sys[id];
    const DevTables& T = *S.tab;
    const int N = S.N, cap = S.cap;
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= N) return;
    const Rec* rec = alt ? alt : S.rec;
    const double tf = S.st->tfalse;
    const Rec ri = rec[i];
    const int idi = dyn_ident(ri.dyn);
    unsigned long long over = 0, lng = 0, sht = 0, first = ~0ull;
    for (int j = i + 1; j < N; ++j) {
        const Rec rj = rec[j];
        const int idj = dyn_ident(rj.dyn);
        const int code = dyn_code(S.ovr[j], i, static_t(T, rj.topo, ri.topo));  // ev_code(j, i)
        if (code == 1 || code >= 15) {
            const double pe = T.ev_param[1][code];
            double sigsq = T.sigma_sq[idi][idj] * (pe * pe);
            if (code >= 22 && code <= 26) {
                const double q = T.sqz610[code - 21][idi > idj ? idi : idj];
                sigsq = sigsq * (q * q);
            }
            Geo g;
            geo(ri, rj, tf, g);
            const double r2 = g.r2 * 1.0000000001;
            if (r2 <= sigsq) {
                ++over;
                first = min(first, (unsigned long long)i * (unsigned long long)N + (unsigned long long)j);
            }
        } else if (code >= 4 && code <= 12 && !S.chaptype2) {  // checkover.f:67: chaptype 1 only
            double blmin, blmax;
            bond_window(T, code, S.bw[i], blmin, blmax);
            blmin = blmin * blmin;
            blmax = blmax * blmax;
            Geo g;
            geo(ri, rj, tf, g);
            const bool lo = g.r2 * 1.0000000001 < blmin, hi = g.r2 * 0.9999999999 > blmax;
            if (hi) ++lng;
            if (lo) ++sht;
            if (lo || hi) first = min(first, (unsigned long long)i * (unsigned long long)N + (unsigned long long)j);
        }
    }
    unsigned long long bb = 0, ub = 0, nss = 0, mss = 0;
    const int nu = S.nup[i];
    const int4 xi = S.extra[i];
    for (int k = 0; k < nu && k < cap; ++k) {
        const int ent = S.nb_up[(size_t)i * cap + k];
        const int j = ent & 0xFFFFFF;
        if (j < 0 || j >= N) continue;
        const Rec rj = rec[j];
        const int idj = dyn_ident(rj.dyn);
        if (dyn_code(S.ovr[j], i, ent >> 24) != 15) continue;
        const bool term = terminal_t(ri.topo) || terminal_t(rj.topo);
        if (dyn_bptnr(ri.dyn) == j) {
            const double rating = term ? 10.0 : (idi < idj ? check_rating(T, rec, N, i, j, tf) : check_rating(T, rec, N, j, i, tf));
            if (rating > 10.0) ++bb;
            if (!term && xi.w == j) ++nss;
        } else {
            Geo g;
            geo(ri, rj, tf, g);
            if (g.r2 - T.welldia_sq[idi][idj] < 0.0) {
                const double rating = term ? 11.0 : (idi < idj ? check_rating(T, rec, N, i, j, tf) : check_rating(T, rec, N, j, i, tf));
                if (rating <= 10.0) ++ub;
                if (!term && xi.w == j) ++nss;
            }
        }
        if (xi.w == j) ++mss;
    }
    if (over) atomicAdd(out + 0, over);
    if (lng) atomicAdd(out + 1, lng);
    if (sht) atomicAdd(out + 2, sht);
    if (first != ~0ull) atomicMin(out + 3, first);
    if (bb) atomicAdd(out + 4, bb);
    if (ub) atomicAdd(out + 5, ub);
    if (nss) atomicAdd(out + 6, nss);
    if (mss) atomicAdd(out + 7, mss);
}

// ------------------------------------------------------------------------
// observables of one system: energy.f:25-101, radgyr.f:18-135,
// end2end.f:14-44
// ------------------------------------------------------------------------
// Latency: three launches, sums in a fixed order, k_obs_parts (bead sums, and
// every chain unwrapped), k_obs_chains (chain sums), k_obs_sum.  One workgroup
// per system with a lane per chain walked 128 beads serially through memory:
// 95 us at 6144 beads on one compute unit.  List update, calendars and
// observables of 16 systems of up to 23 424 beads with either (and with the
// reads below): 4.51 ms, 1.49 ms.
constexpr int kObsT = 256;
constexpr int kObsBeads = 64;  // beads per workgroup: a 16-lane row takes a side chain's pairs
constexpr int kObsSums = 6;    // sumvel, ehh_ii, ehh_ij, hb_ii, hb_ij, hb_alpha
// partial sums in the list rebuild's scratch: 48 bytes per 64 beads, then 16
// per chain of at least 16 beads; sinfo has 16 per bead
__device__ inline double* obs_bead_sums(const SysDev& S) { return reinterpret_cast<double*>(S.sinfo); }
__device__ inline double* obs_chain_sums(const SysDev& S) {
    return obs_bead_sums(S) + kObsSums * ((S.N + kObsBeads - 1) / kObsBeads);
}
// sum over the wavefront in a fixed tree, in every lane
__device__ inline double wave_sum(double v) {
    for (int w = kW / 2; w > 0; w >>= 1) v = v + __shfl_xor(v, w);
    return v;
}
// one coordinate's image next to the unwrapped neighbour's (radgyr.f:48-104)
__device__ inline double unwrap(double a, double b) {
    const double dd = a - b;
    return dd > 0.5 ? a - 1.0 : (dd < -0.5 ? a + 1.0 : a);
}
// Workgroups [0, nb): bead sums (kinetic energy, H-bond counts, side-chain
// well energies over the up lists: every side-chain pair inside a well is
// listed, wells lie inside the list cutoff).  The others: a wavefront per
// chain, backbone unwrapped into spos.
__global__ __launch_bounds__(kObsT) void k_obs_parts(const SysDev* __restrict__ sys, int id, int nb, const int* cstart,
                                                     const int* clen, int nch) {
    const SysDev& S = sys[id];
    const int N = S.N, wave = wave_id(), lane = lane_id();
    const double tf = S.st->tfalse;
    if ((int)blockIdx.x >= nb) {
        const int c = ((int)blockIdx.x - nb) * (kObsT / kW) + wave;
        if (c >= nch) return;
        const int s = cstart[c], L = clen[c];
        double4* q = S.spos;
        auto at = [&](int k) {
            const Rec b = S.rec[k];
            return make_double4(b.x + b.vx * tf, b.y + b.vy * tf, b.z + b.vz * tf, 0.0);
        };
        double4 prev = make_double4(0.0, 0.0, 0.0, 0.0);  // the residue before the chunk's
        for (int base = 0; base < L; base += kW) {
            const int r = base + lane, n = min(kW, L - base);
            const double4 zero = make_double4(0.0, 0.0, 0.0, 0.0);
            double4 ca = r < L ? at(s + r) : zero;
            // each Calpha next to the one before it, in order
            for (int u = 0; u < n; ++u) {
                double4 v = make_double4(readlane_d(ca.x, u), readlane_d(ca.y, u), readlane_d(ca.z, u), 0.0);
                if (base + u > 0) v = make_double4(unwrap(v.x, prev.x), unwrap(v.y, prev.y), unwrap(v.z, prev.z), 0.0);
                if (lane == u) ca = v;
                prev = v;
            }
            if (r < L) {
                q[s + r] = ca;
                // N and C next to their Calpha; the side chain as it is: the
                // second species' sums can reach an earlier chain's
                for (int kind = 1; kind < 3; ++kind) {
                    const double4 v = at(s + kind * L + r);
                    q[s + kind * L + r] =
                        make_double4(unwrap(v.x, ca.x), unwrap(v.y, ca.y), unwrap(v.z, ca.z), 0.0);
                }
                q[s + 3 * L + r] = at(s + 3 * L + r);
            }
        }
        return;
    }
    __shared__ double red[kObsT / kW][kObsSums];
    const DevTables& T = *S.tab;
    double sum[kObsSums] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const int first = (int)blockIdx.x * kObsBeads;
    if ((int)threadIdx.x < kObsBeads && first + (int)threadIdx.x < N) {
        const int i = first + (int)threadIdx.x;
        const Rec r = S.rec[i];
        sum[0] = r.bm * (r.vx * r.vx + r.vy * r.vy + r.vz * r.vz);
        const int j = dyn_bptnr(r.dyn);
        if (j > i) {
            const bool same = topo_chain(r.topo) == topo_chain(S.rec[j].topo);
            sum[3] = same ? 1.0 : 0.0;
            sum[4] = same ? 0.0 : 1.0;
        }
        if (topo_kind(r.topo) == 1 && topo_res(r.topo) >= 5 && j == i + topo_len(r.topo) - 4) sum[5] = 1.0;
    }
    constexpr int kRows = kObsT / 16;
    for (int u = 0; u < kObsBeads / kRows; ++u) {
        const int i = first + u * kRows + (int)threadIdx.x / 16;
        if (i >= N) break;
        const Rec r = S.rec[i];
        if (topo_kind(r.topo) != 3) continue;
        const int nu = min(S.nup[i], S.cap), idi = dyn_ident(r.dyn), j = dyn_bptnr(r.dyn);
        for (int k = lane & 15; k < nu; k += 16) {
            const int ent = S.nb_up[(size_t)i * S.cap + k], m = ent & 0xFFFFFF;
            if ((ent >> 24) != 16 || m == j) continue;
            const Rec rm = S.rec[m];
            Geo g;
            geo(r, rm, tf, g);
            const int idm = dyn_ident(rm.dyn);
            if (g.r2 <= T.welldia_sq[idi][idm]) {
                const double e = T.ep_sqrt[idi][idm];
                if (topo_chain(r.topo) == topo_chain(rm.topo))
                    sum[1] = sum[1] + e;
                else
                    sum[2] = sum[2] + e;
            }
        }
    }
    for (int k = 0; k < kObsSums; ++k) {
        const double v = wave_sum(sum[k]);
        if (lane == 0) red[wave][k] = v;
    }
    __syncthreads();
    if ((int)threadIdx.x < kObsSums) {
        double v = red[0][threadIdx.x];
        for (int w = 1; w < kObsT / kW; ++w) v = v + red[w][threadIdx.x];
        obs_bead_sums(S)[kObsSums * (size_t)blockIdx.x + threadIdx.x] = v;
    }
}
// A wavefront per chain: squared radius of gyration, summed over the
// backbone, and end-to-end distance.  nfirst: chains of the leading species
// block.
__global__ __launch_bounds__(kObsT) void k_obs_chains(const SysDev* __restrict__ sys, int id, const int* cstart,
                                                      const int* clen, int nch, int nfirst) {
    const SysDev& S = sys[id];
    const int c = (int)blockIdx.x * (kObsT / kW) + wave_id(), lane = lane_id();
    if (c >= nch) return;
    const int s = cstart[c], L = clen[c], n = 3 * L;
    // radgyr.f:117-125 sums a chain of the second species block over
    // beads (c-1)*numbeads2+1 .. +3*chnln2 without the first block's
    // offset its unwrapping uses (:78), while those beads exist
    int rb = s;
    if (c >= nfirst && c * 4 * L + 3 * L <= s + 4 * L) rb = c * 4 * L;
    const double4* q = S.spos + rb;
    double cx = 0.0, cy = 0.0, cz = 0.0, rg = 0.0;
    for (int k = lane; k < n; k += kW) {
        const double4 v = q[k];
        cx = cx + v.x;
        cy = cy + v.y;
        cz = cz + v.z;
    }
    cx = wave_sum(cx) / (double)n;
    cy = wave_sum(cy) / (double)n;
    cz = wave_sum(cz) / (double)n;
    for (int k = lane; k < n; k += kW) {
        const double4 v = q[k];
        rg = rg + (v.x - cx) * (v.x - cx) + (v.y - cy) * (v.y - cy) + (v.z - cz) * (v.z - cz);
    }
    rg = wave_sum(rg);
    if (lane == 0) {
        obs_chain_sums(S)[2 * c] = rg;
        // end2end.f: N of residue 1 to C of residue L
        obs_chain_sums(S)[2 * c + 1] = dist_rec(S.rec[s + L], S.rec[s + 3 * L - 1], S.st->tfalse);
    }
}
// outd: ered, tred, sumvel, ehh_ii, ehh_ij, rg_avg, e2e_avg; outi: hb_alpha,
// hb_ii, hb_ij.
__global__ __launch_bounds__(kW) void k_obs_sum(const SysDev* __restrict__ sys, int id, int nb, int nch, double boxl,
                                                double* outd, int* outi) {
    const SysDev& S = sys[id];
    const int N = S.N, lane = lane_id();
    double v[kObsSums] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, rg = 0.0, e2e = 0.0;
    const double* pb = obs_bead_sums(S);
    const double* pc = obs_chain_sums(S);
    for (int b = lane; b < nb; b += kW)
        for (int k = 0; k < kObsSums; ++k) v[k] = v[k] + pb[kObsSums * b + k];
    for (int c = lane; c < nch; c += kW) {
        rg = rg + pc[2 * c];
        e2e = e2e + pc[2 * c + 1];
    }
    for (int k = 0; k < kObsSums; ++k) v[k] = wave_sum(v[k]);
    rg = wave_sum(rg);
    e2e = wave_sum(e2e);
    if (lane == 0) {
        const double sumvel = v[0], eii = v[1], eij = v[2], nbb = (double)(3 * (N / 4));  // backbone beads
        const int hii = (int)v[3], hij = (int)v[4], sum_hb = hii + hij;
        const double sumeps = -(sum_hb * S.tab->ep_sqrt[5][8] + (eii + eij));
        outd[0] = 0.5 * sumvel + sumeps;
        outd[1] = sumvel / 3.0 / (double)N;
        outd[2] = sumvel;
        outd[3] = eii;
        outd[4] = eij;
        outd[5] = sqrt(rg / nbb) * boxl;
        outd[6] = e2e / (double)nch * boxl;
        outi[0] = (int)v[5];
        outi[1] = hii;
        outi[2] = hij;
    }
}

// ------------------------------------------------------------------------
// What the host reads, written by kernels straight into page-locked host
// memory in the host's layout: one launch and one wait.  A state read as three
// blocking copies to pageable memory and a pass over the records on the host
// took 45 us more at 128 to 1536 beads (320 systems advanced by 2000 entries
// and read: 35.1 ms, 20.5 ms).
// ------------------------------------------------------------------------
__global__ __launch_bounds__(kGridT) void k_state(const SysDev* __restrict__ sys, int id, int want, double* out) {
    const SysDev& S = sys[id];
    const int N = S.N, w = (int)(blockIdx.x * kGridT + threadIdx.x);
    const StateLayout at(N);
    int* iout = reinterpret_cast<int*>(out);
    // a lane per output word, so that a wavefront writes whole lines
    if ((want & kStateSv) && w < 6 * N) {
        const int k = w / 6;
        out[w] = gl1(reinterpret_cast<const double*>(S.rec + k) + (w - 6 * k));
    }
    if (w < N + 3) {
        if (want & kStateTim) out[at.tim + w] = gl1(&S.leaf[w].tim);
        if (want & kStateNptnr) {
            const int p = gl1(&S.leaf[w].nptnr);
            iout[at.nptnr + w] = p >= 0 ? p + 1 : p;
        }
        if (want & kStateColtype) iout[at.coltype + w] = leaf_ct(gl1(&S.leaf[w].meta));
    }
    if (w < N) {
        const int dyn = gl1(&S.rec[w].dyn);
        if (want & kStateIdent) iout[at.ident + w] = dyn_ident(dyn);
        if (want & kStateBptnr) iout[at.bptnr + w] = dyn_bptnr(dyn) + 1;
    }
    if ((want & kStateExtra) && w < 4 * N) iout[at.extra + w] = gl1(reinterpret_cast<const int*>(S.extra) + w) + 1;
}
__global__ __launch_bounds__(kGridT) void k_status(const SysDev* __restrict__ sys, const int* ids, int n, int* out) {
    const int k = (int)(blockIdx.x * kGridT + threadIdx.x);
    if (k < n) out[k] = sys[ids[k]].st->status;
}
// The counters, and the row lengths summed over the beads, of system ids[blockIdx.x].
__global__ __launch_bounds__(kStatsT) void k_stats(const SysDev* __restrict__ sys, const int* ids, SysStats* out) {
    __shared__ unsigned long long red[2][kStatsT / kW];
    const SysDev& S = sys[ids[blockIdx.x]];
    const int N = S.N, t = (int)threadIdx.x, lane = lane_id(), wave = wave_id();
    unsigned long long* o = reinterpret_cast<unsigned long long*>(out + blockIdx.x);
    const unsigned long long* st = reinterpret_cast<const unsigned long long*>(S.st);
    for (int k = t; k < (int)(sizeof(SysState) / 8); k += kStatsT) o[k] = st[k];
    int up = 0, dn = 0;  // a wavefront sums at most 65 533 rows of 64 entries
#pragma unroll 4
    for (int k = t; k < N; k += kStatsT) {
        up += S.nup[k];
        dn += S.ndn[k];
    }
    up = __builtin_amdgcn_readlane(wave_scan(up), kW - 1);
    dn = __builtin_amdgcn_readlane(wave_scan(dn), kW - 1);
    if (lane == 0) {
        red[0][wave] = (unsigned long long)up;
        red[1][wave] = (unsigned long long)dn;
    }
    __syncthreads();
    if (t < 2) {
        unsigned long long v = 0;
        for (int w = 0; w < kStatsT / kW; ++w) v += red[t][w];
        o[sizeof(SysState) / 8 + t] = v;
    }
}

// test hook: predicted collision time of listed pairs (1-based in, code
// from ev_code(j,i) as events.f/eventredo_up.f read it)
__global__ void k_predict(const SysDev* sys, int id, int n, const int* pi, const int* pj, double* tij, int* type) {
    const SysDev& S = sys[id];
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int i = pi[k] - 1, j = pj[k] - 1;
    if (i < 0 || j < 0 || i >= S.N || j >= S.N || i == j) {
        tij[k] = 0.0;
        type[k] = -100;
        return;
    }
    const Rec ri = gld(S.rec + (i)), rj = gld(S.rec + (j));
    const int code = dyn_code(gld(S.ovr + (j)), i, static_t(*S.tab, rj.topo, ri.topo));
    double t = 1000000000.0;
    int ty = 0;
    predict(*S.tab, code, ri, rj, dyn_bptnr(ri.dyn) == j, gld(S.bw + (i)), S.st->tfalse, t, ty);
    tij[k] = t;
    type[k] = ty;
}

// predictions of i and j in full, their down sets and a share of the beads
// recomputed (one that finds no room is recomputed on its own)
int engine_maxw(int cap) { return 6 * (cap + 3); }

static size_t r16(size_t b) { return (b + 15) / 16 * 16; }
size_t engine_lds_bytes(int nblk, int maxw, int nw) {
    const size_t b = (size_t)kPoolOff + (size_t)nw * lds_wave_bytes() + lds_multi_bytes(maxw) + r16(sizeof(unsigned) * nblk) +
                     4096;  // the fewest footprint marks
    return std::max(b, (size_t)kPoolOff + kScratch);
}
static int nblk_for(int n) { return (n + 3 + kBlk - 1) / kBlk; }

static hipError_t list_launches(const SysDev* d_sys, const int* d_ids, int n, int max_n, int forced, hipStream_t s) {
    const unsigned beads = (unsigned)(max_n + 3 + kGridT - 1) / kGridT, rows = (unsigned)(2 * max_n + kGridT - 1) / kGridT;
    const unsigned places = kCells * (kGridT / kW), search = ((unsigned)max_n + places - 1) / places;
    const dim3 t(kGridT), g(beads, (unsigned)n);
    hipLaunchKernelGGL(k_list_beads, g, t, 0, s, d_sys, d_ids, forced);
    hipLaunchKernelGGL(k_list_scan, dim3(1, (unsigned)n), dim3(kScanT), 0, s, d_sys, d_ids, forced);
    hipLaunchKernelGGL(k_list_copy, g, t, 0, s, d_sys, d_ids);
    hipLaunchKernelGGL(k_list_search, dim3(search, (unsigned)n), t, 0, s, d_sys, d_ids);
    hipLaunchKernelGGL(k_list_sort, dim3(rows, (unsigned)n), t, 0, s, d_sys, d_ids);
    hipLaunchKernelGGL(k_list_events, g, t, 0, s, d_sys, d_ids);
    return hipGetLastError();
}
hipError_t engine_setup(const SysDev* d_sys, const int* d_ids, int n, int max_n, hipStream_t s) {
    return list_launches(d_sys, d_ids, n, max_n, 0, s);
}
hipError_t engine_rebuild(const SysDev* d_sys, const int* d_ids, int n, int max_n, hipStream_t s) {
    return list_launches(d_sys, d_ids, n, max_n, 1, s);
}
// clears the start word of a budgeted launch (a kernel rather than a memset,
// so that a captured graph replays it faithfully)
__global__ void k_clock_reset(unsigned long long* w) { *w = ~0ull; }

// Shape of a launch of n systems at `waves` event wavefronts each: nw
// wavefronts with work areas (the event wavefronts and the calendar one), all
// that are launched, LDS bytes.
struct RunShape {
    int nw, total;
    size_t lds;
};
static RunShape run_shape(int n, int max_n, int maxw, size_t lds_limit, int waves) {
    static const int ncu = [] {
        int dev = 0, v = 0;
        const bool ok = hipGetDevice(&dev) == hipSuccess &&
                        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess;
        return ok && v > 0 ? v : 1;
    }();
    const int nblk = nblk_for(max_n);
    RunShape r;
    r.nw = 1 + (waves < 1 ? 1 : (waves > kMaxWaves - 1 ? kMaxWaves - 1 : waves));
    // Up to one workgroup per compute unit each takes the whole LDS budget,
    // so every system keeps as many leaves in LDS as fit beside its own block
    // minima.  Beyond that, a compute unit holds eight wavefronts of the
    // registers that k_run takes, so workgroups of at most four share it two
    // by two: a wavefront less costs a system far less than waiting for
    // another one's whole launch.  257 systems at four wavefronts asked for,
    // two by two / one by one: 128 beads 9.5 / 15.7 ms, 1536 8.2 / 11.1, 23 424
    // 3.8 / 5.3; at eight 9.4 / 15.9, 8.2 / 7.7, 3.8 / 3.6, where one by one would
    // be the better form from some 1000 beads on.
    size_t room = lds_limit;
    const int nw2 = std::min(r.nw, kMaxWaves / 2);
    if (n > ncu && engine_lds_bytes(nblk, maxw, nw2) <= lds_limit / 2) {
        room = lds_limit / 2;
        r.nw = nw2;
    }
    while (r.nw > 2 && engine_lds_bytes(nblk, maxw, r.nw) > lds_limit) --r.nw;
    const size_t base = engine_lds_bytes(nblk, maxw, r.nw);
    r.lds = room;
    if (n > ncu) r.lds = std::min(room, base + (sizeof(Leaf) + sizeof(unsigned)) * (size_t)(max_n + 4));
    if (r.lds < base) r.lds = base;
    // A workgroup alone on its compute unit takes all the wavefronts that the
    // unit holds: those beyond nw wait at the barriers, for nothing, except
    // where the whole workgroup works, above all in list updates (512 beads at
    // one event wavefront: 18.8 ms for 2500 entries without them, 17.6 with;
    // 1920 dense beads at four: 14.8 ms, 13.7).
    r.total = n > ncu ? r.nw : kMaxWaves;
    return r;
}
hipError_t engine_run(const SysDev* d_sys, const int* d_ids, const long long* d_inc, int n, int max_n, int maxw,
                      size_t lds_limit, hipStream_t s, long long budget_ticks, int flags, int waves,
                      unsigned long long* launch_t0) {
    const RunShape r = run_shape(n, max_n, maxw, lds_limit, waves);
    if (budget_ticks > 0) {
        if (!launch_t0) return hipErrorInvalidValue;
        hipLaunchKernelGGL(k_clock_reset, dim3(1), dim3(1), 0, s, launch_t0);
    }
    hipLaunchKernelGGL(k_run, dim3(n), dim3(kW * r.total), r.lds, s, d_sys, d_ids, d_inc, maxw, (int)r.lds, r.nw - 1,
                       budget_ticks, flags, launch_t0);
    return hipGetLastError();
}
int engine_max_waves(int n, int max_n, int maxw, size_t lds_limit) {
    return run_shape(n, max_n, maxw, lds_limit, kMaxWaves).nw - 1;
}
hipError_t engine_predict(const SysDev* d_sys, int id, int n, const int* pi, const int* pj, double* tij, int* type,
                          hipStream_t s) {
    hipLaunchKernelGGL(k_predict, dim3((n + 255) / 256), dim3(256), 0, s, d_sys, id, n, pi, pj, tij, type);
    return hipGetLastError();
}
hipError_t engine_check(const SysDev* d_sys, int id, int n, const Rec* alt, unsigned long long* out, hipStream_t s) {
    hipLaunchKernelGGL(k_check, dim3((n + 255) / 256), dim3(256), 0, s, d_sys, id, alt, out);
    return hipGetLastError();
}
hipError_t engine_observables(const SysDev* d_sys, int id, int n, const int* cstart, const int* clen, int nch, int nfirst,
                              double boxl, double* outd, int* outi, hipStream_t s) {
    const int nb = (n + kObsBeads - 1) / kObsBeads, nc = (nch + kObsT / kW - 1) / (kObsT / kW);
    hipLaunchKernelGGL(k_obs_parts, dim3(nb + nc), dim3(kObsT), 0, s, d_sys, id, nb, cstart, clen, nch);
    hipLaunchKernelGGL(k_obs_chains, dim3(nc), dim3(kObsT), 0, s, d_sys, id, cstart, clen, nch, nfirst);
    hipLaunchKernelGGL(k_obs_sum, dim3(1), dim3(kW), 0, s, d_sys, id, nb, nch, boxl, outd, outi);
    return hipGetLastError();
}
hipError_t engine_state(const SysDev* d_sys, int id, int n, int want, double* out, hipStream_t s) {
    hipLaunchKernelGGL(k_state, dim3((6 * n + kGridT - 1) / kGridT), dim3(kGridT), 0, s, d_sys, id, want, out);
    return hipGetLastError();
}
hipError_t engine_status(const SysDev* d_sys, const int* d_ids, int n, int* out, hipStream_t s) {
    hipLaunchKernelGGL(k_status, dim3((n + kGridT - 1) / kGridT), dim3(kGridT), 0, s, d_sys, d_ids, n, out);
    return hipGetLastError();
}
hipError_t engine_stats(const SysDev* d_sys, const int* ids, int n, SysStats* out, hipStream_t s) {
    hipLaunchKernelGGL(k_stats, dim3(n), dim3(kStatsT), 0, s, d_sys, ids, out);
    return hipGetLastError();
}

hipError_t engine_prepare(size_t lds_limit) {
    return hipFuncSetAttribute((const void*)k_run, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_limit);
}

}  // namespace pdmd
