// RTAMC2D transient solver on the GPU: one lane per particle history,
// lanes refill from a particle counter when their particle ends.
//
// Reference: src/RTA_MC2D.cpp
//   Init_generator (wall part)  272-533   -> rta_start()
//   diffusive_bouncing::bounce  635-678   -> per-(side, mode) alias rows
//   process_segment (transient) 699-769   -> tally_segment()
//   evolparticle (transient)    990-1386  -> rta_fly(), rta_slow()
//   history loop                2228-2317 -> rta_histories()
//   post-processing             2326-2435 -> rta_postprocess()
#include "flight_log.hpp"
#include "runtime.hpp"
#include <algorithm>
#include <chrono>
#include <cstring>
#include <numeric>
#include <tuple>
#include <limits>
#include <mutex>
#include <rocblas/rocblas.h>

namespace bte {

struct RtaGen {
    double p1x, p1y, ndx, ndy;
    int32_t idi, sign, pad0, pad1;
};

// One run of a batch: its particle-id range, seed, tables and options. All
// box, generator and table indices are absolute in the batch's arrays.
struct RtaRunDev {
    uint64_t first, count, seed;
    int32_t gen0, ngen, gsel0, pad2;
    int32_t ballistic, gmask, pad0, pad1;  // gmask: sides whose specularity gets a gradient
    double wscale;                         // scattering-rate factor of the run
    float spec[4];                         // specular probability per side
};

// Tally mode 3: one run of the batch and its rows in the FP64 LDS block of a
// workgroup that follows its histories.
struct RtaRunRows {
    int32_t lrow0;       // global LDS row of the run's first regular box
    int32_t lrows;       // the run's regular boxes
    int32_t lbins;       // leading time bins of each row held in LDS
    int32_t wgs;         // workgroups that begin with this run
    int32_t box0, nbox, side0, nsides;  // the run's boxes and polygon sides
};

// One mode as the history kernels read it: 64 bytes in one cache line, so a
// new mode costs one line (velocity, inverse velocity, rate and the range of
// its diffuse-bounce table) instead of one line in each of three arrays.
struct __align__(64) RtaMode {
    double vx, vy, ivx, ivy;       // inverses are 0 where the component is 0
    double w, iw;                  // rate and 1 / w
    int32_t lo, len, base, pad;    // Lambert table: first partner, partners, offset
};
static_assert(sizeof(RtaMode) == 64, "one mode record is half a 128-byte line");

// One box as the history kernels read it.
struct __align__(16) RtaBox {
    double xmin, xmax, ymin, ymax;
    int32_t side_nbr[4];  // as DevBox
    int32_t kind, lrow;  // lrow: LDS tally row of a regular box
    int32_t s0, ns;      // polygon geometries: first side and sides
};
static_assert(sizeof(RtaBox) == 64, "box record");

struct RtaParams {
    const RtaMode* rmodes;
    const RtaBox* rboxes;
    const int32_t* mirror; // [2][n]: partner with vx -> -vx (sides 0, 3), vy -> -vy (sides 1, 2)
    const uint2* scat;     // BE_derivative alias per run (n each)
    const DevBox* boxes;
    const DevContact* cts;
    const double4* cseg;    // contact segments (periodic translation)
    const DevCross* cross;  // contacts as translate_rect reads them
    const double2* ptrans;  // periodic translation per box
    // polygon geometries (POLY kernels): sides, side range and centre per box
    const DevSide* sides;
    const int2* srange;
    const double2* center;
    const RtaGen* gens;
    const uint2* gen_sel;  // alias over each run's generators
    const uint2* gen_tab;  // per generator, n entries
    const uint2* lam_tab;
    const int32_t* perm;   // omega-sorted position -> mode
    const double* timegrid;
    const RtaRunDev* runs;
    double* gz;
    double* jx;
    double* jy;
    double* dgz;           // [4][cells] score-weighted gz per side (gradient runs)
    const int32_t* box_loc; // spectral location of each box, -1 none
    double* spec;          // [nloc][nt][n] per-mode gz of the spectral locations (null: none)
    unsigned long long* counters;  // events, crossings, next id, stuck, bad mirror, bad translation
    uint64_t total;        // particles over all runs
    uint64_t cells;
    double maxtime;
    int32_t n, nt, nruns, pad;
    // LDS tallies: the global cell of each LDS row (a regular box); the rows
    // and their leading time bins held in LDS. Mode 1: lt_arrays FP32 arrays
    // [lrows][lbins]: gz, jx, jy, then array lt_goff[s] of side s for each
    // differentiated side (-1: none). Mode 2: FP64 gz, jx, jy; each workgroup
    // writes its block to part[blockIdx.x] at the end.
    const uint64_t* lrow_cell;
    int32_t lrows, lbins;
    int32_t lt_goff[4], lt_arrays;
    double* part;
    // geometry in LDS (GL kernels): boxes and sides of the batch (modes 0 to
    // 2), the byte offsets of the sides and the time grid after the boxes and
    // of the tallies after both
    int32_t nboxes, nsides, geo_side, geo_grid, geo_bytes;
    int32_t mig;    // byte offset of the mailbox (-1: none)
    int32_t waves;  // waves that share the particles (modes 0 to 2)
    double idt;  // nt / maxtime: time -> bin estimate on the uniform grid
    // tally mode 3: the runs' rows, the run each workgroup begins with (-1:
    // none), and per run the next particle (from 0) and the workgroups on it
    const RtaRunRows* rows;
    const int32_t* first_run;
    unsigned long long* run_next;
    unsigned long long* run_wgs;
};

// Per-XCD copies of the f64 tallies. Device-wide f64 atomics to a few
// thousand cells are the RTAMC2D kernel's main cost; spread over one copy
// per XCD they run about 25 % faster.
#define RTA_NCOPY 8
// the XCD (XCC) this wave runs on, from the hardware register HW_REG_XCC_ID

static __device__ const LogEntry rta_log_table[FLIGHT_LOG_N] = FLIGHT_LOG_TABLE;

// Boxes, polygon sides and the time grid of the history kernels: in LDS (GL),
// behind the table of the flight logarithm, when they take at most
// RTA_GEO_LDS bytes, else in global memory. Every
// lane of a wave reads its own box, side and time bin, and such a scattered
// load occupies the vector memory pipe for one cycle per lane: with the
// geometry, the grid and the mode record read from global memory for every
// segment, 57 loads per wave and segment kept that pipe busy all the time
// (16 runs of 3000 modes, 5.5e6 particles: 68 ms). LDS serves them 128 bytes a
// cycle. A box takes 80 bytes of LDS: a stride of 20 banks starts 16
// consecutive boxes at 16 different 16-byte groups, where 64 bytes would put
// them on four.
#define RTA_GEO_LDS 20480
#define RTA_BOX_LDS 80
template <bool GL>
struct RtaGeo {
    const unsigned char* box;
    const DevSide* side;
    const double* grid;
    const LogEntry* log;
    int32_t bo;      // tally mode 3: first box of the run (staged indices are local)
    int32_t run;     // tally mode 3: the run of every lane, and its rate factor
    double wscale, iws;  // and 1 / wscale
    __device__ inline RtaBox at(int i) const {
        return *reinterpret_cast<const RtaBox*>(box + (size_t)i * (GL ? RTA_BOX_LDS : sizeof(RtaBox)));
    }
};

// Copy nb boxes from bo on and ns sides from so on (with local indices), and
// the time grid and the logarithm's table, into LDS. The caller synchronises.
template <bool POLY>
__device__ inline void rta_stage_boxes(const RtaParams& P, unsigned char* lds, int bo, int nb, int so, int ns, int lrow0) {
    for (int i = threadIdx.x; i < nb; i += blockDim.x) {
        RtaBox b = P.rboxes[bo + i];
        for (int k = 0; k < 4; k++)
            if (b.side_nbr[k] >= 0) b.side_nbr[k] -= bo;
        b.lrow -= lrow0;
        b.s0 -= so;
        *reinterpret_cast<RtaBox*>(lds + FLIGHT_LOG_BYTES + (size_t)i * RTA_BOX_LDS) = b;
    }
    if constexpr (POLY) {
        DevSide* S = reinterpret_cast<DevSide*>(lds + P.geo_side);
        for (int i = threadIdx.x; i < ns; i += blockDim.x) {
            DevSide s = P.sides[so + i];
            if (s.nbr >= 0) s.nbr -= bo;
            S[i] = s;
        }
    }
}
__device__ inline void rta_stage_grid(const RtaParams& P, unsigned char* lds) {
    LogEntry* t = reinterpret_cast<LogEntry*>(lds);
    for (int i = threadIdx.x; i < FLIGHT_LOG_N; i += blockDim.x) t[i] = rta_log_table[i];
    double* g = reinterpret_cast<double*>(lds + P.geo_grid);
    for (int i = threadIdx.x; i <= P.nt; i += blockDim.x) g[i] = P.timegrid[i];
}

// get_bin_index (RTA_MC2D.cpp:140-148): lower_bound - 1 clamped to
// [0, nt-1], of a time target >= 0. The grid is uniform (t_i = i maxtime /
// nt), so the bin is estimated from target * nt / maxtime and corrected
// against the grid values themselves, which keeps lower_bound's result
// exactly (a target on a grid point t_j belongs to bin j - 1). upper: the
// bin's upper grid value.
__device__ inline int time_bin(const double* grid, int nt, double idt, double target, double& upper) {
    int k = min((int)fmin(target * idt, 2.0e9), nt - 1);
    double lower = grid[k];
    upper = grid[k + 1];
    while (k > 0 && lower >= target) {
        k--;
        upper = lower;
        lower = grid[k];
    }
    while (k < nt - 1 && upper < target) {
        k++;
        upper = grid[k + 1];
    }
    return k;
}

// Where a workgroup's tallies go. Cells are numbered by one key: keys below
// lc are cells of the LDS block (row * lbins + bin), the others lc + the
// cell of the XCD's copy (box * nt + bin, boxes from the first box of the
// tallied range on).
struct RtaTally {
    void* lds;           // FP64 [3][rows][lbins] (modes 2, 3) or FP32 arrays (mode 1)
    uint32_t lbins, lc;  // time bins of a row held in LDS; rows * lbins
    int32_t row0;        // box records' row of the block's first row
    double* g;           // gz of the XCD's copy at cell 0 of the tallied range
    double* dg;          // score-weighted gz of side 0 there (gradient runs)
};

// A lane's running sum of consecutive contributions to one tally cell
// (box, time bin); it is added to the tallies when the lane's next
// contribution falls in another cell and when the lane's histories end.
// Successive segments of a history often share a cell (several flights in
// one box within one time bin), and each cell update costs three adds.
template <bool D>
struct TallyAcc {
    uint32_t key = ~0u;
    double g = 0., x = 0., y = 0.;
    double d[D ? 4 : 1] = {};  // score-weighted sums per side
};

// Adds the accumulator into the tallies: an LDS cell under modes 2 and 3,
// else the XCD's copy by device atomics.
template <int TM, bool D>
__device__ inline void acc_flush(const RtaParams& P, const RtaTally& T, TallyAcc<D>& a) {
    if (a.key == ~0u) return;
    if ((TM == 2 || TM == 3) && a.key < T.lc) {
        // an LDS pointer by type: with generic ones the compiler merges the
        // tails of both branches into flat atomics
        auto* L = (__attribute__((address_space(3))) double*)T.lds + a.key;
        __builtin_amdgcn_ds_atomic_fadd_f64(L, a.g);
        __builtin_amdgcn_ds_atomic_fadd_f64(L + T.lc, a.x);
        __builtin_amdgcn_ds_atomic_fadd_f64(L + 2 * T.lc, a.y);
    } else {
        const uint64_t k = a.key - T.lc;
        atomicAdd(T.g + k, a.g);
        atomicAdd(T.g + P.cells + k, a.x);
        atomicAdd(T.g + 2 * P.cells + k, a.y);
        if constexpr (D) {
#pragma unroll
            for (int s = 0; s < 4; s++)
                if (a.d[s] != 0.) atomicAdd(T.dg + (uint64_t)s * P.cells + k, a.d[s]);
        }
    }
    a.key = ~0u;
}

// State of a lane. FRESH draws a flight and then flies; FLY continues one
// across boxes; the pending states wait for rta_slow; DEAD waits for the
// next particle id; DONE has none left.
enum { RTA_DEAD = 0, RTA_FRESH = 1, RTA_FLY = 2, RTA_WALL = 3, RTA_MIXED = 4, RTA_TRANS = 5, RTA_DONE = 6 };

// The state of one particle history between events.
struct RtaState {
    Pcg32 rng;
    uint64_t look;             // generator state after the look-ahead draws
    double x, y, t, dtrem;
    double vx, vy, ivx, ivy;   // of the mode in flight
    uint2 se;                  // look-ahead alias entry of the next scattering
    uint32_t sk, su, budget;
    int mode, box, still, bin, st, aux;  // aux: side (WALL) or side mask (MIXED)
    int run;                   // modes 0 to 2: the lane's run and its rate factor
    double wscale, iws;        // and 1 / wscale
    int sign, ballistic, gmask;
    float score[4];
};

struct RtaCounts {
    uint32_t events = 0, crossings = 0;
};

// Adds a segment's contribution c to time bin i of the lane's box (lrow: its
// LDS row); gradient runs also add it weighted by the particle's running
// score for each active side.
// TM (tally mode) 0: FP64 device atomics. 1: the workgroup's FP32 partial
// sums in LDS for the leading lbins bins, later ones by device atomics. 2: the
// same with FP64 partial sums. 3: as 2 with the LDS block holding only the
// rows of the run that the workgroup follows. All modes but 1
// merge consecutive contributions to one cell in the lane's accumulator.
template <bool GRAD, int TM, bool D>
__device__ inline void tally_bin(const RtaParams& P, const RtaTally& T, TallyAcc<D>& A, const RtaState& S, int lrow,
                                 double* spec, int i, double c) {
    if (c == 0.) return;
    const uint32_t row0 = (uint32_t)(lrow - T.row0) * T.lbins, cell0 = (uint32_t)S.box * (uint32_t)P.nt;
    if constexpr (TM == 1) {
        if ((uint32_t)i < T.lbins) {
            float* L = (float*)T.lds + row0 + i;
            atomicAdd(L, (float)c);
            atomicAdd(L + T.lc, (float)(S.vx * c));
            atomicAdd(L + 2 * T.lc, (float)(S.vy * c));
            if (GRAD) {
#pragma unroll
                for (int s = 0; s < 4; s++)
                    if (P.lt_goff[s] >= 0 && ((S.gmask >> s) & 1) && S.score[s] != 0.f)
                        atomicAdd(L + (uint32_t)P.lt_goff[s] * T.lc, (float)(c * (double)S.score[s]));
            }
        } else {
            const uint64_t k = cell0 + (uint32_t)i;
            atomicAdd(T.g + k, c);
            atomicAdd(T.g + P.cells + k, S.vx * c);
            atomicAdd(T.g + 2 * P.cells + k, S.vy * c);
            if (GRAD) {
#pragma unroll
                for (int s = 0; s < 4; s++)
                    if (((S.gmask >> s) & 1) && S.score[s] != 0.f)
                        atomicAdd(T.dg + (uint64_t)s * P.cells + k, c * (double)S.score[s]);
            }
        }
    } else {
        if (TM == 0 && !GRAD && spec) atomicAdd(spec + (size_t)i * P.n, c);
        const uint32_t key = (TM == 0 || (uint32_t)i >= T.lbins) ? T.lc + cell0 + (uint32_t)i : row0 + (uint32_t)i;
        if (key != A.key) {
            acc_flush<TM, D>(P, T, A);
            A.key = key;
            A.g = A.x = A.y = 0.;
            if constexpr (D) A.d[0] = A.d[1] = A.d[2] = A.d[3] = 0.;
        }
        A.g += c;
        A.x += S.vx * c;
        A.y += S.vy * c;
        if constexpr (D) {
#pragma unroll
            for (int s = 0; s < 4; s++)
                if ((S.gmask >> s) & 1) A.d[s] += c * (double)S.score[s];
        }
    }
}

// process_segment (RTA_MC2D.cpp:699-769) from the lane's time to t1, which
// becomes the lane's time. The lane keeps its time bin: the bin of a
// segment's start is that of the previous one's end. In bin i the segment
// [t0, t1] covers [max(t_i - t0, 0), min(t_i+1 - t0, t1 - t0)], where only the
// first bin's lower and the last bin's upper bound are not grid differences.
template <bool GRAD, int TM, bool GL, bool D>
__device__ inline void tally_segment(const RtaParams& P, const RtaGeo<GL>& G, const RtaTally& T, TallyAcc<D>& A,
                                     RtaState& S, int lrow, double t1) {
    const double t0 = S.t, delta = t1 - t0;
    double upper;
    const int b1 = time_bin(G.grid, P.nt, P.idt, t1, upper);
    double* spec = nullptr;
    if (TM == 0 && !GRAD && P.spec) {
        // spectral locations tally per mode; the Gamma-broadened spectra are
        // one matrix product after the run (the reference adds the broadened
        // weights of every segment, RTA_MC2D.cpp:718-766)
        const int l = P.box_loc[S.box];
        if (l >= 0) spec = P.spec + (size_t)l * P.nt * P.n + S.mode;
    }
    double lo = 0.;
    for (int i = S.bin; i < b1; i++) {
        const double g = G.grid[i + 1] - t0;
        tally_bin<GRAD, TM, D>(P, T, A, S, lrow, spec, i, S.sign * fmax(g - lo, 0.));
        lo = g;
    }
    tally_bin<GRAD, TM, D>(P, T, A, S, lrow, spec, b1, S.sign * fmax(fmin(upper - t0, delta) - lo, 0.));
    S.bin = b1;
    S.still = t1 == t0 ? S.still + 1 : 0;
    S.t = t1;
}

// the run holding global particle id pid (first ids ascending)
__device__ inline int find_run(const RtaParams& P, uint64_t pid) {
    int lo = 0, hi = P.nruns - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (P.runs[mid].first <= pid) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// The workgroup's LDS partial sums into the FP64 tallies (the XCD's copy).
template <bool GRAD>
__device__ inline void lt_flush(const RtaParams& P, const RtaTally& T) {
    const float* lt = (const float*)T.lds;
    for (uint32_t j = threadIdx.x; j < T.lc; j += blockDim.x) {
        const uint32_t row = j / T.lbins;
        const uint64_t g = P.lrow_cell[row] + (j - row * T.lbins);
        for (int a = 0; a < 3; a++) {
            const float v = lt[(size_t)a * T.lc + j];
            if (v != 0.f) atomicAdd(T.g + (uint64_t)a * P.cells + g, (double)v);
        }
        if (GRAD) {
            for (int s = 0; s < 4; s++) {
                if (P.lt_goff[s] < 0) continue;
                const float v = lt[(size_t)P.lt_goff[s] * T.lc + j];
                if (v != 0.f) atomicAdd(T.dg + (uint64_t)s * P.cells + g, (double)v);
            }
        }
    }
}

// Event and crossing counts of the workgroup through LDS (16-byte aligned,
// 16 waves at most), one global atomic per counter; every thread calls this.
extern __shared__ __align__(16) unsigned char rta_lds[];
__device__ inline void rta_add_counts(const RtaParams& P, const RtaCounts& C) {
    unsigned long long* part = reinterpret_cast<unsigned long long*>(rta_lds);
    unsigned long long ev = C.events, cr = C.crossings;
    for (int d = 32; d > 0; d >>= 1) {
        ev += __shfl_down(ev, d, 64);
        cr += __shfl_down(cr, d, 64);
    }
    __syncthreads();  // the block's LDS has been read
    if ((threadIdx.x & 63) == 0) {
        part[2 * (threadIdx.x >> 6)] = ev;
        part[2 * (threadIdx.x >> 6) + 1] = cr;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        unsigned long long t = 0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += part[2 * w + threadIdx.x];
        if (t) atomicAdd(P.counters + threadIdx.x, t);
    }
}

// The kernel's parameters for code off the main path: read from the kernel
// argument segment where they are used. Kept in scalar registers over the
// whole loop, the pointers of these paths would push those of the main path
// into vector lanes (a lane read for each use).
__device__ inline const RtaParams& rta_cold_params() {
    auto* p = (const __attribute__((address_space(4))) RtaParams*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const RtaParams*)p;
}

// Init_generator (RTA_MC2D.cpp:436-484): particle pid of its run at t = 0.
template <bool GRAD, int TM, bool POLY, bool GL>
__device__ inline void rta_start(const RtaGeo<GL>& G, RtaState& S, uint64_t pid) {
    const RtaParams& P = rta_cold_params();
    S.budget = 0;
    S.still = -1;  // the first event of a history never counts as standing still
    if (TM != 3) S.run = find_run(P, pid);
    const RtaRunDev& R = P.runs[TM == 3 ? G.run : S.run];
    S.wscale = R.wscale;
    S.iws = 1.0 / S.wscale;
    S.rng.seed(R.seed, pid - R.first);
    S.ballistic = R.ballistic;
    S.gmask = R.gmask;
    if (GRAD) S.score[0] = S.score[1] = S.score[2] = S.score[3] = 0.f;
    bool ng;
    int gi = R.gen0 + (int)alias_pick(P.gen_sel + R.gsel0, (uint32_t)R.ngen, S.rng, ng);
    const RtaGen g = P.gens[gi];
    double u = S.rng.uniform();
    S.x = g.p1x + u * g.ndx;
    S.y = g.p1y + u * g.ndy;
    S.box = g.idi - G.bo;
    const RtaBox B = G.at(S.box);
    const bool in = POLY ? poly_inside(G.side, make_int2(B.s0, B.ns), S.x, S.y)
                         : S.x >= B.xmin && S.x <= B.xmax && S.y >= B.ymin && S.y <= B.ymax;
    if (!in) {
        const double ccx = POLY ? P.center[g.idi].x : 0.5 * (B.xmin + B.xmax);
        const double ccy = POLY ? P.center[g.idi].y : 0.5 * (B.ymin + B.ymax);
        double dx = ccx - S.x, dy = ccy - S.y;
        double dn = sqrt(dx * dx + dy * dy);
        S.x += 1.0e-6 * dx / dn;
        S.y += 1.0e-6 * dy / dn;
    }
    S.mode = (int)alias_pick(P.gen_tab + (size_t)gi * P.n, (uint32_t)P.n, S.rng, ng);
    S.sign = g.sign;
    S.t = 0.;
    S.bin = 0;
    S.st = RTA_FRESH;
}

// The scattering that ends a flight inside the box draws the next two numbers
// of the stream (alias_pick). They are taken ahead, once per flight, on a copy
// of the generator, and the alias entry is loaded while the flight is
// computed and flown; the copy replaces the generator only on that path, so
// every stream is consumed as without the look-ahead.
template <int TM, bool GL>
__device__ inline void rta_look(const RtaParams& P, const RtaGeo<GL>& G, RtaState& S) {
    Pcg32 r = S.rng;
    S.sk = r.bounded((uint32_t)P.n);
    S.su = r.next();
    S.look = r.state;
    S.se = P.scat[(size_t)(TM == 3 ? G.run : S.run) * (uint32_t)P.n + S.sk];
}

// One event of evolparticle (RTA_MC2D.cpp:990-1386) for lanes in FRESH or FLY:
// the flight draw of the history loop (2262-2288), the segment to the next
// scattering or box side and its tally, the scattering or the crossing into
// the one box that shares the side. What few lanes meet at a time (void
// sides, corners and partly shared sides, periodic boxes) is left to
// rta_slow.
template <bool GRAD, int TM, bool POLY, bool GL, bool D>
__device__ inline void rta_fly(const RtaParams& P, const RtaGeo<GL>& G, const RtaTally& T, TallyAcc<D>& A,
                               RtaState& S, RtaCounts& C) {
    // every history ends: a particle that exceeds the iteration budget or
    // makes 64 events in a row without advancing in time is dropped
    if (++S.budget > (1u << 26) || S.still > 64) {
        atomicAdd(P.counters + 3, 1ULL);
        S.st = RTA_DEAD;
        return;
    }
    if (S.st == RTA_FRESH) {
        // exponential flight, truncated at maxtime
        if (!(S.t < P.maxtime)) {
            S.st = RTA_DEAD;
            return;
        }
        const RtaMode* M = P.rmodes + S.mode;
        const double2 v = make_double2(M->vx, M->vy), iv = make_double2(M->ivx, M->ivy);
        const double w = M->w, iw = M->iw;
        const double u = 1.0 - S.rng.uniform();
        rta_look<TM>(P, G, S);
        S.vx = v.x;
        S.vy = v.y;
        S.ivx = iv.x;
        S.ivy = iv.y;
        // -log u / (w wscale): the quotient from the reciprocal, corrected by
        // its remainder (Markstein), which rounds as the division does
        const double a = -flight_log(G.log, u);
        const double den = w * (TM == 3 ? G.wscale : S.wscale), rec = iw * (TM == 3 ? G.iws : S.iws);
        const double q = a * rec;
        S.dtrem = fma(fma(-q, den, a), rec, q);
        // also where a rate whose reciprocal overflows has left no number
        if (!(S.t + S.dtrem <= P.maxtime)) S.dtrem = P.maxtime - S.t + 1.0e-8;
        if (almost_equal(S.dtrem, 0.)) {
            S.still++;
            return;
        }
        S.st = RTA_FLY;
    }
    const RtaBox B = G.at(S.box);
    if (B.kind != 0) {
        S.still++;
        if (B.kind == 2) {
            S.st = RTA_TRANS;
        } else {  // reservoir: absorbed (RTA_MC2D.cpp:1046-1053)
            C.events++;
            S.st = RTA_DEAD;
        }
        return;
    }
    const double vx = S.vx, vy = S.vy;
    double nx = S.x + S.dtrem * vx, ny = S.y + S.dtrem * vy, step = S.dtrem;
    const int2 sr = make_int2(B.s0, B.ns);
    const bool inside = POLY ? poly_inside(G.side, sr, nx, ny)
                             : (nx >= B.xmin) & (nx <= B.xmax) & (ny >= B.ymin) & (ny <= B.ymax);
    int fast = SIDE_MIXED;
    if (!inside) {
        if constexpr (POLY) {
            int mask;
            step = poly_exit(G.side, sr, S.x, S.y, vx, vy, mask, nx, ny);
            fast = poly_side_fast(G.side, sr, mask, nx, ny, vx, vy, S.aux);
            if (fast == SIDE_MIXED) S.aux = mask;
        } else {
            fast = rect_exit(B, S.x, S.y, vx, vy, S.ivx, S.ivy, step, nx, ny, S.aux);
        }
    }
    tally_segment<GRAD, TM, GL, D>(P, G, T, A, S, B.lrow, S.t + step);
    S.x = nx;
    S.y = ny;
    if (inside) {
        if (!S.ballistic) {
            // alias_pick with the draws taken ahead
            S.mode = S.su < S.se.x ? (int)S.sk : (int)(S.se.y & 0x3fffffffu);
            S.rng.state = S.look;
        }
        C.events++;
        S.st = RTA_FRESH;
        return;
    }
    double left = S.dtrem - step;
    if (almost_equal(left, 0.)) left = 0.;
    S.dtrem = left;
    if (fast >= 0) {
        S.box = fast;
        C.crossings++;
        S.st = left == 0. ? RTA_FRESH : RTA_FLY;
    } else {
        S.st = fast == SIDE_VOID ? RTA_WALL : RTA_MIXED;
    }
}

// The rest of an event for lanes in WALL (a void side reached), MIXED (an exit
// that the general neighbour search decides) or TRANS (a periodic box).
template <bool GRAD, int TM, bool POLY, bool GL>
__device__ inline void rta_slow(const RtaGeo<GL>& G, RtaState& S, RtaCounts& C) {
    const RtaParams& P = rta_cold_params();
    const int abox = S.box + G.bo;  // the box in the batch's arrays
    const double vx = S.vx, vy = S.vy;
    if (S.st == RTA_TRANS) {
        // periodic box: translate, keep the remaining flight (RTA_MC2D.cpp:1034-1043)
        const int nb = POLY ? translate_poly(P.boxes, P.sides, P.srange, P.cts, P.cseg, P.ptrans, abox, S.x, S.y,
                                             vx, vy, S.rng)
                            : translate_rect(P.boxes, P.cross, P.ptrans, abox, S.x, S.y, vx, vy, S.rng);
        if (nb < 0) {
            atomicAdd(P.counters + 5, 1ULL);
            S.st = RTA_DEAD;
            return;
        }
        S.box = nb - G.bo;
        S.st = RTA_FLY;
        rta_look<TM>(P, G, S);  // the translation may have drawn
        return;
    }
    int s = S.aux;
    if (S.st == RTA_MIXED) {
        const int mask = S.aux;
        const DevBox B = P.boxes[abox];
        const int2 sr = POLY ? P.srange[abox] : make_int2(0, 0);
        Ids4 pb{};
        const int npb = POLY ? poly_find_pboxes(P.sides, P.srange, P.cts, B, S.x, S.y, vx, vy, pb)
                             : find_pboxes(P.boxes, P.cts, B, S.x, S.y, vx, vy, pb);
        if (npb > 0) {
            int nbox;
            if (npb == 1) {
                nbox = pb.a;
            } else {
                // several candidate boxes at a corner (RTA_MC2D.cpp:1316-1380)
                Ids4 cand{};
                int nc = 0;
                const double cx = S.x + 1.0e-6 * vx, cy = S.y + 1.0e-6 * vy;
                for (int k = 0; k < npb && k < 4; k++) {
                    const bool in = POLY ? poly_inside(P.sides, P.srange[pb.get(k)], cx, cy)
                                         : box_inside(P.boxes[pb.get(k)], cx, cy);
                    if (in) cand.set(nc++, pb.get(k));
                }
                if (nc > 0) {
                    nbox = cand.get((int)S.rng.bounded((uint32_t)nc));
                } else {
                    nbox = pb.get((int)S.rng.bounded((uint32_t)(npb < 4 ? npb : 4)));
                    double ccx, ccy;
                    if constexpr (POLY) {
                        ccx = P.center[nbox].x;
                        ccy = P.center[nbox].y;
                    } else {
                        const DevBox nb = P.boxes[nbox];
                        ccx = 0.5 * (nb.xmin + nb.xmax);
                        ccy = 0.5 * (nb.ymin + nb.ymax);
                    }
                    double dx = ccx - S.x, dy = ccy - S.y;
                    double dn = sqrt(dx * dx + dy * dy);
                    S.x += 1.0e-6 * dx / dn;
                    S.y += 1.0e-6 * dy / dn;
                }
                rta_look<TM>(P, G, S);  // the choice has drawn
            }
            S.box = nbox - G.bo;
            C.crossings++;
            S.st = S.dtrem == 0. ? RTA_FRESH : RTA_FLY;
            return;
        }
        s = __popc(mask) == 1 ? __ffs(mask) - 1
            : (POLY ? poly_pick_void_side(P.sides, P.srange, P.cts, B, sr, mask, S.x, S.y, S.rng.next())
                    : pick_void_side(P.boxes, P.cts, B, mask, S.x, S.y, S.rng.next()));
    }
    // specular with probability p (mirror partner of the mode), else
    // diffuse; a draw is made only when 0 < p < 1 (polygon runs: diffuse)
    const float p = POLY ? 0.f : P.runs[TM == 3 ? G.run : S.run].spec[s];
    bool specular = p >= 1.f;
    if (p > 0.f && p < 1.f) {
        specular = S.rng.uniform() < (double)p;
        if (GRAD && ((S.gmask >> s) & 1)) {
            // d/dp log P(outcome): 1/p for specular, -1/(1-p) for diffuse
            const float d = specular ? 1.f / p : -1.f / (1.f - p);
            // selects keep the scores in registers
#pragma unroll
            for (int k = 0; k < 4; k++) S.score[k] = s == k ? S.score[k] + d : S.score[k];
        }
    }
    if (specular) {
        const int partner = P.mirror[(s == 0 || s == 3 ? 0 : (size_t)P.n) + S.mode];
        if (partner < 0) {
            atomicAdd(P.counters + 4, 1ULL);
            S.st = RTA_DEAD;
            return;
        }
        S.mode = partner;
    } else {
        // Lambert re-emission (RTA_MC2D.cpp:635-678)
        const RtaMode* M = P.rmodes + S.mode;
        const int lo = M->lo, len = M->len, base = M->base;
        const int tabk = POLY ? P.sides[P.srange[abox].x + s].nid : s;
        bool ng;
        const int k = (int)alias_pick(P.lam_tab + base + (size_t)tabk * len, (uint32_t)len, S.rng, ng);
        S.mode = P.perm[lo + k];
    }
    // the remaining flight is discarded (RTA_MC2D.cpp:1259)
    C.events++;
    S.st = RTA_FRESH;
}

// Histories change waves within a workgroup once the particle ids have run
// out. History lengths are heavy-tailed (a ribbon of 1 um over 5 ns: 160
// events on average, 2900 for a particle that stays to the end), so the waves
// would run on with a few lanes each: 19 of 64 on average over a run of 1e6
// particles, and a pass costs a wave the same with 5 lanes as with 64. A wave
// donates its idle lanes to RtaMig::free. A wave whose live histories fit in
// lanes that other waves donated reserves them, writes the histories to the
// mailbox and ends; waves with idle lanes take them from there. The first
// keep_waves waves of a workgroup (one per SIMD of the CU) never give theirs
// away. A wave leaves with idle lanes only after withdrawing its donation, so
// reserved lanes always exist and every wait ends.
struct RtaMig {
    int32_t free;   // donated idle lanes not reserved
    int32_t lock;   // the mailbox is in use
    int32_t n;      // histories in the mailbox not yet claimed
    int32_t total, read;  // its size and the histories read
    int32_t pad[3];
};
#define RTA_MAIL_WORDS 12
#define RTA_MIG_BYTES (sizeof(RtaMig) + 64 * RTA_MAIL_WORDS * sizeof(uint64_t))
// between barriers; the caller synchronises
__device__ inline void rta_mig_init(const RtaParams& P) {
    if (P.mig >= 0 && threadIdx.x < sizeof(RtaMig) / sizeof(int32_t))
        reinterpret_cast<int32_t*>(rta_lds + P.mig)[threadIdx.x] = 0;
}
__device__ inline int wg_load(const int32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline bool wg_cas(int32_t* p, int& expect, int v) {
    return __hip_atomic_compare_exchange_strong(p, &expect, v, __ATOMIC_ACQ_REL, __ATOMIC_ACQUIRE,
                                                __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline int wg_add(int32_t* p, int v) {
    return __hip_atomic_fetch_add(p, v, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// takes n from *p unless less than n is there (one lane of a wave calls it)
__device__ inline bool wg_take(int32_t* p, int need, int n) {
    int f = wg_load(p);
    while (f >= need)
        if (wg_cas(p, f, f - n)) return true;
    return false;
}

template <bool GRAD>
__device__ inline void rta_mail_write(uint64_t* w, const RtaState& S) {
    auto pair = [](int a, int b) { return (uint64_t)(uint32_t)a | (uint64_t)(uint32_t)b << 32; };
    w[0 * 64] = S.rng.state;
    w[1 * 64] = S.rng.inc;
    w[2 * 64] = (uint64_t)__double_as_longlong(S.x);
    w[3 * 64] = (uint64_t)__double_as_longlong(S.y);
    w[4 * 64] = (uint64_t)__double_as_longlong(S.t);
    w[5 * 64] = (uint64_t)__double_as_longlong(S.dtrem);
    w[6 * 64] = pair(S.mode, S.box);
    w[7 * 64] = pair(S.still, S.st | S.aux << 8);
    w[8 * 64] = pair(S.bin, S.run);
    w[9 * 64] = pair((int)S.budget, (S.sign < 0 ? 1 : 0) | (S.ballistic ? 2 : 0) | S.gmask << 2);
    if (GRAD) {
        w[10 * 64] = pair(__float_as_int(S.score[0]), __float_as_int(S.score[1]));
        w[11 * 64] = pair(__float_as_int(S.score[2]), __float_as_int(S.score[3]));
    }
}
template <bool GRAD, int TM, bool GL>
__device__ inline void rta_mail_read(const RtaParams& P, const RtaGeo<GL>& G, const uint64_t* w, RtaState& S) {
    auto lo = [](uint64_t v) { return (int)(uint32_t)v; };
    auto hi = [](uint64_t v) { return (int)(uint32_t)(v >> 32); };
    S.rng.state = w[0 * 64];
    S.rng.inc = w[1 * 64];
    S.x = __longlong_as_double((long long)w[2 * 64]);
    S.y = __longlong_as_double((long long)w[3 * 64]);
    S.t = __longlong_as_double((long long)w[4 * 64]);
    S.dtrem = __longlong_as_double((long long)w[5 * 64]);
    S.mode = lo(w[6 * 64]);
    S.box = hi(w[6 * 64]);
    S.still = lo(w[7 * 64]);
    S.st = hi(w[7 * 64]) & 255;
    S.aux = hi(w[7 * 64]) >> 8;
    S.bin = lo(w[8 * 64]);
    S.run = hi(w[8 * 64]);
    S.budget = (uint32_t)lo(w[9 * 64]);
    const int f = hi(w[9 * 64]);
    S.sign = (f & 1) ? -1 : 1;
    S.ballistic = (f >> 1) & 1;
    S.gmask = f >> 2;
    if (GRAD) {
        S.score[0] = __int_as_float(lo(w[10 * 64]));
        S.score[1] = __int_as_float(hi(w[10 * 64]));
        S.score[2] = __int_as_float(lo(w[11 * 64]));
        S.score[3] = __int_as_float(hi(w[11 * 64]));
    }
    if (TM != 3) {
        S.wscale = P.runs[S.run].wscale;
        S.iws = 1.0 / S.wscale;
    }
    // of the flight under way: the mode's velocity and the look-ahead
    const RtaMode* M = P.rmodes + S.mode;
    S.vx = M->vx;
    S.vy = M->vy;
    S.ivx = M->ivx;
    S.ivy = M->ivy;
    rta_look<TM>(P, G, S);
}

// How a wave shares `total` particles with `waves` waves. With fewer particles
// than lanes they are spread over all waves (a wave with few lanes skips the
// paths none of them takes, and all SIMDs work); ids are handed out in pieces
// of at most a quarter of a wave's share, so that no wave is left with a
// piece when the others have finished. Histories stay where they are when
// every wave has only a few.
struct RtaShare {
    int lanes;       // lanes that follow histories
    int chunk;       // particle ids taken at a time
    int keep_waves;  // leading waves of the workgroup that keep their histories
};
__device__ inline RtaShare rta_share(unsigned long long total, unsigned waves, int threads) {
    const unsigned long long per = (total + waves - 1) / waves;
    RtaShare W;
    W.lanes = (int)min(64ULL, max(1ULL, per));
    W.chunk = (int)min(64ULL, max(1ULL, per / 4));
    W.keep_waves = W.lanes < 16 ? threads / 64 : max(1, threads / 64 / 3);
    return W;
}

// Follows histories until the ids run out: one particle history per lane at a
// time. Per pass the lanes in FRESH or FLY make one event; the lanes that
// wait (pending sides, ended histories) are served together once an eighth of
// the live lanes wait for a side or RTA_REFILL_MIN for an id, or no lane of the
// wave can fly, so the code of those paths, which a few lanes per pass would
// run with the rest of the wave idle, runs every few passes with more lanes
// in it. take(lo, hi) hands the wave a range of at least one id (ids at or
// past `end` mean that there is none left). Streams are keyed by the
// particle id and kept with the history, so the order of ids and of events
// between lanes changes nothing in any history.
#define RTA_REFILL_MIN 8
template <bool GRAD, int TM, bool POLY, bool GL, bool D, class Take>
__device__ inline void rta_histories(const RtaParams& P, const RtaGeo<GL>& G, const RtaTally& T, RtaCounts& C,
                                     unsigned long long end, RtaShare W, Take take) {
    TallyAcc<D> A;
    RtaState S;
    const int lane = threadIdx.x & 63;
    const unsigned long long below = (1ULL << lane) - 1ULL;
    S.st = lane < W.lanes ? RTA_DEAD : RTA_DONE;
    const auto can_fly = [&S] { return S.st == RTA_FRESH || S.st == RTA_FLY; };
    unsigned long long pool_lo = 0, pool_hi = 0;
    bool exhausted = false;  // no id left
    RtaMig* M = reinterpret_cast<RtaMig*>(rta_lds + P.mig);
    uint64_t* mail = reinterpret_cast<uint64_t*>(rta_lds + P.mig + sizeof(RtaMig));
    const bool may_give = (int)(threadIdx.x >> 6) >= W.keep_waves;
    int donated = 0;
    uint32_t tick = 0;
    for (;;) {
        unsigned long long flying = __ballot(can_fly());
        const unsigned long long pend = __ballot(S.st >= RTA_WALL && S.st <= RTA_TRANS);
        if (pend && 8 * __popcll(pend) >= __popcll(flying | pend)) {
            if ((pend >> lane) & 1ULL) rta_slow<GRAD, TM, POLY, GL>(G, S, C);
            flying = __ballot(can_fly());
        }
        unsigned long long dead = __ballot(S.st == RTA_DEAD);
        if (dead && (!flying || exhausted || __popcll(dead) >= RTA_REFILL_MIN)) {
            unsigned long long pid = ~0ULL;
            while (dead && !exhausted) {
                if (pool_lo == pool_hi) {
                    take(pool_lo, pool_hi);
                    exhausted = pool_lo >= end;
                }
                const unsigned long long rank = (unsigned long long)__popcll(dead & below);
                const unsigned long long n = min((unsigned long long)__popcll(dead), pool_hi - pool_lo);
                const bool mine = (dead >> lane) & 1ULL;
                if (mine && rank < n) pid = pool_lo + rank;
                pool_lo += n;
                dead = __ballot(S.st == RTA_DEAD && pid == ~0ULL);
            }
            if (S.st == RTA_DEAD) {
                if (pid >= end) {
                    S.st = RTA_DONE;
                } else {
                    rta_start<GRAD, TM, POLY, GL>(G, S, pid);
                    // the lane's 32-bit counts: far from wrapping between two particles
                    if ((C.events | C.crossings) & 0x80000000u) {
                        atomicAdd(P.counters + 0, (unsigned long long)C.events);
                        atomicAdd(P.counters + 1, (unsigned long long)C.crossings);
                        C.events = C.crossings = 0;
                    }
                }
            }
            flying = __ballot(can_fly());
        }
        if (exhausted && (!flying || (++tick & 7) == 0)) {
            unsigned long long idle = __ballot(S.st == RTA_DONE);
            if (P.mig < 0) {
                if (idle == ~0ULL) break;
            } else {
                const int nidle = __popcll(idle);
                if (nidle > donated) {
                    if (lane == 0) wg_add(&M->free, nidle - donated);
                    donated = nidle;
                }
                // take histories from the mailbox into idle lanes
                int got = 0, at = 0;
                if (lane == 0 && nidle > 0) {
                    int n = wg_load(&M->n);
                    while (n > 0) {
                        got = min(nidle, n);
                        at = n - got;
                        if (wg_cas(&M->n, n, at)) break;
                        got = 0;
                    }
                }
                got = __builtin_amdgcn_readfirstlane(got);
                if (got > 0) {
                    at = __builtin_amdgcn_readfirstlane(at);
                    const int rank = __popcll(idle & below);
                    if (S.st == RTA_DONE && rank < got)
                        rta_mail_read<GRAD, TM, GL>(P, G, mail + at + rank, S);
                    donated -= got;
                    if (lane == 0) {
                        const int total = M->total;
                        if (wg_add(&M->read, got) + got == total) {
                            M->read = 0;
                            __hip_atomic_store(&M->lock, 0, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
                        }
                    }
                    idle = __ballot(S.st == RTA_DONE);
                    flying = __ballot(can_fly());
                }
                const int alive = 64 - __popcll(idle);
                if (alive == 0) {
                    int ok = 0;
                    if (lane == 0) ok = wg_take(&M->free, donated, donated);
                    if (__builtin_amdgcn_readfirstlane(ok)) break;
                    __builtin_amdgcn_s_sleep(8);  // reserved lanes: their histories are on the way
                    continue;
                }
                // hand the wave's histories over
                if (may_give) {
                    int ok = 0;
                    if (lane == 0) {
                        ok = wg_take(&M->free, donated + alive, donated + alive);
                        int z = 0;
                        if (ok && !wg_cas(&M->lock, z, 1)) {
                            wg_add(&M->free, donated + alive);
                            ok = 0;
                        }
                    }
                    if (__builtin_amdgcn_readfirstlane(ok)) {
                        if (S.st != RTA_DONE) rta_mail_write<GRAD>(mail + __popcll(~idle & below), S);
                        if (lane == 0) {
                            M->total = alive;
                            __hip_atomic_store(&M->n, alive, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
                        }
                        break;
                    }
                }
            }
        }
        if (!flying) {
            if (!exhausted && __ballot(S.st != RTA_DONE) == 0ULL) exhausted = true;  // no lane follows histories
            continue;  // lanes that wait are served in the next pass
        }
        if ((flying >> lane) & 1ULL) rta_fly<GRAD, TM, POLY, GL, D>(P, G, T, A, S, C);
    }
    if constexpr (TM != 1) acc_flush<TM, D>(P, T, A);
}

// Particle ids base + 0, 1, ... from a counter in global memory, `chunk` at a time.
struct RtaTake {
    unsigned long long* next;
    unsigned long long base;
    int chunk;
    __device__ inline void operator()(unsigned long long& lo, unsigned long long& hi) const {
        unsigned long long b = 0;
        if ((threadIdx.x & 63) == 0) b = atomicAdd(next, (unsigned long long)chunk);
        lo = base + __shfl(b, 0, 64);
        hi = lo + chunk;
    }
};

// One launch follows the histories of all runs of a batch; ids of all runs
// form one range, so a batch of runs of any sizes fills the GPU.
// Bound by VALU issue while ids last (a pass was about 400 vector
// instructions, three waves per SIMD) and by the latency of a pass times the
// passes of the longest history after that. 1 um x 200 nm, 100 bins, 200 time
// bins, 3000 modes, 1e6 particles: 16.2 ms with geometry, grid and mode
// arrays read from global memory for every segment (57 scattered loads per
// wave and segment; 15 of 64 lanes active), 10.7 ms with the geometry in LDS,
// the mode in registers and the rare paths deferred, 7.0 ms with histories
// changing waves, 6.2 ms with the exit test in selects, the segment's bins
// found once and the rare paths' parameters read where they are used, 5.65 ms
// with the flight drawn by table and reciprocal (some 330 vector instructions).
template <bool GRAD, int TMK, bool POLY, bool GL>
__global__ __launch_bounds__(TMK ? 768 : 512) void rta_history_kernel(RtaParams P) {
    constexpr bool D = GRAD && TMK == 0;
    const uint64_t xc = xcd_id() % RTA_NCOPY;
    RtaGeo<GL> G;
    G.bo = 0;
    if constexpr (GL) {
        rta_stage_boxes<POLY>(P, rta_lds, 0, P.nboxes, 0, P.nsides, 0);
        rta_stage_grid(P, rta_lds);
        G.box = rta_lds + FLIGHT_LOG_BYTES;
        G.log = reinterpret_cast<const LogEntry*>(rta_lds);
        G.side = reinterpret_cast<const DevSide*>(rta_lds + P.geo_side);
        G.grid = reinterpret_cast<const double*>(rta_lds + P.geo_grid);
    } else {
        G.log = rta_log_table;
        G.box = reinterpret_cast<const unsigned char*>(P.rboxes);
        G.side = P.sides;
        G.grid = P.timegrid;
    }
    RtaTally T;
    T.lds = rta_lds + P.geo_bytes;
    T.row0 = 0;
    T.lbins = (uint32_t)P.lbins;
    T.lc = (TMK == 1 || TMK == 2) ? (uint32_t)P.lrows * (uint32_t)P.lbins : 0u;
    T.g = P.gz + xc * 3 * P.cells;
    T.dg = GRAD ? P.dgz + xc * 4 * P.cells : nullptr;
    uint32_t words = 0;  // 8-byte words of the LDS tallies
    if constexpr (TMK == 1) words = (P.lt_arrays * T.lc + 1) / 2;
    if constexpr (TMK == 2) words = 3 * T.lc;
    for (uint32_t j = threadIdx.x; j < words; j += blockDim.x) ((double*)T.lds)[j] = 0.;
    rta_mig_init(P);
    __syncthreads();
    RtaCounts C;
    const RtaShare W = rta_share(P.total, (unsigned)P.waves, (int)blockDim.x);
    rta_histories<GRAD, TMK, POLY, GL, D>(P, G, T, C, P.total, W,
                                             RtaTake{P.counters + 2, 0, W.chunk});
    if constexpr (TMK == 1) {
        __syncthreads();  // every history of the workgroup has ended
        lt_flush<GRAD>(P, T);
    } else if constexpr (TMK == 2) {
        __syncthreads();  // every lane has added its last cell
        // the workgroup's block, stored whole (rta_sum_parts_kernel adds the
        // blocks of all workgroups)
        const double* g = (const double*)T.lds;
        double* dst = P.part + (size_t)blockIdx.x * words;
        for (uint32_t j = threadIdx.x; j < words; j += blockDim.x) dst[j] = g[j];
    }
    rta_add_counts(P, C);
}

// Tally mode 3: persistent workgroups (768 threads, one per CU) follow one run's
// histories at a time, with the run's boxes, time grid and rows (as many
// leading time bins as fit) in an FP64 LDS block. Ids come from the run's
// counter, so a workgroup stays on its run until every id is taken; once its
// last history has ended, the block is added into the XCD's tally copy and the
// workgroup joins the run with the most particles left per workgroup. Later
// bins go to the copies by device atomics, as under mode 2. A batch whose runs
// each fit a block of their own thus gets LDS sums where one block for all
// runs would not hold a single time bin.
// The wait for the longest history (2900 passes against 160 on average for
// 1 um over 5 ns) is paid once per run that a workgroup follows: 16 runs of
// 3e4 to 1e6 particles took 17.3 ms (15.8 ms now, see flight_log.hpp), against 28.6 ms with the
// ids in items of 4096 or more, each of which ended with that wait.

// The run a workgroup turns to, by its first wave: the first_run entry, then
// the run with the most particles left per workgroup on it, where those fill
// the lanes of one more (or nobody follows it). -1: none is left.
__device__ inline int rta_pick_run(const RtaParams& P, bool first) {
    const int lane = threadIdx.x & 63;
    int run = first ? P.first_run[blockIdx.x] : -1;
    if (run < 0) {
        unsigned long long best = 0;
        for (int r = lane; r < P.nruns; r += 64) {
            const unsigned long long n = P.runs[r].count;
            const unsigned long long at = __hip_atomic_load(P.run_next + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long w = __hip_atomic_load(P.run_wgs + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (at >= n || (w > 0 && n - at < (w + 1) * blockDim.x)) continue;
            const unsigned long long share = (n - at) / (w + 1) + 1;
            if (share > best) {
                best = share;
                run = r;
            }
        }
        for (int d = 32; d > 0; d >>= 1) {
            const unsigned long long b = __shfl_xor(best, d, 64);
            const int r = __shfl_xor(run, d, 64);
            if (b > best || (b == best && r > run)) {
                best = b;
                run = r;
            }
        }
    }
    if (run >= 0 && lane == 0) atomicAdd(P.run_wgs + run, 1ULL);
    return run;
}

template <bool POLY, bool GL>
__global__ __launch_bounds__(768) void rta_history_runs_kernel(RtaParams P) {
    __shared__ int picked;
    const uint64_t xc = xcd_id() % RTA_NCOPY;
    if constexpr (GL) rta_stage_grid(P, rta_lds);
    double* L = reinterpret_cast<double*>(rta_lds + P.geo_bytes);
    RtaCounts C;
    for (bool first = true;; first = false) {
        __syncthreads();  // the previous run's block has been read
        if (threadIdx.x < 64) {
            const int r = rta_pick_run(P, first);
            if (threadIdx.x == 0) picked = r;
        }
        __syncthreads();
        const int run = __builtin_amdgcn_readfirstlane(picked);
        if (run < 0) break;
        // the run's fields as uniform scalars
        const RtaRunRows& I = P.rows[run];
        const uint32_t lbins = (uint32_t)I.lbins, lrow0 = (uint32_t)I.lrow0;
        const uint32_t lc = (uint32_t)I.lrows * lbins, nf = 3u * lc;
        const unsigned long long count = P.runs[run].count, first_id = P.runs[run].first;
        RtaGeo<GL> G;
        G.bo = I.box0;
        G.run = run;
        G.wscale = P.runs[run].wscale;
        G.iws = 1.0 / G.wscale;
        if constexpr (GL) {
            rta_stage_boxes<POLY>(P, rta_lds, I.box0, I.nbox, I.side0, I.nsides, (int)lrow0);
            G.box = rta_lds + FLIGHT_LOG_BYTES;
            G.log = reinterpret_cast<const LogEntry*>(rta_lds);
            G.side = reinterpret_cast<const DevSide*>(rta_lds + P.geo_side);
            G.grid = reinterpret_cast<const double*>(rta_lds + P.geo_grid);
        } else {
            // global boxes keep the batch's indices
            G.bo = 0;
            G.log = rta_log_table;
            G.box = reinterpret_cast<const unsigned char*>(P.rboxes);
            G.side = P.sides;
            G.grid = P.timegrid;
        }
        RtaTally T;
        T.lds = L;
        T.row0 = GL ? 0 : (int32_t)lrow0;  // staged records hold the run's own rows
        T.lbins = lbins;
        T.lc = lc;
        T.g = P.gz + xc * 3 * P.cells + (GL ? (uint64_t)I.box0 * (uint64_t)P.nt : 0);
        T.dg = nullptr;
        for (uint32_t j = threadIdx.x; j < nf; j += blockDim.x) L[j] = 0.;
        rta_mig_init(P);
        __syncthreads();
        // a workgroup that begins with the run takes its share of the
        // particles, one that joins fills its lanes
        const RtaShare W = rta_share(count, first ? (unsigned)I.wgs * (blockDim.x / 64) : 1u, (int)blockDim.x);
        rta_histories<false, 3, POLY, GL, false>(P, G, T, C, first_id + count, W,
                                                 RtaTake{P.run_next + run, first_id, W.chunk});
        __syncthreads();  // every history of the run has ended and added its last cell
        for (uint32_t j = threadIdx.x; j < nf; j += blockDim.x) {
            const double v = L[j];
            if (v == 0.) continue;
            const uint32_t a = j / lc, r = j - a * lc, row = r / lbins;
            const uint64_t cell = P.lrow_cell[lrow0 + row] + (r - row * lbins);
            atomicAdd(P.gz + xc * 3 * P.cells + (uint64_t)a * P.cells + cell, v);
        }
        if (threadIdx.x == 0) atomicAdd(P.run_wgs + run, ~0ULL);  // - 1
    }
    rta_add_counts(P, C);
}

// clears the tallies and counters (a kernel rather than a memset so that the
// launch sequence can be captured in a graph)
__global__ __launch_bounds__(256) void rta_clear_kernel(double* a, uint64_t n, unsigned long long* cnt,
                                                       int ncnt) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        a[i] = 0.;
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < ncnt; i += blockDim.x) cnt[i] = 0ULL;
}

// running sum over the time bins of every (location, mode) column: the step
// response, taken before the spectral products (they commute)
__global__ __launch_bounds__(256) void rta_spec_cumsum_kernel(double* S, int nloc, int nt, int n) {
    const uint64_t col = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= (uint64_t)nloc * n) return;
    double* p = S + (col / n) * (uint64_t)nt * n + col % n;
    double acc = 0.;
    for (int t = 0; t < nt; t++) {
        acc += p[(size_t)t * n];
        p[(size_t)t * n] = acc;
    }
}

// Tally mode 2: the LDS blocks of all workgroups, part[blk][3][lrows][lbins],
// summed per cell and added into copy 0 of the tallies (cells of the first
// lbins time bins receive no device atomics, so the add is a plain store).
// Each workgroup sums 32 neighbouring cells (256 bytes of every block) with 16
// threads per cell: one thread per cell left most CUs idle behind a chain of
// 256 to 512 loads (3000 cells of 512 blocks: 123 us, now 5.1 us; 19200
// cells of 256: 77 us, now 9.8 us).
#define RTA_SUM_CELLS 32
__global__ __launch_bounds__(512) void rta_sum_parts_kernel(double* tally, const double* part, int nblk,
                                                            uint32_t lrows, uint32_t lbins,
                                                            const uint64_t* lrow_cell, uint64_t cells) {
    constexpr int NG = 512 / RTA_SUM_CELLS;
    __shared__ double sum[NG][RTA_SUM_CELLS];
    const uint32_t lc = lrows * lbins, nf = 3u * lc;
    const uint32_t q = threadIdx.x % RTA_SUM_CELLS, g = threadIdx.x / RTA_SUM_CELLS;
    const uint32_t j = blockIdx.x * RTA_SUM_CELLS + q;
    double v = 0.;
    if (j < nf) {
#pragma unroll 8
        for (int b = (int)g; b < nblk; b += NG) v += part[(size_t)b * nf + j];
    }
    sum[g][q] = v;
    __syncthreads();
    if (g == 0 && j < nf) {
        for (int k = 1; k < NG; k++) v += sum[k][q];
        const uint32_t a = j / lc, r = j - a * lc, row = r / lbins;
        tally[(uint64_t)a * cells + lrow_cell[row] + (r - row * lbins)] += v;
    }
}

// a[i] = sum over the RTA_NCOPY copies a[x n + i], for i < n
__global__ __launch_bounds__(256) void rta_sum_copies_kernel(double* a, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        double v = a[i];
        for (int x = 1; x < RTA_NCOPY; x++) v += a[(uint64_t)x * n + i];
        a[i] = v;
    }
}

struct RtaBatch {
    Ctx* ctx = nullptr;
    const Modes* m = nullptr;
    std::vector<bte_rta_run_desc> desc;
    std::vector<const Geom*> geoms;
    double thickness = 1, dt = 1, maxtime = 1, sigma = 0.25;
    int ntime = 0, nruns = 0;
    std::vector<double> timegrid;
    std::vector<double> Eeff, cv;
    std::vector<int> box0, nbox;
    std::vector<uint64_t> cell0;   // first tally cell of each run
    uint64_t cells = 0, total = 0;
    bool any_grad = false;
    bool poly = false;  // some run's geometry has polygon boxes: POLY kernels
    std::vector<RtaRunDev> runs;
    DevBuf<DevSide> d_sides;
    DevBuf<int2> d_srange;
    DevBuf<double2> d_center;
    DevBuf<RtaMode> d_rmodes;
    DevBuf<RtaBox> d_rboxes;
    DevBuf<int32_t> d_mirror, d_perm;
    DevBuf<uint2> d_scat, d_gen_sel, d_gen_tab, d_lam_tab;
    DevBuf<RtaGen> d_gens;
    DevBuf<DevBox> d_boxes;
    DevBuf<DevContact> d_cts;
    DevBuf<double4> d_cseg;
    DevBuf<DevCross> d_cross;
    DevBuf<double2> d_ptrans;
    DevBuf<double> d_timegrid, d_tally, d_dgz;
    DevBuf<RtaRunDev> d_runs, d_trial_runs;
    DevBuf<unsigned long long> d_counters;
    // spectral decomposition (one run): locations, per-mode tallies, the
    // weight matrix [n][3 nomega + nq] and the products [nloc][nt][ncols]
    int nloc = 0, nomega = 0, ncols = 0;
    std::vector<int32_t> spec_boxes;
    std::vector<double> omegagrid, spec_host;
    DevBuf<int32_t> d_box_loc;
    DevBuf<double> d_spec, d_specw, d_specout;
    int block = 256, blocks = 0;
    // tally: 0 FP64 device atomics into per-XCD copies; 1 FP32 per-workgroup
    // partial sums in LDS (one 768-thread workgroup per CU), added in FP64;
    // 2 FP64 per-workgroup partial sums of the first lbins time bins in LDS
    // (one 768-thread workgroup per CU), later bins by device atomics
    int tally = 0, lt_goff[4] = {-1, -1, -1, -1};
    uint32_t lrows = 0;
    int lt_arrays = 3;            // mode 1: FP32 arrays
    int nboxes = 0, nsides = 0;   // over all runs
    std::vector<int> side0, nside;  // per run: first polygon side and sides
    DevBuf<uint64_t> d_lrow_cell;
    DevBuf<double> d_part;  // mode 2: [blocks][3][lrows][lbins]
    // 3: per run, the first LDS row and the rows of its regular boxes; their
    // device records, the run each workgroup begins with and the LDS bytes
    std::vector<int32_t> run_lrow0, run_lrows;
    DevBuf<RtaRunRows> d_rows;
    DevBuf<int32_t> d_first_run;
    size_t l3_bytes = 0;
    int l3_nbox = 0, l3_nside = 0;  // boxes and sides of the largest run
    bool l3_mail = true;
    bool use_graph = false;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    ~RtaBatch() {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        if (ev0) (void)hipEventDestroy(ev0);
        if (ev1) (void)hipEventDestroy(ev1);
    }
};

static void upload_alias(DevBuf<uint2>& buf, const std::vector<uint32_t>& th,
                         const std::vector<uint32_t>& al, hipStream_t s) {
    std::vector<uint2> v(th.size());
    for (size_t i = 0; i < th.size(); i++) v[i] = make_uint2(th[i], al[i]);
    buf.upload(v, s);
}

// Lambert tables (RTA_MC2D.cpp:556-626): for mode i the partners f are the
// modes with nonzero omega within nsigma * hypot(sigma_i, sigma_f) in omega,
// weighted for each outward side normal n of the geometry (the four sides of
// rectangles; table k of a mode for normal k) by max(-n.v_f, 0) times the normal pdf of
// omega_i - omega_f with width hypot(sigma_i, sigma_f). sigma_i is the mode
// table's per-mode broadening (base_sigma of a q-grid) raised to the floor
// exp(p25 - 1.5 (p75 - p25)) of log sigma (RTA_MC2D.cpp:566-576), or the
// constant sigma for every mode when the table has none. The partners of i
// lie in one contiguous window of the omega-sorted order (the window of the
// widest pair); pairs outside their own cut get weight 0.
// The windows and the pairs' normal pdf are computed here, the rest, for every
// normal and mode, by rta_lambert_kernel into tab.
struct RtaLambert {
    const int4* info;
    const int32_t* perm;
    const double *omega, *vx, *vy;
    const double2* normals;
    const double* e;    // per pair from mode i0 on: the pdf's exponential, 0 outside the cut
    const double* pre;  // its factor 1 / (sigma sqrt(2 pi)), 0 outside the cut, with per-mode sigma, else null
    double* q;          // scratch: scaled weights and the two stacks, per entry
    int32_t* list;
    uint2* tab;
    unsigned long long* err;  // least 2 (mode, normal) + kind of an error
    int32_t nn, i0, ni;
};
// One lane per mode and normal: the weights of the window and their alias
// table, step by step as build_alias makes it (no contraction, sums in
// ascending order: the same bits). Bound by the chain of dependent loads and
// stores of a lane. On the host these tables were most of making a run: 5.1
// ms for 1000 modes, 42 ms for 3000 and 119 ms for 5000 (sigma 0.5 rad/ps,
// four normals), now 1.6, 4.6 and 12 ms.
__global__ __launch_bounds__(64) void rta_lambert_kernel(RtaLambert L) {
#pragma clang fp contract(off)
    const int t = (int)(blockIdx.x * 64 + threadIdx.x);
    if (t >= L.ni * L.nn) return;
    const int i = L.i0 + t % L.ni, u = t / L.ni;
    const int4 I = L.info[i];
    const int lo = I.x, len = I.y;
    const int base0 = L.info[L.i0].z;
    const size_t row = (size_t)I.z + (size_t)u * len, srow = row - base0;
    const size_t pair = (size_t)(I.z - base0) / L.nn;
    const double nx = L.normals[u].x, ny = L.normals[u].y;
    double* q = L.q + srow;
    int32_t* list = L.list + srow;
    uint2* tab = L.tab + row;
    const auto fail = [&](int kind) { atomicMin(L.err, 2ull * ((unsigned long long)i * L.nn + u) + kind); };
    double tot = 0.;
    int self = 0;
    for (int k = 0; k < len; k++) {
        const int f = L.perm[lo + k];
        const double vn = -(nx * L.vx[f] + ny * L.vy[f]);
        double w = 0.;
        if (!(vn < 0. || almost_equal(vn, 0.))) {
            w = vn * L.e[pair + k];
            if (L.pre) w = w * L.pre[pair + k];
        }
        if (!(w >= 0.)) return fail(0);
        if (f == i) self = k;
        tot += w;
        q[k] = w;
    }
    if (!(tot > 0.)) {
        // a mode that can reach this side needs a partner leaving it
        if (nx * L.vx[i] + ny * L.vy[i] > 0. && !almost_equal(0., L.omega[i])) return fail(1);
        for (int k = 0; k < len; k++) tab[k] = make_uint2(0u, (uint32_t)self);
        return;
    }
    // two stacks in one array: below 1 from its front, the others from its end
    int ns = 0, nl = 0;
    for (int k = 0; k < len; k++) {
        const double v = q[k] * len / tot;
        q[k] = v;
        if (v < 1.0) list[ns++] = k;
        else list[len - 1 - nl++] = k;
    }
    if (nl > 0) {
        int l = list[len - nl];
        double ql = q[l];
        while (ns > 0) {
            const int a = list[--ns];
            const double qs = q[a];
            const double x = ldexp(qs, 32);
            tab[a] = make_uint2(x >= 4294967295.0 ? 0xffffffffu : (uint32_t)llround(x), (uint32_t)l);
            ql = (ql + qs) - 1.0;
            if (ql < 1.0) {
                q[l] = ql;
                nl--;
                list[ns++] = l;
                if (nl == 0) break;
                l = list[len - nl];
                ql = q[l];
            }
        }
    }
    for (int k = 0; k < nl; k++) {
        const int l = list[len - 1 - k];
        tab[l] = make_uint2(0xffffffffu, (uint32_t)l);
    }
    for (int k = 0; k < ns; k++) tab[list[k]] = make_uint2(0xffffffffu, (uint32_t)list[k]);
}
// entries of scratch at a time (12 bytes each)
#define RTA_LAMBERT_ENTRIES ((size_t)1 << 24)

static void build_lambert(const Modes& m, double sigma, const std::vector<double2>& normals, std::vector<int4>& info,
                          DevBuf<uint2>& tab, DevBuf<int32_t>& d_perm, hipStream_t s) {
    const double nsig = 2.828427124746190097603377448419396157138;
    const double rt2pi = 2.506628274631000502415765284811045253;
    int n = m.n;
    std::vector<double> bs(n, sigma);
    if (!m.sigma.empty()) {
        std::vector<double> ls(n);
        for (int i = 0; i < n; i++) ls[i] = m.sigma[i] == 0. ? std::numeric_limits<double>::lowest() : std::log(m.sigma[i]);
        std::sort(ls.begin(), ls.end());
        const double p0 = ls[25 * (size_t)n / 100], p1 = ls[75 * (size_t)n / 100];
        const double lb = std::exp(p0 - 1.5 * (p1 - p0));
        for (int i = 0; i < n; i++) bs[i] = std::max(m.sigma[i], lb);
    }
    const double bmax = *std::max_element(bs.begin(), bs.end());
    std::vector<int32_t> perm(n);
    std::iota(perm.begin(), perm.end(), 0);
    std::stable_sort(perm.begin(), perm.end(), [&](int a, int b) { return m.omega[a] < m.omega[b]; });
    std::vector<double> sw(n);
    for (int k = 0; k < n; k++) sw[k] = m.omega[perm[k]];
    info.assign(n, make_int4(0, 0, 0, 0));
    const size_t nn = normals.size();
    size_t entries = 0;
    for (int i = 0; i < n; i++) {
        double oi = m.omega[i];
        const double cut = nsig * std::hypot(bs[i], bmax);
        int lo = (int)(std::lower_bound(sw.begin(), sw.end(), oi - cut) - sw.begin());
        int hi = (int)(std::upper_bound(sw.begin(), sw.end(), oi + cut) - sw.begin());
        // the float window edges may admit a partner just outside |d| <= cut
        while (lo < hi && std::fabs(oi - sw[lo]) > cut) lo++;
        while (hi > lo && std::fabs(oi - sw[hi - 1]) > cut) hi--;
        int len = hi - lo;
        if (len <= 0) throw Error(BTE_EINVAL, "empty Lambert window");
        info[i] = make_int4(lo, len, (int)entries, 0);
        entries += nn * (size_t)len;
    }
    DevBuf<int4> d_info;
    DevBuf<double2> d_normals;
    DevBuf<double> d_e, d_pre, d_q;
    DevBuf<int32_t> d_list;
    DevBuf<unsigned long long> d_err;
    const std::vector<unsigned long long> none(1, ~0ull);
    std::vector<unsigned long long> err(1);
    tab.alloc(entries);
    d_perm.upload(perm, s);
    d_info.upload(info, s);
    d_normals.upload(normals, s);
    d_err.upload(none, s);
    const bool own = !m.sigma.empty();
    const double sig0 = std::hypot(sigma, sigma);
    std::vector<double> e, pre;
    for (int i0 = 0, i1; i0 < n; i0 = i1) {
        size_t part = 0;
        e.clear();
        pre.clear();
        for (i1 = i0; i1 < n && (i1 == i0 || part + nn * info[i1].y <= RTA_LAMBERT_ENTRIES); i1++) {
            const double oi = m.omega[i1];
            for (int k = 0; k < info[i1].y; k++) {
                const int f = perm[info[i1].x + k];
                const double sig = own ? std::hypot(bs[i1], bs[f]) : sig0;
                const double d = std::fabs(oi - m.omega[f]);
                const bool ok = !almost_equal(0., m.omega[f]) && d <= nsig * sig;
                e.push_back(ok ? std::exp(-0.5 * d * d / (sig * sig)) : 0.);
                // the pdf's 1 / (sig sqrt(2 pi)) differs between pairs only with per-mode sigma
                // (a pair of weight 0 may have width 0)
                if (own) pre.push_back(ok ? 1.0 / (sig * rt2pi) : 0.);
            }
            part += nn * info[i1].y;
        }
        d_e.upload(e, s);
        if (own) d_pre.upload(pre, s);
        if (d_q.n < part) d_q.alloc(part);
        if (d_list.n < part) d_list.alloc(part);
        const RtaLambert L{d_info.p, d_perm.p, m.d_omega.p, m.d_vx.p, m.d_vy.p, d_normals.p, d_e.p, own ? d_pre.p : nullptr,
                           d_q.p, d_list.p, tab.p, d_err.p, (int32_t)nn, i0, i1 - i0};
        hipLaunchKernelGGL(rta_lambert_kernel, dim3((unsigned)(((size_t)(i1 - i0) * nn + 63) / 64)), dim3(64), 0, s, L);
        HIPCHECK(hipGetLastError());
        if (i1 < n) HIPCHECK(hipStreamSynchronize(s));  // e is refilled
    }
    HIPCHECK(hipMemcpyAsync(err.data(), d_err.p, sizeof(err[0]), hipMemcpyDeviceToHost, s));
    HIPCHECK(hipStreamSynchronize(s));
    if (err[0] != ~0ull) {
        if ((err[0] & 1) == 0) throw Error(BTE_EINVAL, "probabilities must be >= 0.");
        throw Error(BTE_EINVAL, "mode " + std::to_string(err[0] / 2 / nn) +
                                    " has no diffuse partner within the Lambert window; raise sigma_bounce");
    }
}


// mirror partners: same omega and |v| components with one velocity
// component negated (exact float match), -1 where there is none
static void build_mirrors(const Modes& m, std::vector<int32_t>& mir) {
    const int n = m.n;
    mir.assign(2 * (size_t)n, -1);
    std::map<std::tuple<double, double, double>, int> idx;
    for (int i = 0; i < n; i++) idx.emplace(std::make_tuple(m.omega[i], m.vx[i], m.vy[i]), i);
    for (int i = 0; i < n; i++) {
        auto a = idx.find(std::make_tuple(m.omega[i], -m.vx[i], m.vy[i]));
        auto b = idx.find(std::make_tuple(m.omega[i], m.vx[i], -m.vy[i]));
        if (a != idx.end()) mir[i] = a->second;
        if (b != idx.end()) mir[(size_t)n + i] = b->second;
    }
}

static RtaParams batch_params(RtaBatch* b, const RtaRunDev* runs, uint64_t total) {
    RtaParams P{};
    P.rmodes = b->d_rmodes.p;
    P.rboxes = b->d_rboxes.p;
    P.mirror = b->d_mirror.p;
    P.scat = b->d_scat.p;
    P.boxes = b->d_boxes.p;
    P.cts = b->d_cts.p;
    P.cseg = b->d_cseg.p;
    P.cross = b->d_cross.p;
    P.ptrans = b->d_ptrans.p;
    P.sides = b->d_sides.p;
    P.srange = b->d_srange.p;
    P.center = b->d_center.p;
    P.gens = b->d_gens.p;
    P.gen_sel = b->d_gen_sel.p;
    P.gen_tab = b->d_gen_tab.p;
    P.lam_tab = b->d_lam_tab.p;
    P.perm = b->d_perm.p;
    P.timegrid = b->d_timegrid.p;
    P.runs = runs;
    P.gz = b->d_tally.p;
    P.jx = b->d_tally.p + b->cells;
    P.jy = b->d_tally.p + 2 * b->cells;
    P.dgz = b->any_grad ? b->d_dgz.p : nullptr;
    P.box_loc = b->nloc ? b->d_box_loc.p : nullptr;
    P.spec = b->nloc ? b->d_spec.p : nullptr;
    P.counters = b->d_counters.p;
    P.total = total;
    P.cells = b->cells;
    P.maxtime = b->maxtime;
    P.n = b->m->n;
    P.nt = b->ntime - 1;
    P.nruns = b->nruns;
    P.lrow_cell = b->d_lrow_cell.p;
    P.lrows = (int32_t)b->lrows;
    for (int k = 0; k < 4; k++) P.lt_goff[k] = b->lt_goff[k];
    P.lt_arrays = b->lt_arrays;
    P.nboxes = b->nboxes;
    P.nsides = b->nsides;
    P.part = b->d_part.p;
    P.idt = (double)(b->ntime - 1) / b->maxtime;
    P.rows = b->d_rows.p;
    P.first_run = b->d_first_run.p;
    P.run_next = b->d_counters.p + 8;
    P.run_wgs = P.run_next + b->nruns;
    return P;
}

// LDS of a workgroup of the history kernels: the geometry and the time grid
// when they take at most RTA_GEO_LDS bytes (see RtaGeo), then the tallies. (The
// 2 KB of the logarithm's table beside such a geometry, at most 256 boxes,
// never take a time bin's last room.)
struct RtaLds {
    bool gl = false;
    int32_t side = 0, grid = 0, geo = 0;  // byte offsets: sides, grid, tallies
    int32_t mig = -1;                     // of the mailbox, before the tallies
    uint32_t lbins = 0;                   // leading time bins of a tally row
    size_t bytes = 0;
};
static RtaLds rta_lds_layout(int nboxes, int nsides, int nt) {
    RtaLds L;
    auto up16 = [](size_t v) { return (v + 15) & ~(size_t)15; };
    const size_t side = FLIGHT_LOG_BYTES + (size_t)RTA_BOX_LDS * nboxes, grid = up16(side + sizeof(DevSide) * (size_t)nsides);
    const size_t geo = up16(grid + sizeof(double) * ((size_t)nt + 1));
    L.gl = geo <= FLIGHT_LOG_BYTES + RTA_GEO_LDS;
    if (L.gl) {
        L.side = (int32_t)side;
        L.grid = (int32_t)grid;
        L.geo = (int32_t)geo;
    }
    L.mig = L.geo;
    L.geo += (int32_t)RTA_MIG_BYTES;
    L.bytes = std::max<size_t>((size_t)L.geo, 16 * 2 * sizeof(uint64_t));  // rta_add_counts' space
    return L;
}
// without the mailbox, where it would leave no room for one time bin
static void drop_mail(RtaLds& L) {
    L.geo = L.mig;
    L.mig = -1;
}
// layout of tally modes 0, 1 and 2: rows of `arrays` tallies of `width`
// bytes per bin, as many leading time bins as the workgroup's LDS holds (the
// early bins carry most of the segments: particles enter at t = 0 and leave
// through the reservoirs)
static RtaLds rta_lds_of(const RtaBatch* b, int tally) {
    const int nt = b->ntime - 1;
    RtaLds L = rta_lds_layout(b->nboxes, b->nsides, nt);
    if ((tally == 1 || tally == 2) && b->lrows) {
        const size_t arrays = tally == 1 ? (size_t)b->lt_arrays : 3, width = tally == 1 ? sizeof(float) : sizeof(double);
        const size_t per_bin = arrays * b->lrows * width;
        if ((size_t)L.geo + per_bin > b->ctx->lds_per_block) drop_mail(L);
        L.lbins = (uint32_t)std::min<size_t>((size_t)nt, (b->ctx->lds_per_block - (size_t)L.geo) / per_bin);
        L.bytes = std::max<size_t>(L.bytes, ((size_t)L.geo + per_bin * L.lbins + 7) & ~(size_t)7);
    }
    return L;
}
static void set_lds(RtaParams& P, const RtaLds& L) {
    P.geo_side = L.side;
    P.geo_grid = L.grid;
    P.geo_bytes = L.geo;
    P.mig = L.mig;
    P.lbins = (int32_t)L.lbins;
}
// waves that run at a time: a CU holds 12 of these kernels (at most 168 registers)
static int32_t share_waves(int block, int blocks, int cus) { return std::min(blocks * (block / 64), 12 * cus); }

using RtaKernel = void (*)(RtaParams);
// the history kernel of a tally mode (0, 1 or 2) by [polygons][geometry in LDS]
static RtaKernel rta_kernel(int tally, bool grad, bool poly, bool gl) {
    static const RtaKernel plain[3][2][2] = {
        {{rta_history_kernel<false, 0, false, false>, rta_history_kernel<false, 0, false, true>},
         {rta_history_kernel<false, 0, true, false>, rta_history_kernel<false, 0, true, true>}},
        {{rta_history_kernel<false, 1, false, false>, rta_history_kernel<false, 1, false, true>},
         {rta_history_kernel<false, 1, true, false>, rta_history_kernel<false, 1, true, true>}},
        {{rta_history_kernel<false, 2, false, false>, rta_history_kernel<false, 2, false, true>},
         {rta_history_kernel<false, 2, true, false>, rta_history_kernel<false, 2, true, true>}}};
    // rectangles only (specular sides)
    static const RtaKernel with_grad[2][2] = {
        {rta_history_kernel<true, 0, false, false>, rta_history_kernel<true, 0, false, true>},
        {rta_history_kernel<true, 1, false, false>, rta_history_kernel<true, 1, false, true>}};
    return grad ? with_grad[tally][gl] : plain[tally][poly][gl];
}
static RtaKernel rta_runs_kernel(bool poly, bool gl) {
    return poly ? (gl ? rta_history_runs_kernel<true, true> : rta_history_runs_kernel<true, false>)
                : (gl ? rta_history_runs_kernel<false, true> : rta_history_runs_kernel<false, false>);
}
static void allow_lds(RtaKernel k, size_t bytes) {
    HIPCHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
}

static void launch_batch(RtaBatch* b, RtaParams P, int block, int blocks, hipStream_t s) {
    hipLaunchKernelGGL(rta_clear_kernel, dim3(1024), dim3(256), 0, s, b->d_tally.p, RTA_NCOPY * 3 * b->cells,
                       b->d_counters.p, 8 + 2 * b->nruns);
    if (b->any_grad)
        hipLaunchKernelGGL(rta_clear_kernel, dim3(1024), dim3(256), 0, s, b->d_dgz.p, RTA_NCOPY * 4 * b->cells,
                           b->d_counters.p, 0);
    if (b->nloc)
        hipLaunchKernelGGL(rta_clear_kernel, dim3(1024), dim3(256), 0, s, b->d_spec.p,
                           (uint64_t)b->nloc * (b->ntime - 1) * b->m->n, b->d_counters.p, 0);
    P.waves = share_waves(block, blocks, b->ctx->cu_count);
    if (b->tally == 3) {
        RtaLds L = rta_lds_layout(b->l3_nbox, b->l3_nside, b->ntime - 1);
        if (!b->l3_mail) drop_mail(L);
        set_lds(P, L);
        hipLaunchKernelGGL(rta_runs_kernel(b->poly, L.gl), dim3(blocks), dim3(block), b->l3_bytes, s, P);
    } else {
        const RtaLds L = rta_lds_of(b, b->tally);
        set_lds(P, L);
        hipLaunchKernelGGL(rta_kernel(b->tally, b->any_grad, b->poly, L.gl), dim3(blocks), dim3(block), L.bytes, s, P);
        if (b->tally == 2) {
            const uint32_t nf = 3u * b->lrows * L.lbins;
            hipLaunchKernelGGL(rta_sum_parts_kernel, dim3((nf + RTA_SUM_CELLS - 1) / RTA_SUM_CELLS), dim3(512), 0, s,
                               b->d_tally.p, b->d_part.p, blocks, b->lrows, L.lbins, b->d_lrow_cell.p, b->cells);
        }
    }
    // the per-XCD copies into copy 0
    hipLaunchKernelGGL(rta_sum_copies_kernel, dim3(1024), dim3(256), 0, s, b->d_tally.p, 3 * b->cells);
    if (b->any_grad)
        hipLaunchKernelGGL(rta_sum_copies_kernel, dim3(1024), dim3(256), 0, s, b->d_dgz.p, 4 * b->cells);
}

static void batch_create(RtaBatch* b) {
    Ctx* c = b->ctx;
    const Modes* m = b->m;
    const int n = m->n;
    hipStream_t s = c->stream;
    if (!(b->dt > 0) || !(b->maxtime > 0) || !(b->thickness > 0)) throw Error(BTE_EINVAL, "bad RTA configuration");
    for (int i = 0; i < n; i++)
        if (m->w[i] == 0.) throw Error(BTE_EINVAL, "invalid scattering rate");
    // time grid (RTA_MC2D.cpp:2121-2124)
    b->ntime = (int)std::floor(b->maxtime / b->dt + 1.0e-6) + 1;
    if (b->ntime < 2) throw Error(BTE_EINVAL, "maxtime shorter than dt");
    b->maxtime = (b->ntime - 1) * b->dt;
    b->timegrid.resize(b->ntime);
    for (int i = 0; i < b->ntime; i++) b->timegrid[i] = (double)i * b->maxtime / (b->ntime - 1);
    const int nt = b->ntime - 1;
    std::vector<int32_t> mir;
    build_mirrors(*m, mir);
    b->d_mirror.upload(mir, s);
    const double vuc = m->V * b->thickness / m->lattz;
    std::vector<DevBox> boxes;
    std::vector<DevContact> cts;
    std::vector<double4> cseg;
    std::vector<DevCross> cross;
    std::vector<double2> ptrans;
    std::vector<uint64_t> lrow_cell;
    std::vector<RtaBox> rboxes;
    std::vector<RtaGen> gens;
    std::vector<uint2> gsel, gtab, scat;
    std::vector<double> pmf(n);
    std::vector<uint32_t> th(n), al(n);
    // polygon geometries: the sides of every run's boxes, their ranges and
    // centres, and the distinct outward normals of the batch (one Lambert
    // table per normal and mode); rectangles use the four axis normals
    std::vector<DevSide> sides;
    std::vector<int2> srange;
    std::vector<double2> center, normals;
    b->poly = false;
    for (const Geom* g : b->geoms) b->poly = b->poly || (g && g->poly);
    if (!b->poly)
        for (int k = 0; k < 4; k++) {
            double nx, ny;
            side_normal(k, nx, ny);
            normals.push_back(make_double2(nx, ny));
        }
    b->nruns = (int)b->desc.size();
    b->total = 0;
    b->cells = 0;
    for (int r = 0; r < b->nruns; r++) {
        const bte_rta_run_desc& D = b->desc[r];
        const Geom* g = b->geoms[r];
        if (!g || D.nparticles == 0) throw Error(BTE_EINVAL, "run " + std::to_string(r) + ": no geometry or particles");
        if (!(D.wscale > 0)) throw Error(BTE_EINVAL, "run " + std::to_string(r) + ": wscale must be positive");
        const int nb = (int)g->boxes.size();
        for (auto& bx : g->boxes)
            if (bx.kind == 0) {
                if (bx.Teq != D.T0) throw Error(BTE_EINVAL, "Tref in xml is different from provided T0");
                if (bx.Tinit != bx.Teq) throw Error(BTE_EINVAL, "Initial temperature out of reference is not allowed");
            }
        RtaRunDev R{};
        R.first = b->total;
        R.count = D.nparticles;
        R.seed = D.seed;
        R.ballistic = D.ballistic ? 1 : 0;
        R.wscale = D.wscale;
        for (int k = 0; k < 4; k++) {
            if (!(D.specularity[k] >= 0. && D.specularity[k] <= 1.))
                throw Error(BTE_EINVAL, "specularity must lie in [0, 1]");
            R.spec[k] = (float)D.specularity[k];
            if (D.grad && D.specularity[k] > 0. && D.specularity[k] < 1.) R.gmask |= 1 << k;
            if (b->poly && (D.specularity[k] > 0. || D.grad))
                throw Error(BTE_EINVAL, "specular sides and dT/dp need rectangular boxes (diffuse sides only on polygons)");
        }
        if (R.gmask) b->any_grad = true;
        const int bo = (int)boxes.size(), co = (int)cts.size();
        b->box0.push_back(bo);
        b->nbox.push_back(nb);
        b->cell0.push_back(b->cells);
        b->run_lrow0.push_back((int32_t)b->lrows);
        b->side0.push_back((int)sides.size());
        for (int i = 0; i < nb; i++) {
            DevBox d = g->dboxes[i];
            if (d.kind == 2 && d.tgt < 0)
                throw Error(BTE_EGEOM, "periodic box " + std::to_string(i) + " has no translation");
            if (d.tgt >= 0) d.tgt += bo;
            ptrans.push_back(g->ptrans[i]);
            d.c0 += co;
            d.c1 += co;
            for (int k = 0; k < 4; k++)
                if (d.side_nbr[k] >= 0) d.side_nbr[k] += bo;
            boxes.push_back(d);
            RtaBox rb{d.xmin, d.xmax, d.ymin, d.ymax, {d.side_nbr[0], d.side_nbr[1], d.side_nbr[2], d.side_nbr[3]},
                      d.kind, 0, (int)sides.size(), b->poly ? g->srange[i].y : 0};
            if (b->poly) {
                const int2 sr = g->srange[i];
                srange.push_back(make_int2((int)sides.size(), sr.y));
                for (int k = 0; k < sr.y; k++) {
                    DevSide q = g->sides[sr.x + k];
                    if (q.nbr >= 0) q.nbr += bo;
                    int id = -1;
                    for (size_t u = 0; u < normals.size() && id < 0; u++)
                        if (std::hypot(normals[u].x - q.nx, normals[u].y - q.ny) < 1.0e-9) id = (int)u;
                    if (id < 0) {
                        id = (int)normals.size();
                        normals.push_back(make_double2(q.nx, q.ny));
                    }
                    q.nid = id;
                    sides.push_back(q);
                }
                center.push_back(make_double2(g->boxes[i].cx(), g->boxes[i].cy()));
            }
            // only regular boxes tally (reservoirs absorb, periodic boxes
            // translate); box i of the batch has the cells i nt ... i nt + nt - 1
            if (d.kind == 0) {
                rb.lrow = (int32_t)b->lrows++;
                lrow_cell.push_back(b->cells + (uint64_t)i * nt);
            }
            rboxes.push_back(rb);
        }
        b->nside.push_back((int)sides.size() - b->side0.back());
        for (auto ct : g->dcontacts) {
            ct.box += bo;
            cts.push_back(ct);
        }
        cseg.insert(cseg.end(), g->cseg.begin(), g->cseg.end());
        for (auto q : g->cross) {
            q.box += bo;
            cross.push_back(q);
        }
        b->cells += (uint64_t)nb * nt;
        b->run_lrows.push_back((int32_t)b->lrows - b->run_lrow0.back());
        // BE_derivative sampler at the run temperature (sampling.cpp:47-68)
        for (int i = 0; i < n; i++) pmf[i] = m->omega[i] <= 0. ? 0. : h_be_kernel(m->omega[i], D.T0) * m->w[i];
        if (!build_alias(pmf.data(), n, th.data(), al.data())) throw Error(BTE_EINVAL, "empty scattering pmf");
        for (int i = 0; i < n; i++) scat.push_back(make_uint2(th[i], al[i]));
        // isothermal wall generators (RTA_MC2D.cpp:296-347, 366-397)
        std::vector<double> gw;
        R.gen0 = (int32_t)gens.size();
        for (int sid = 0; sid < nb; sid++) {
            const RectBox& sb = g->boxes[sid];
            if (sb.kind != 1) continue;
            for (auto& hc : g->contacts[sid]) {
                const RectBox& cb = g->boxes[hc.box];
                if (cb.kind != 0) continue;
                if (almost_equal(hc.length(), 0.)) continue;
                if (almost_equal(sb.Teq, cb.Teq)) continue;
                double cum = wall_pmf(*m, sb.Teq, cb.Teq, hc.npx, hc.npy, pmf.data());
                int sg = (sb.Teq - cb.Teq) >= 0 ? 1 : -1;
                double jd = sg * cum / (m->nq * vuc);
                gw.push_back(std::fabs(jd) * hc.length() * b->thickness);
                if (!build_alias(pmf.data(), n, th.data(), al.data())) throw Error(BTE_EINVAL, "empty wall pmf");
                for (int i = 0; i < n; i++) gtab.push_back(make_uint2(th[i], al[i]));
                gens.push_back(RtaGen{hc.p1x, hc.p1y, hc.p2x - hc.p1x, hc.p2y - hc.p1y, hc.box + bo, sg, 0, 0});
            }
        }
        R.ngen = (int32_t)gens.size() - R.gen0;
        if (R.ngen == 0) throw Error(BTE_EINVAL, "no isothermal generators (reservoirs at a different Teq)");
        const double einfo1 = std::accumulate(gw.begin(), gw.end(), 0.);
        b->Eeff.push_back(einfo1 / (double)D.nparticles);
        b->cv.push_back(h_calc_cv(*m, D.T0));
        std::vector<uint32_t> gth(gw.size()), gal(gw.size());
        build_alias(gw.data(), (int)gw.size(), gth.data(), gal.data());
        R.gsel0 = (int32_t)gsel.size();
        for (size_t k = 0; k < gw.size(); k++) gsel.push_back(make_uint2(gth[k], gal[k]));
        b->runs.push_back(R);
        b->total += D.nparticles;
    }
    b->d_boxes.upload(boxes, s);
    b->d_rboxes.upload(rboxes, s);
    b->nboxes = (int)boxes.size();
    b->nsides = (int)sides.size();
    if (b->poly) {
        b->d_sides.upload(sides, s);
        b->d_srange.upload(srange, s);
        b->d_center.upload(center, s);
    }
    b->d_cts.upload(cts.empty() ? std::vector<DevContact>(1) : cts, s);
    b->d_cseg.upload(cseg.empty() ? std::vector<double4>(1) : cseg, s);
    b->d_cross.upload(cross.empty() ? std::vector<DevCross>(1) : cross, s);
    b->d_ptrans.upload(ptrans, s);
    b->d_lrow_cell.upload(lrow_cell.empty() ? std::vector<uint64_t>(1) : lrow_cell, s);
    // arrays of the FP32 tallies: gz, jx, jy, then one per side that some run
    // differentiates
    int gunion = 0;
    for (auto& R : b->runs) gunion |= R.gmask;
    b->lt_arrays = 3;
    for (int k = 0; k < 4; k++)
        if ((gunion >> k) & 1) b->lt_goff[k] = b->lt_arrays++;
    b->d_gens.upload(gens, s);
    b->d_gen_sel.upload(gsel, s);
    b->d_gen_tab.upload(gtab, s);
    b->d_scat.upload(scat, s);
    b->d_runs.upload(b->runs, s);
    // Lambert tables (shared: they depend on the modes only)
    std::vector<int4> info;
    build_lambert(*m, b->sigma > 0 ? b->sigma : 0.25, normals, info, b->d_lam_tab, b->d_perm, s);
    std::vector<RtaMode> rm(n);
    for (int i = 0; i < n; i++)
        rm[i] = RtaMode{m->vx[i], m->vy[i], m->vx[i] != 0. ? 1.0 / m->vx[i] : 0., m->vy[i] != 0. ? 1.0 / m->vy[i] : 0.,
                        m->w[i], 1.0 / m->w[i], info[i].x, info[i].y, info[i].z, 0};
    b->d_rmodes.upload(rm, s);
    b->d_timegrid.upload(b->timegrid, s);
    b->d_tally.alloc((size_t)RTA_NCOPY * 3 * b->cells);
    if (b->any_grad) b->d_dgz.alloc((size_t)RTA_NCOPY * 4 * b->cells);
    b->d_counters.alloc(8 + 2 * (size_t)b->nruns);  // and tally mode 3's counters per run
    b->blocks = c->cu_count * 8;
    HIPCHECK(hipEventCreate(&b->ev0));
    HIPCHECK(hipEventCreate(&b->ev1));
    HIPCHECK(hipStreamSynchronize(s));
}

// The spectral arrays of every location as one strided-batched FP64 GEMM:
// out_l [nt][ncols] = cumsum_t(S_l) [nt][n] x W [n][ncols] (row-major)
static void spectral_products(RtaBatch* b) {
    Ctx* c = b->ctx;
    hipStream_t s = c->stream;
    const int nt = b->ntime - 1, n = b->m->n;
    const uint64_t ncolsum = (uint64_t)b->nloc * n;
    hipLaunchKernelGGL(rta_spec_cumsum_kernel, dim3((unsigned)((ncolsum + 255) / 256)), dim3(256), 0, s, b->d_spec.p,
                       b->nloc, nt, n);
    HIPCHECK(hipGetLastError());
    rocblas_handle hb = (rocblas_handle)blas_handle(c);
    const double one = 1.0, zero = 0.0;
    const rocblas_status st = rocblas_dgemm_strided_batched(
        hb, rocblas_operation_none, rocblas_operation_none, b->ncols, nt, n, &one, b->d_specw.p, b->ncols, 0,
        b->d_spec.p, n, (rocblas_stride)nt * n, &zero, b->d_specout.p, b->ncols, (rocblas_stride)nt * b->ncols,
        b->nloc);
    if (st != rocblas_status_success) throw Error(BTE_EHIP, "rocblas_dgemm_strided_batched failed");
    b->spec_host.resize((size_t)b->nloc * nt * b->ncols);
    HIPCHECK(hipMemcpyAsync(b->spec_host.data(), b->d_specout.p, b->spec_host.size() * sizeof(double),
                            hipMemcpyDeviceToHost, s));
    HIPCHECK(hipStreamSynchronize(s));
}

static void batch_execute(RtaBatch* b, double* T_out, double* jx_out, double* jy_out, double* dTdp,
                          double* Eeff_out, bte_rta_batch_report* rep) {
    Ctx* c = b->ctx;
    HIPCHECK(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    const int nt = b->ntime - 1;
    const uint64_t cells = b->cells;
    const RtaParams P = batch_params(b, b->d_runs.p, b->total);
    if (b->use_graph) {
        if (!b->gexec) {
            HIPCHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
            launch_batch(b, P, b->block, b->blocks, s);
            HIPCHECK(hipStreamEndCapture(s, &b->graph));
            HIPCHECK(hipGraphInstantiate(&b->gexec, b->graph, nullptr, nullptr, 0));
        }
        HIPCHECK(hipEventRecord(b->ev0, s));
        HIPCHECK(hipGraphLaunch(b->gexec, s));
        HIPCHECK(hipEventRecord(b->ev1, s));
    } else {
        HIPCHECK(hipEventRecord(b->ev0, s));
        launch_batch(b, P, b->block, b->blocks, s);
        HIPCHECK(hipGetLastError());
        HIPCHECK(hipEventRecord(b->ev1, s));
    }
    std::vector<double> tally(3 * cells), dg(b->any_grad ? 4 * cells : 0);
    unsigned long long cnt[8];
    HIPCHECK(hipMemcpyAsync(tally.data(), b->d_tally.p, 3 * cells * sizeof(double), hipMemcpyDeviceToHost, s));
    if (b->any_grad)
        HIPCHECK(hipMemcpyAsync(dg.data(), b->d_dgz.p, 4 * cells * sizeof(double), hipMemcpyDeviceToHost, s));
    HIPCHECK(hipMemcpyAsync(cnt, b->d_counters.p, sizeof(cnt), hipMemcpyDeviceToHost, s));
    HIPCHECK(hipStreamSynchronize(s));
    float ms = 0;
    HIPCHECK(hipEventElapsedTime(&ms, b->ev0, b->ev1));
    if (cnt[3] != 0)
        throw Error(BTE_EGEOM, std::to_string(cnt[3]) + " particle histories exceeded the iteration budget");
    if (cnt[4] != 0)
        throw Error(BTE_EINVAL, "specular reflection of a mode without a mirror partner in the mode table");
    if (cnt[5] != 0) throw Error(BTE_EGEOM, "Error in translation, no box found");
    if (b->nloc) spectral_products(b);
    // post-processing per run (RTA_MC2D.cpp:2336-2435): scale, cumulative
    // sum over time (step response), T = gz / (Cv / vcorr) + T0
    const double th = b->thickness, vcorr = th / b->m->lattz;
    uint64_t out0 = 0;
    for (int r = 0; r < b->nruns; r++) {
        const Geom* g = b->geoms[r];
        const int nb = b->nbox[r];
        const double E = b->Eeff[r], cvr = b->cv[r];
        double* gz = tally.data() + b->cell0[r];
        double* jx = gz + cells;
        double* jy = jx + cells;
        for (int bx = 0; bx < nb; bx++) {
            const double vbox = g->boxes[bx].area() * th;
            double agz = 0, ajx = 0, ajy = 0;
            double ad[4] = {0, 0, 0, 0};
            for (int k = 0; k < nt; k++) {
                const size_t cidx = (size_t)bx * nt + k;
                agz += gz[cidx] * E / vbox;
                ajx += jx[cidx] * E * 1e30 / vbox;
                ajy += jy[cidx] * E * 1e30 / vbox;
                const size_t o = out0 + (size_t)k * nb + bx;
                T_out[o] = agz / (cvr / vcorr) + b->desc[r].T0;
                jx_out[o] = ajx;
                jy_out[o] = ajy;
                if (dTdp) {
                    for (int q = 0; q < 4; q++) {
                        if (b->any_grad) ad[q] += dg[(size_t)q * cells + b->cell0[r] + cidx] * E / vbox;
                        dTdp[4 * out0 + (size_t)q * nt * nb + (size_t)k * nb + bx] = ad[q] / (cvr / vcorr);
                    }
                }
            }
        }
        if (Eeff_out) Eeff_out[r] = E;
        out0 += (uint64_t)nt * nb;
    }
    if (rep) {
        rep->events = cnt[0];
        rep->crossings = cnt[1];
        rep->kernel_ms = ms;
        rep->ntime = b->ntime;
        rep->block = b->block;
        rep->blocks = b->blocks;
    }
}

// Launch-shape autotuner: times the batch with every run scaled to a
// fraction of its particles for each candidate (block size, workgroups per
// CU) and keeps the fastest.
// FP32 LDS tallies on (mode 1) or off (mode 0); see bte_rta_batch_set_tally.
static void batch_set_tally(RtaBatch* b, int mode) {
    if (mode < 0 || mode > 3)
        throw Error(BTE_EINVAL,
                    "tally mode must be 0 (FP64 atomics), 1 (FP32 LDS), 2 (FP64 LDS, leading time bins) or 3 "
                    "(FP64 LDS per run, leading time bins)");
    if (mode == 3) {
        if (b->nloc) throw Error(BTE_EINVAL, "LDS tallies do not cover spectral locations");
        if (b->any_grad) throw Error(BTE_EINVAL, "tally mode 3 does not carry dT/dp; use mode 1 or 0");
        const int nt = b->ntime - 1;
        // the block: the largest run's geometry and the time grid (see RtaGeo),
        // then [3][rows][bins] doubles; a margin for the kernel's static LDS
        b->l3_nbox = *std::max_element(b->nbox.begin(), b->nbox.end());
        b->l3_nside = *std::max_element(b->nside.begin(), b->nside.end());
        RtaLds L = rta_lds_layout(b->l3_nbox, b->l3_nside, nt);
        const int32_t max_rows = *std::max_element(b->run_lrows.begin(), b->run_lrows.end());
        b->l3_mail = (size_t)L.geo + 3 * sizeof(double) * (size_t)max_rows <= b->ctx->lds_per_block - 1024;
        if (!b->l3_mail) drop_mail(L);
        const size_t avail = b->ctx->lds_per_block - 1024 - (size_t)L.geo;
        b->l3_bytes = L.bytes;
        std::vector<int32_t> lb(b->nruns, 0);
        for (int r = 0; r < b->nruns; r++) {
            const size_t rows = (size_t)b->run_lrows[r];
            if (rows == 0) continue;
            if (16 + 3 * sizeof(double) * rows > b->ctx->lds_per_block - 1024)
                throw Error(BTE_EINVAL, "run " + std::to_string(r) + ": FP64 LDS tallies need " +
                                            std::to_string(16 + 3 * sizeof(double) * rows) +
                                            " bytes of LDS for one time bin, the device has " +
                                            std::to_string(b->ctx->lds_per_block - 1024) + " per workgroup");
            lb[r] = (int32_t)std::min<size_t>((size_t)nt, avail / (3 * sizeof(double) * rows));
            b->l3_bytes = std::max(b->l3_bytes, (size_t)L.geo + 3 * sizeof(double) * rows * (size_t)lb[r]);
        }
        allow_lds(rta_runs_kernel(b->poly, L.gl), b->l3_bytes);
        b->block = 768;
        b->blocks = b->ctx->cu_count;
        // workgroups per run in proportion to its particles (largest remainder),
        // one at least while there are as many workgroups as runs; with more
        // runs the largest begin and the others are picked as workgroups end
        std::vector<int> order(b->nruns), wgs(b->nruns, 0);
        for (int r = 0; r < b->nruns; r++) order[r] = r;
        std::stable_sort(order.begin(), order.end(),
                         [&](int x, int y) { return b->runs[x].count > b->runs[y].count; });
        int left = b->blocks;
        for (int r : order)
            if (left > 0) {
                wgs[r] = 1;
                left--;
            }
        if (left > 0) {
            std::vector<std::pair<double, int>> rest;
            const int spare = left;
            for (int r = 0; r < b->nruns; r++) {
                const double share = (double)spare * (double)b->runs[r].count / (double)b->total;
                wgs[r] += (int)share;
                left -= (int)share;
                rest.push_back({share - std::floor(share), r});
            }
            std::stable_sort(rest.begin(), rest.end(), [](auto& x, auto& y) { return x.first > y.first; });
            for (int k = 0; k < left; k++) wgs[rest[k % rest.size()].second]++;
        }
        std::vector<int32_t> first;
        for (int r : order) first.insert(first.end(), wgs[r], r);
        first.resize(b->blocks, -1);
        std::vector<RtaRunRows> rows(b->nruns);
        for (int r = 0; r < b->nruns; r++)
            rows[r] = RtaRunRows{b->run_lrow0[r], b->run_lrows[r], lb[r], wgs[r],
                                 b->box0[r], b->nbox[r], b->side0[r], b->nside[r]};
        // the same buffers when the mode is set again: a captured graph holds their addresses
        b->d_rows.upload(rows.data(), rows.size(), b->ctx->stream);
        b->d_first_run.upload(first.data(), first.size(), b->ctx->stream);
        HIPCHECK(hipStreamSynchronize(b->ctx->stream));  // the host arrays end here
    } else if (mode == 2) {
        if (b->nloc) throw Error(BTE_EINVAL, "LDS tallies do not cover spectral locations");
        if (b->any_grad) throw Error(BTE_EINVAL, "tally mode 2 does not carry dT/dp; use mode 1 or 0");
        const RtaLds L = rta_lds_of(b, 2);
        if (L.lbins == 0)
            throw Error(BTE_EINVAL, "FP64 LDS tallies need " + std::to_string(3 * sizeof(double) * b->lrows) +
                                        " bytes of LDS for one time bin, the device has " +
                                        std::to_string(b->ctx->lds_per_block) + " per workgroup");
        allow_lds(rta_kernel(2, false, b->poly, L.gl), b->ctx->lds_per_block);
        // one 768-thread workgroup per CU, also where two blocks fit its LDS:
        // the kernels' 139 registers leave each SIMD three waves, so a second
        // one would begin when the first has ended and the ids are gone
        b->block = 768;
        b->blocks = b->ctx->cu_count;
        const size_t np = (size_t)b->blocks * 3 * b->lrows * L.lbins;
        if (b->d_part.n < np) b->d_part.alloc(np);  // kept: a captured graph holds its address
    } else if (mode == 1) {
        if (b->nloc) throw Error(BTE_EINVAL, "FP32 LDS tallies do not cover spectral locations");
        // every time bin of every array has to fit next to nothing else: what
        // the geometry displaces goes to device atomics
        const size_t need = std::max<size_t>((size_t)b->lt_arrays * b->lrows * (size_t)(b->ntime - 1) * sizeof(float),
                                             16 * 5 * sizeof(uint64_t));
        if (need > b->ctx->lds_per_block)
            throw Error(BTE_EINVAL, "FP32 LDS tallies need " + std::to_string(need) + " bytes of LDS, the device has " +
                                        std::to_string(b->ctx->lds_per_block) + " per workgroup");
        allow_lds(rta_kernel(1, b->any_grad, b->poly, rta_lds_of(b, 1).gl), b->ctx->lds_per_block);
        b->block = 768;
        b->blocks = b->ctx->cu_count;
    } else if (b->tally != 0) {
        b->block = 256;
        b->blocks = b->ctx->cu_count * 8;
    }
    if (mode != b->tally && b->gexec) {
        (void)hipGraphExecDestroy(b->gexec);
        (void)hipGraphDestroy(b->graph);
        b->gexec = nullptr;
        b->graph = nullptr;
    }
    b->tally = mode;
}

static void batch_tune(RtaBatch* b, double fraction) {
    if (b->tally != 0) return;  // one 768-thread workgroup per CU: the LDS holds one tally block
    Ctx* c = b->ctx;
    hipStream_t s = c->stream;
    std::vector<RtaRunDev> tr = b->runs;
    uint64_t tot = 0;
    for (auto& R : tr) {
        R.count = std::max<uint64_t>(1, (uint64_t)(R.count * fraction));
        R.first = tot;
        tot += R.count;
    }
    b->d_trial_runs.upload(tr, s);
    const RtaParams P = batch_params(b, b->d_trial_runs.p, tot);
    const int cand[][2] = {{256, 4}, {256, 8}, {256, 16}, {128, 8}, {128, 16}, {128, 32}, {512, 2}, {512, 4}};
    double best = 1e300;
    int bb = b->block, bn = b->blocks;
    for (auto& cd : cand) {
        const int blocks = c->cu_count * cd[1];
        launch_batch(b, P, cd[0], blocks, s);  // warm-up
        HIPCHECK(hipEventRecord(b->ev0, s));
        launch_batch(b, P, cd[0], blocks, s);
        HIPCHECK(hipEventRecord(b->ev1, s));
        HIPCHECK(hipStreamSynchronize(s));
        float ms = 0;
        HIPCHECK(hipEventElapsedTime(&ms, b->ev0, b->ev1));
        if (ms < best) {
            best = ms;
            bb = cd[0];
            bn = blocks;
        }
    }
    if (bb != b->block || bn != b->blocks) {
        b->block = bb;
        b->blocks = bn;
        if (b->gexec) {
            (void)hipGraphExecDestroy(b->gexec);
            (void)hipGraphDestroy(b->graph);
            b->gexec = nullptr;
            b->graph = nullptr;
        }
    }
}

// ---- the allocation-free variant of bte_rta_execute ----
//
// Its tally copies, counters and per-workgroup LDS blocks live in this
// file-scope device array instead of buffers of the handle. Every GPU the
// library runs on holds one copy until the process ends; the host reaches it
// only through the address hipGetSymbolAddress gives for the current device
// (the array's name is not a device address in host code).
#define RTA_SCRATCH_BYTES (64ull << 20)
static __device__ __align__(256) unsigned char scratch[RTA_SCRATCH_BYTES];

static std::mutex g_scratch_mu;
static std::vector<void*> g_scratch_ptr;  // per device, looked up once

// the scratch array's device address on device dev (current device)
static void* scratch_address(int dev) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (dev < 0) throw Error(BTE_EINVAL, "bad device");
    if ((size_t)dev >= g_scratch_ptr.size()) g_scratch_ptr.resize((size_t)dev + 1, nullptr);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            throw Error(BTE_EHIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}

// Post-processing of one run on the device (RTA_MC2D.cpp:2336-2435, the
// same arithmetic as batch_execute): per box the cumulative sums over time
// of gz E / vbox, jx E 1e30 / vbox, jy E 1e30 / vbox, T = sum / (Cv / vcorr)
// + T0; outputs [nt][nbox]. One thread per box.
__global__ __launch_bounds__(256) void rta_post_kernel(const double* tally, uint64_t cells, const DevBox* boxes,
                                                       int nbox, int nt, double E, double th, double cv,
                                                       double vcorr, double T0, double* T, double* JX,
                                                       double* JY, const unsigned long long* cnt,
                                                       unsigned long long* cnt_out) {
    const int bx = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x < 6) cnt_out[threadIdx.x] = cnt[threadIdx.x];
    if (bx >= nbox) return;
    const DevBox b = boxes[bx];
    const double vbox = (b.xmax - b.xmin) * (b.ymax - b.ymin) * th;
    const double* gz = tally + (uint64_t)bx * nt;
    const double* jx = gz + cells;
    const double* jy = jx + cells;
    double agz = 0., ajx = 0., ajy = 0.;
    for (int k = 0; k < nt; k++) {
        agz += gz[k] * E / vbox;
        ajx += jx[k] * E * 1e30 / vbox;
        ajy += jy[k] * E * 1e30 / vbox;
        const size_t o = (size_t)k * nbox + bx;
        T[o] = agz / (cv / vcorr) + T0;
        JX[o] = ajx;
        JY[o] = ajy;
    }
}

static void rta_execute_noalloc(RtaBatch* b, double* d_T, double* d_jx, double* d_jy, unsigned long long* d_counts) {
    Ctx* c = b->ctx;
    if (b->nruns != 1) throw Error(BTE_EINVAL, "bte_rta_execute_noalloc takes a single-run handle");
    if (b->nloc) throw Error(BTE_EINVAL, "bte_rta_execute_noalloc does not tally spectral locations");
    if (b->any_grad) throw Error(BTE_EINVAL, "bte_rta_execute_noalloc does not tally the gradient sides");
    if (b->poly) throw Error(BTE_EINVAL, "bte_rta_execute_noalloc takes rectangular boxes only");
    if (!d_T || !d_jx || !d_jy || !d_counts) throw Error(BTE_EINVAL, "null argument");
    HIPCHECK(hipSetDevice(c->device));
    double* base = (double*)scratch_address(c->device);
    // the tally mode bte_rta_execute picks, without touching the handle's
    const RtaLds L2 = rta_lds_of(b, 2);
    const int mode = L2.lbins > 0 ? 2 : 0;
    const RtaLds L = mode == 2 ? L2 : rta_lds_of(b, 0);
    const int block = mode == 2 ? 768 : 256, blocks = mode == 2 ? c->cu_count : c->cu_count * 8;
    const size_t ncopy = (size_t)RTA_NCOPY * 3 * b->cells;
    const size_t ncnt = 8;  // the counters, as unsigned 64-bit words
    // the limit counts the time bins that a workgroup's whole LDS holds
    const size_t full_bins = mode == 2 ? std::min<size_t>((size_t)(b->ntime - 1),
                                                          c->lds_per_block / (3 * sizeof(double) * b->lrows)) : 0;
    const size_t npart = mode == 2 ? (size_t)blocks * 3 * b->lrows * full_bins : 0;
    const size_t need = (ncopy + ncnt + npart) * sizeof(double);
    if (need > RTA_SCRATCH_BYTES)
        throw Error(BTE_EINVAL, "bte_rta_execute_noalloc needs " + std::to_string(need) +
                                    " bytes of scratch for this run's tallies; the limit is " +
                                    std::to_string(RTA_SCRATCH_BYTES));
    RtaParams P = batch_params(b, b->d_runs.p, b->total);
    P.gz = base;
    P.jx = base + b->cells;
    P.jy = base + 2 * b->cells;
    P.dgz = nullptr;
    P.counters = (unsigned long long*)(base + ncopy);
    P.part = base + ncopy + ncnt;
    hipStream_t s = c->stream;
    // the scratch keeps the previous call's contents: the tally copies and
    // the counters start at zero (a kernel, not a memset, so that a graph
    // capture records no memset node); the partial blocks are overwritten
    hipLaunchKernelGGL(rta_clear_kernel, dim3(1024), dim3(256), 0, s, base, (uint64_t)ncopy, P.counters, 8);
    set_lds(P, L);
    P.waves = share_waves(block, blocks, c->cu_count);
    const RtaKernel k = rta_kernel(mode, false, false, L.gl);
    if (mode == 2) allow_lds(k, c->lds_per_block);
    hipLaunchKernelGGL(k, dim3(blocks), dim3(block), L.bytes, s, P);
    if (mode == 2) {
        const uint32_t nf = 3u * b->lrows * L.lbins;
        hipLaunchKernelGGL(rta_sum_parts_kernel, dim3((nf + RTA_SUM_CELLS - 1) / RTA_SUM_CELLS), dim3(512), 0, s,
                           base, P.part, blocks, b->lrows, L.lbins, b->d_lrow_cell.p, b->cells);
    }
    hipLaunchKernelGGL(rta_sum_copies_kernel, dim3(1024), dim3(256), 0, s, base, 3 * b->cells);
    const int nb = b->nbox[0], nt = b->ntime - 1;
    const double th = b->thickness;
    hipLaunchKernelGGL(rta_post_kernel, dim3((nb + 255) / 256), dim3(256), 0, s, base, b->cells, b->d_boxes.p, nb, nt,
                       b->Eeff[0], th, b->cv[0], th / b->m->lattz, b->desc[0].T0, d_T, d_jx, d_jy, P.counters,
                       d_counts);
    HIPCHECK(hipGetLastError());
}

}  // namespace bte

using namespace bte;

extern "C" {

int bte_rta_batch_create(bte_ctx* ctx, const bte_modes* mm, int nruns, const bte_rta_run_desc* runs,
                         double thickness, double dt, double maxtime, double sigma_bounce, int use_graph,
                         bte_rta_batch** out) {
    BTE_GUARD_BEGIN
    auto* c = reinterpret_cast<Ctx*>(ctx);
    auto* m = reinterpret_cast<const Modes*>(mm);
    if (!c || !m || !runs || !out || nruns <= 0) throw Error(BTE_EINVAL, "bad arguments to bte_rta_batch_create");
    HIPCHECK(hipSetDevice(c->device));
    auto* b = new RtaBatch();
    std::unique_ptr<RtaBatch> guard(b);
    b->ctx = c;
    b->m = m;
    b->desc.assign(runs, runs + nruns);
    for (int r = 0; r < nruns; r++) b->geoms.push_back(reinterpret_cast<const Geom*>(runs[r].geom));
    b->thickness = thickness;
    b->dt = dt;
    b->maxtime = maxtime;
    b->sigma = sigma_bounce;
    b->use_graph = use_graph != 0;
    batch_create(b);
    *out = reinterpret_cast<bte_rta_batch*>(guard.release());
    BTE_GUARD_END
}

int bte_rta_batch_set_tally(bte_rta_batch* bb, int mode) {
    BTE_GUARD_BEGIN
    auto* b = reinterpret_cast<RtaBatch*>(bb);
    if (!b) throw Error(BTE_EINVAL, "null batch");
    HIPCHECK(hipSetDevice(b->ctx->device));
    batch_set_tally(b, mode);
    BTE_GUARD_END
}

int bte_rta_batch_tune(bte_rta_batch* bb, double fraction, int* block, int* blocks) {
    BTE_GUARD_BEGIN
    auto* b = reinterpret_cast<RtaBatch*>(bb);
    if (!b || !(fraction > 0) || fraction > 1) throw Error(BTE_EINVAL, "bad arguments to bte_rta_batch_tune");
    HIPCHECK(hipSetDevice(b->ctx->device));
    batch_tune(b, fraction);
    if (block) *block = b->block;
    if (blocks) *blocks = b->blocks;
    BTE_GUARD_END
}

int bte_rta_batch_execute(bte_rta_batch* bb, double* T_out, double* jx_out, double* jy_out, double* dTdp,
                          double* Eeff, bte_rta_batch_report* rep) {
    BTE_GUARD_BEGIN
    auto* b = reinterpret_cast<RtaBatch*>(bb);
    if (!b || !T_out || !jx_out || !jy_out) throw Error(BTE_EINVAL, "null argument");
    batch_execute(b, T_out, jx_out, jy_out, dTdp, Eeff, rep);
    BTE_GUARD_END
}

int bte_rta_batch_destroy(bte_rta_batch* bb) {
    BTE_GUARD_BEGIN
    delete reinterpret_cast<RtaBatch*>(bb);
    BTE_GUARD_END
}

// single runs: a batch of one, with the reference's diffuse walls
int bte_rta_create(bte_ctx* ctx, const bte_modes* m, const bte_geom* g, const bte_rta_cfg* cfg, bte_rta** out) {
    BTE_GUARD_BEGIN
    if (!cfg || !out || !g) throw Error(BTE_EINVAL, "null argument");
    if (!(cfg->dt > 0) || !(cfg->maxtime > 0) || cfg->nparticles == 0 || !(cfg->thickness > 0))
        throw Error(BTE_EINVAL, "bad RTA configuration");
    bte_rta_run_desc d{};
    d.geom = g;
    d.T0 = cfg->T0;
    d.nparticles = cfg->nparticles;
    d.seed = cfg->seed;
    d.ballistic = cfg->ballistic;
    d.wscale = 1.0;
    bte_rta_batch* b = nullptr;
    int rc = bte_rta_batch_create(ctx, m, 1, &d, cfg->thickness, cfg->dt, cfg->maxtime, cfg->sigma_bounce, 0, &b);
    if (rc != BTE_OK) return rc;
    *out = reinterpret_cast<bte_rta*>(b);
    BTE_GUARD_END
}

int bte_rta_execute(bte_rta* rr, double* T_out, double* jx_out, double* jy_out, bte_rta_report* rep) {
    BTE_GUARD_BEGIN
    auto* b = reinterpret_cast<RtaBatch*>(rr);
    if (!b || !T_out || !jx_out || !jy_out) throw Error(BTE_EINVAL, "null argument");
    HIPCHECK(hipSetDevice(b->ctx->device));
    // FP64 LDS partial sums of the leading time bins (tally mode 2: the same
    // histories and FP64 sums) whenever one time bin of every box fits;
    // device atomics with spectral locations
    const int want = (!b->nloc && !b->any_grad && rta_lds_of(b, 2).lbins > 0) ? 2 : 0;
    if (b->tally != want) batch_set_tally(b, want);
    bte_rta_batch_report br{};
    double E = 0;
    batch_execute(b, T_out, jx_out, jy_out, nullptr, &E, &br);
    if (rep) {
        rep->events = br.events;
        rep->crossings = br.crossings;
        rep->Eeff = E;
        rep->kernel_ms = br.kernel_ms;
        rep->ntime = br.ntime;
    }
    BTE_GUARD_END
}

int bte_rta_spectral(bte_rta* rr, int nloc, const int32_t* boxes, int nomega, const double* sigma) {
    BTE_GUARD_BEGIN
    auto* b = reinterpret_cast<RtaBatch*>(rr);
    if (!b || nloc < 0 || (nloc > 0 && (!boxes || nomega < 1))) throw Error(BTE_EINVAL, "bad arguments to bte_rta_spectral");
    if (b->nruns != 1) throw Error(BTE_EINVAL, "spectral decomposition needs a single-run handle");
    Ctx* c = b->ctx;
    HIPCHECK(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    const Modes* m = b->m;
    const int n = m->n, nbox = b->nbox[0], nq = m->nq;
    b->nloc = 0;
    if (nloc == 0) return BTE_OK;
    std::vector<int32_t> loc((size_t)b->box0[0] + nbox, -1);
    for (int l = 0; l < nloc; l++) {
        if (boxes[l] < 0 || boxes[l] >= nbox) throw Error(BTE_EINVAL, "spectral location out of range");
        loc[(size_t)b->box0[0] + boxes[l]] = l;
    }
    // omega ticks: LinSpaced(nomega, 0, maxomega) + delta/2, delta =
    // maxomega / nomega (RTA_MC2D.cpp:2040-2045)
    double maxomega = 0;
    for (int i = 0; i < n; i++) maxomega = std::max(maxomega, m->omega[i]);
    const double delta = maxomega / nomega;
    b->omegagrid.resize(nomega);
    for (int i = 0; i < nomega; i++)
        b->omegagrid[i] = (nomega > 1 ? maxomega * i / (nomega - 1) : maxomega) + 0.5 * delta;
    const int ncols = 3 * nomega + nq;
    std::vector<double> W;
    spectral_weights(*m, sigma ? sigma : (m->sigma.empty() ? nullptr : m->sigma.data()), b->sigma, nomega,
                     b->omegagrid.data(), W);
    const int nt = b->ntime - 1;
    b->d_box_loc.upload(loc, s);
    b->d_specw.upload(W, s);
    b->d_spec.alloc((size_t)nloc * nt * n);
    b->d_specout.alloc((size_t)nloc * nt * ncols);
    HIPCHECK(hipStreamSynchronize(s));
    b->spec_boxes.assign(boxes, boxes + nloc);
    b->nloc = nloc;
    b->nomega = nomega;
    b->ncols = ncols;
    b->spec_host.clear();
    // a captured launch would miss the spectral tally
    if (b->gexec) {
        (void)hipGraphExecDestroy(b->gexec);
        (void)hipGraphDestroy(b->graph);
        b->gexec = nullptr;
        b->graph = nullptr;
    }
    BTE_GUARD_END
}

int bte_rta_spectral_get(const bte_rta* rr, int k, double* omega, double* dT, double* jx, double* jy, double* fd_q) {
    BTE_GUARD_BEGIN
    auto* b = reinterpret_cast<const RtaBatch*>(rr);
    if (!b || k < 0 || k >= b->nloc) throw Error(BTE_EINVAL, "no such spectral location");
    if (b->spec_host.empty()) throw Error(BTE_EINVAL, "bte_rta_spectral_get before bte_rta_execute");
    const int nt = b->ntime - 1, nw = b->nomega, nq = b->m->nq, nc = b->ncols;
    const RectBox& bx = b->geoms[0]->boxes[b->spec_boxes[k]];
    const double th = b->thickness, vbox = bx.area() * th, vcorr = th / b->m->lattz, E = b->Eeff[0];
    // post-processing (RTA_MC2D.cpp:2349-2405): gz_omega * Eeff / vbox /
    // (Cv / vcorr), fluxes * Eeff 1e30 / vbox, fd * Eeff vcorr NQ /
    // (vbox 1e12 hbar); the time sums are already taken
    const double sT = E / vbox / (b->cv[0] / vcorr), sJ = E * 1e30 / vbox, sF = E * vcorr * nq / (vbox * 1.0e12 * hbar);
    if (omega) std::copy(b->omegagrid.begin(), b->omegagrid.end(), omega);
    for (int t = 0; t < nt; t++) {
        const double* r = b->spec_host.data() + ((size_t)k * nt + t) * nc;
        for (int j = 0; j < nw; j++) {
            if (dT) dT[(size_t)t * nw + j] = r[j] * sT;
            if (jx) jx[(size_t)t * nw + j] = r[nw + j] * sJ;
            if (jy) jy[(size_t)t * nw + j] = r[2 * nw + j] * sJ;
        }
        if (fd_q)
            for (int q = 0; q < nq; q++) fd_q[(size_t)t * nq + q] = r[3 * nw + q] * sF;
    }
    BTE_GUARD_END
}

int bte_spectra(bte_ctx* ctx, const bte_modes* mm, const double* sigma, double sigma_default, int nomega,
                const double* grid, int nrows, const double* X, double* out) {
    BTE_GUARD_BEGIN
    auto* c = reinterpret_cast<Ctx*>(ctx);
    auto* m = reinterpret_cast<const Modes*>(mm);
    if (!c || !m || !grid || !X || !out || nomega < 1 || nrows < 0) throw Error(BTE_EINVAL, "bad arguments to bte_spectra");
    if (nrows == 0) return BTE_OK;
    HIPCHECK(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    std::vector<double> W;
    spectral_weights(*m, sigma ? sigma : (m->sigma.empty() ? nullptr : m->sigma.data()), sigma_default, nomega,
                     grid, W);
    const int n = m->n, ncols = 3 * nomega + m->nq;
    DevBuf<double> dW, dX, dO;
    dW.upload(W, s);
    dX.upload(X, (size_t)nrows * n, s);
    dO.alloc((size_t)nrows * ncols);
    // out [nrows][ncols] = X [nrows][n] x W [n][ncols], row-major
    rocblas_handle hb = (rocblas_handle)blas_handle(c);
    const double one = 1.0, zero = 0.0;
    if (rocblas_dgemm(hb, rocblas_operation_none, rocblas_operation_none, ncols, nrows, n, &one, dW.p, ncols, dX.p, n,
                      &zero, dO.p, ncols) != rocblas_status_success)
        throw Error(BTE_EHIP, "rocblas_dgemm failed");
    HIPCHECK(hipMemcpyAsync(out, dO.p, (size_t)nrows * ncols * sizeof(double), hipMemcpyDeviceToHost, s));
    HIPCHECK(hipStreamSynchronize(s));
    BTE_GUARD_END
}

int bte_rta_execute_noalloc(bte_rta* rr, double* d_T, double* d_jx, double* d_jy, unsigned long long* d_counts) {
    BTE_GUARD_BEGIN
    auto* b = reinterpret_cast<RtaBatch*>(rr);
    if (!b) throw Error(BTE_EINVAL, "null handle");
    rta_execute_noalloc(b, d_T, d_jx, d_jy, d_counts);
    BTE_GUARD_END
}

int bte_rta_destroy(bte_rta* rr) {
    BTE_GUARD_BEGIN
    delete reinterpret_cast<RtaBatch*>(rr);
    BTE_GUARD_END
}

int bte_rta_run(bte_ctx* ctx, const bte_modes* m, const bte_geom* g, const bte_rta_cfg* cfg,
                double* T_out, double* jx_out, double* jy_out, bte_rta_report* rep) {
    bte_rta* r = nullptr;
    int rc = bte_rta_create(ctx, m, g, cfg, &r);
    if (rc != BTE_OK) return rc;
    rc = bte_rta_execute(r, T_out, jx_out, jy_out, rep);
    bte_rta_destroy(r);
    return rc;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// RTAMC2D steady branch (nonzero <gradient>, RTA_MC2D.cpp:2544-2782): a
// generation iteration. Each generation every particle makes one flight:
// a relaxation inside a box adds its sign to phi(box) (process_segment with
// evalphi, RTA_MC2D.cpp:771-826), a diffuse wall bounce carries it into the
// next generation, a reservoir absorbs it; then |phi(box)| particles of sign
// phi are re-emitted uniformly in each box from BE_derivative. gz, jx, jy
// accumulate over generations until the relative change falls below the
// <convergence> thresholds or no particle is left.
namespace bte {

struct RtaSPart {
    double x, y;
    uint32_t mode, boxsign;  // box << 1 | (sign < 0)
    uint64_t id;
};

struct RtaSteadyParams {
    const double4* modes;
    const double2* ivel;
    const uint2* scat;
    const DevBox* boxes;
    const DevContact* cts;
    const double4* cseg;
    const DevCross* cross;
    const double2* ptrans;
    const DevSide* sides;     // polygon geometries: sides, side range and centre per box
    const int2* srange;
    const double2* center;
    const int4* lam_info;
    const uint2* lam_tab;
    const int32_t* perm;
    const RtaGen* gens;
    const uint2* gen_sel;
    const uint2* gen_tab;
    const int32_t* gbox;     // boxes with a gradient generator
    const uint2* gbox_sel;   // alias over their energies
    const uint2* gtab;       // per gradient box: [2][n] alias (0: sign +, 1: sign -)
    const int32_t* gclass;   // per gradient box: bit 0 has +, bit 1 has -
    const uint64_t* regen;   // prefix of re-emission counts [nbox + 1]
    double* acc;             // [3][nbox] gz, jx, jy over all generations
    double* phi;             // [nbox] this generation
    const RtaSPart* pin;
    RtaSPart* pout;
    unsigned long long* counters;  // [0] appended, [1] flights, [2] stuck, [3] bad translation
    uint64_t nin, seed, key;
    double pwall;            // share of wall generators in the initial energy
    unsigned long long max_iters;
    int32_t n, nbox, ngen, ngbox, lds_tally;
};

__device__ inline void steady_append(const RtaSteadyParams& P, bool want, const RtaSPart& q) {
    const unsigned long long m = __ballot(want);
    if (m == 0ULL) return;
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll((long long)m) - 1;
    unsigned long long base = 0;
    if (lane == leader) base = atomicAdd(P.counters + 0, (unsigned long long)__popcll(m));
    base = __shfl(base, leader, 64);
    if (want) P.pout[base + __popcll(m & ((1ULL << lane) - 1ULL))] = q;
}

// get_random_point of box b (geometry_2d.hpp:332-348): x, then y in the
// bounding box, until covered by the box (polygons; a rectangle takes the
// first draw). A box that a few thousand draws miss is counted as stuck and
// gets its centre.
template <bool POLY>
__device__ inline void steady_box_point(const RtaSteadyParams& P, int b, Pcg32& rng, double& x, double& y,
                                        unsigned long long& stuck) {
    const DevBox B = P.boxes[b];
    x = B.xmin + rng.uniform() * (B.xmax - B.xmin);
    y = B.ymin + rng.uniform() * (B.ymax - B.ymin);
    if constexpr (POLY) {
        const int2 sr = P.srange[b];
        int tries = 0;
        while (!poly_inside(P.sides, sr, x, y)) {
            if (++tries > 4096) {
                stuck++;
                x = P.center[b].x;
                y = P.center[b].y;
                return;
            }
            x = B.xmin + rng.uniform() * (B.xmax - B.xmin);
            y = B.ymin + rng.uniform() * (B.ymax - B.ymin);
        }
    }
}

// initial particles (Init_generator, RTA_MC2D.cpp:436-533)
template <bool POLY>
__global__ __launch_bounds__(256) void rta_steady_init_kernel(RtaSteadyParams P, uint64_t np) {
    unsigned long long stuck = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < np; i += (uint64_t)gridDim.x * blockDim.x) {
        Pcg32 rng;
        rng.seed(P.seed, i);
        RtaSPart q{0., 0., 0u, 0u, i};
        const double r = rng.uniform();
        bool ng;
        if (P.ngen > 0 && r <= P.pwall) {
            const int gi = (int)alias_pick(P.gen_sel, (uint32_t)P.ngen, rng, ng);
            const RtaGen g = P.gens[gi];
            const double u = rng.uniform();
            double x = g.p1x + u * g.ndx, y = g.p1y + u * g.ndy;
            const DevBox bi = P.boxes[g.idi];
            if (!(POLY ? poly_inside(P.sides, P.srange[g.idi], x, y) : box_inside(bi, x, y))) {
                const double ccx = POLY ? P.center[g.idi].x : 0.5 * (bi.xmin + bi.xmax);
                const double ccy = POLY ? P.center[g.idi].y : 0.5 * (bi.ymin + bi.ymax);
                double dx = ccx - x, dy = ccy - y;
                double dn = sqrt(dx * dx + dy * dy);
                x += 1.0e-6 * dx / dn;
                y += 1.0e-6 * dy / dn;
            }
            q.x = x;
            q.y = y;
            q.mode = alias_pick(P.gen_tab + (size_t)gi * P.n, (uint32_t)P.n, rng, ng);
            q.boxsign = ((uint32_t)g.idi << 1) | (g.sign < 0 ? 1u : 0u);
        } else {
            const int k = (int)alias_pick(P.gbox_sel, (uint32_t)P.ngbox, rng, ng);
            const int b = P.gbox[k];
            steady_box_point<POLY>(P, b, rng, q.x, q.y, stuck);
            // signs alternate with the id; a class without modes gives way
            const int cls = P.gclass[k];
            int neg = (i & 1) ? 0 : 1;
            if (neg && !(cls & 2)) neg = 0;
            if (!neg && !(cls & 1)) neg = 1;
            q.mode = alias_pick(P.gtab + ((size_t)k * 2 + neg) * P.n, (uint32_t)P.n, rng, ng);
            q.boxsign = ((uint32_t)b << 1) | (uint32_t)neg;
        }
        P.pout[i] = q;
    }
    if (POLY) block_add_u64(P.counters + 2, stuck);
}

// one flight per particle (steady evolparticle, RTA_MC2D.cpp:1406-1799)
template <bool POLY>
__global__ __launch_bounds__(256) void rta_steady_flight_kernel(RtaSteadyParams P) {
    extern __shared__ __align__(16) unsigned char sdyn[];
    double* sacc = (double*)sdyn;  // [4][nbox]: gz, jx, jy, phi
    const bool lds = P.lds_tally != 0;
    if (lds)
        for (int i = threadIdx.x; i < 4 * P.nbox; i += blockDim.x) sacc[i] = 0.;
    __syncthreads();
    double* tgz = lds ? sacc : P.acc;
    double* tjx = tgz + P.nbox;
    double* tjy = tjx + P.nbox;
    double* tphi = lds ? sacc + 3 * P.nbox : P.phi;
    unsigned long long flights = 0, stuck = 0, badtrans = 0;
    const uint64_t nloop = (P.nin + 63) & ~63ULL;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i - (threadIdx.x & 63) < nloop;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const bool valid = i < P.nin;
        RtaSPart p{};
        bool bounced = false;
        if (valid) {
            p = P.pin[i];
            Pcg32 rng;
            rng.seed(P.key, i);
            int mode = (int)p.mode, box = (int)(p.boxsign >> 1);
            const int sign = (p.boxsign & 1u) ? -1 : 1;
            double4 md = P.modes[mode];
            double dt = -log(1.0 - rng.uniform()) / md.z;
            flights++;
            unsigned long long it = 0;
            int still = 0;  // consecutive crossings without advance
            double x = p.x, y = p.y;
            while (!almost_equal(dt, 0.)) {
                if (++it > P.max_iters || still > 64) { stuck++; break; }
                const DevBox B = P.boxes[box];
                if (B.kind == 2) {
                    const int nb = POLY ? translate_poly(P.boxes, P.sides, P.srange, P.cts, P.cseg, P.ptrans, box, x,
                                                         y, md.x, md.y, rng)
                                        : translate_rect(P.boxes, P.cross, P.ptrans, box, x, y, md.x, md.y, rng);
                    if (nb < 0) { badtrans++; break; }
                    box = nb;
                    continue;
                }
                if (B.kind == 1) break;  // absorbed
                const double vx = md.x, vy = md.y;
                const double nx = x + dt * vx, ny = y + dt * vy;
                int2 sr = make_int2(0, 0);
                if constexpr (POLY) sr = P.srange[box];
                if (POLY ? poly_inside(P.sides, sr, nx, ny) : box_inside(B, nx, ny)) {
                    atomicAdd(tgz + box, sign * dt);
                    atomicAdd(tjx + box, vx * sign * dt);
                    atomicAdd(tjy + box, vy * sign * dt);
                    atomicAdd(tphi + box, (double)sign);
                    break;
                }
                int mask;
                double ex, ey;
                double tf;
                if constexpr (POLY) {
                    tf = poly_exit(P.sides, sr, x, y, vx, vy, mask, ex, ey);
                } else {
                    const double2 iv = P.ivel[mode];
                    tf = box_exit(B, x, y, vx, vy, iv.x, iv.y, mask, ex, ey);
                }
                double left = dt - tf;
                if (almost_equal(left, 0.)) left = 0.;
                still = tf == 0. ? still + 1 : 0;
                atomicAdd(tgz + box, sign * tf);
                atomicAdd(tjx + box, vx * sign * tf);
                atomicAdd(tjy + box, vy * sign * tf);
                int side = 0;
                const int fast = POLY ? poly_side_fast(P.sides, sr, mask, ex, ey, vx, vy, side)
                                      : side_fast(B, mask, ex, ey, vx, vy, side);
                Ids4 pb{};
                int npb;
                if (fast >= 0) {
                    pb.a = fast;
                    npb = 1;
                } else if (fast == SIDE_VOID) {
                    npb = 0;
                } else {
                    npb = POLY ? poly_find_pboxes(P.sides, P.srange, P.cts, B, ex, ey, vx, vy, pb)
                               : find_pboxes(P.boxes, P.cts, B, ex, ey, vx, vy, pb);
                }
                if (npb == 0) {
                    // diffuse wall: Lambert bounce, carried to the next generation
                    const int s = fast == SIDE_VOID ? side
                                : (__popc(mask) == 1 ? __ffs(mask) - 1
                                   : (POLY ? poly_pick_void_side(P.sides, P.srange, P.cts, B, sr, mask, ex, ey, rng.next())
                                           : pick_void_side(P.boxes, P.cts, B, mask, ex, ey, rng.next())));
                    const int4 li = P.lam_info[mode];
                    const int tabk = POLY ? P.sides[sr.x + s].nid : s;
                    bool ng;
                    const int k = (int)alias_pick(P.lam_tab + li.z + (size_t)tabk * li.y, (uint32_t)li.y, rng, ng);
                    mode = P.perm[li.x + k];
                    x = ex;
                    y = ey;
                    bounced = true;
                    break;
                }
                x = ex;
                y = ey;
                if (npb == 1) {
                    box = pb.a;
                } else {
                    Ids4 cand{};
                    int nc = 0;
                    const double cx = ex + 1.0e-6 * vx, cy = ey + 1.0e-6 * vy;
                    for (int k = 0; k < npb && k < 4; k++) {
                        const bool in = POLY ? poly_inside(P.sides, P.srange[pb.get(k)], cx, cy)
                                             : box_inside(P.boxes[pb.get(k)], cx, cy);
                        if (in) cand.set(nc++, pb.get(k));
                    }
                    if (nc > 0) {
                        box = cand.get((int)rng.bounded((uint32_t)nc));
                    } else {
                        box = pb.get((int)rng.bounded((uint32_t)(npb < 4 ? npb : 4)));
                        const DevBox nb = P.boxes[box];
                        if (nb.kind != 2) {
                            const double ccx = POLY ? P.center[box].x : 0.5 * (nb.xmin + nb.xmax);
                            const double ccy = POLY ? P.center[box].y : 0.5 * (nb.ymin + nb.ymax);
                            double dx = ccx - x, dy = ccy - y;
                            double dn = sqrt(dx * dx + dy * dy);
                            x += 1.0e-6 * dx / dn;
                            y += 1.0e-6 * dy / dn;
                        }
                    }
                }
                dt = left;  // a flight ending on a crossing leaves the particle out (as the reference's loop)
            }
            p.x = x;
            p.y = y;
            p.mode = (uint32_t)mode;
            p.boxsign = ((uint32_t)box << 1) | (sign < 0 ? 1u : 0u);
        }
        steady_append(P, bounced, p);
    }
    if (lds) {
        __syncthreads();
        for (int i = threadIdx.x; i < 4 * P.nbox; i += blockDim.x) {
            const double v = sacc[i];
            if (v != 0.) atomicAdd(i < 3 * P.nbox ? P.acc + i : P.phi + (i - 3 * P.nbox), v);
        }
    }
    block_add_u64(P.counters + 1, flights);
    block_add_u64(P.counters + 2, stuck);
    block_add_u64(P.counters + 3, badtrans);
}

// re-emission of |phi(box)| particles per box (RTA_MC2D.cpp:2637-2654)
template <bool POLY>
__global__ __launch_bounds__(256) void rta_steady_regen_kernel(RtaSteadyParams P, uint64_t out0, uint64_t total) {
    unsigned long long stuck = 0;
    for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (uint64_t)gridDim.x * blockDim.x) {
        int lo = 0, hi = P.nbox - 1;  // box b holds [regen[b], regen[b+1])
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (P.regen[mid] <= k) lo = mid; else hi = mid - 1;
        }
        const int b = lo;
        Pcg32 rng;
        rng.seed(P.key ^ 0x5eed5eed5eed5eedULL, k);
        RtaSPart q;
        steady_box_point<POLY>(P, b, rng, q.x, q.y, stuck);
        bool ng;
        q.mode = alias_pick(P.scat, (uint32_t)P.n, rng, ng);
        q.boxsign = ((uint32_t)b << 1) | (P.phi[b] < 0. ? 1u : 0u);
        q.id = out0 + k;
        P.pout[out0 + k] = q;
    }
    if (POLY) block_add_u64(P.counters + 2, stuck);
}

}  // namespace bte

extern "C" int bte_rta_steady_run(bte_ctx* ctx, const bte_modes* mm, const bte_geom* gg, const bte_rta_steady_cfg* cfg,
                                  double* T_out, double* jx_out, double* jy_out, bte_rta_steady_report* rep) {
    BTE_GUARD_BEGIN
    auto* c = reinterpret_cast<Ctx*>(ctx);
    auto* m = reinterpret_cast<const Modes*>(mm);
    auto* g = reinterpret_cast<const Geom*>(gg);
    if (!c || !m || !g || !cfg || !T_out || !jx_out || !jy_out) throw Error(BTE_EINVAL, "null argument");
    if (cfg->nparticles == 0 || !(cfg->thickness > 0)) throw Error(BTE_EINVAL, "bad steady configuration");
    HIPCHECK(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    const int n = m->n, nbox = (int)g->boxes.size();
    for (auto& b : g->boxes)
        if (b.kind == 0) {
            if (b.Teq != cfg->T0) throw Error(BTE_EINVAL, "Tref in xml is different from provided T0");
            if (b.Tinit != b.Teq) throw Error(BTE_EINVAL, "Initial temperature out of reference is not allowed");
        }
    for (int i = 0; i < n; i++)
        if (m->w[i] == 0.) throw Error(BTE_EINVAL, "invalid scattering rate");
    for (int i = 0; i < nbox; i++)
        if (g->dboxes[i].kind == 2 && g->dboxes[i].tgt < 0)
            throw Error(BTE_EGEOM, "periodic box " + std::to_string(i) + " has no translation");
    const double vuc = m->V * cfg->thickness / m->lattz;
    std::vector<double> pmf(n);
    std::vector<uint32_t> th(n), al(n);
    DevBuf<double4> d_modes;
    DevBuf<double2> d_ivel;
    std::vector<double4> md(n);
    std::vector<double2> iv(n);
    for (int i = 0; i < n; i++) {
        md[i] = make_double4(m->vx[i], m->vy[i], m->w[i], m->omega[i]);
        iv[i] = make_double2(m->vx[i] != 0. ? 1.0 / m->vx[i] : 0., m->vy[i] != 0. ? 1.0 / m->vy[i] : 0.);
    }
    d_modes.upload(md, s);
    d_ivel.upload(iv, s);
    // BE_derivative at T0 (re-emission)
    for (int i = 0; i < n; i++) pmf[i] = m->omega[i] <= 0. ? 0. : h_be_kernel(m->omega[i], cfg->T0) * m->w[i];
    if (!build_alias(pmf.data(), n, th.data(), al.data())) throw Error(BTE_EINVAL, "empty scattering pmf");
    DevBuf<uint2> d_scat, d_gen_sel, d_gen_tab, d_gbox_sel, d_gtab, d_lam_tab;
    upload_alias(d_scat, th, al, s);
    // wall generators (RTA_MC2D.cpp:296-347, 366-397)
    std::vector<RtaGen> gens;
    std::vector<double> gw;
    std::vector<uint2> gtab;
    for (int sid = 0; sid < nbox; sid++) {
        const RectBox& sb = g->boxes[sid];
        if (sb.kind != 1) continue;
        for (auto& hc : g->contacts[sid]) {
            const RectBox& cb = g->boxes[hc.box];
            if (cb.kind != 0 || almost_equal(hc.length(), 0.) || almost_equal(sb.Teq, cb.Teq)) continue;
            double cum = wall_pmf(*m, sb.Teq, cb.Teq, hc.npx, hc.npy, pmf.data());
            int sg = (sb.Teq - cb.Teq) >= 0 ? 1 : -1;
            gw.push_back(std::fabs(sg * cum / (m->nq * vuc)) * hc.length() * cfg->thickness);
            if (!build_alias(pmf.data(), n, th.data(), al.data())) throw Error(BTE_EINVAL, "empty wall pmf");
            for (int i = 0; i < n; i++) gtab.push_back(make_uint2(th[i], al[i]));
            gens.push_back(RtaGen{hc.p1x, hc.p1y, hc.p2x - hc.p1x, hc.p2y - hc.p1y, hc.box, sg, 0, 0});
        }
    }
    double Ewall = 0;
    for (double w : gw) Ewall += w;
    // gradient generators: Nabla_T_distribution per regular box
    // (sampling.cpp:118-187; energy vol/vuc * cumulsum / nq, RTA_MC2D.cpp:402-427)
    const double gx = cfg->gradient[0], gy = cfg->gradient[1];
    std::vector<int32_t> gbox, gclass;
    std::vector<double> gE;
    std::vector<uint2> gt;
    if (!almost_equal(std::hypot(gx, gy), 0.)) {
        std::vector<double> pp(n), pm(n);
        for (int b = 0; b < nbox; b++) {
            const RectBox& B = g->boxes[b];
            if (B.kind != 0) continue;
            double acc = 0;
            for (int i = 0; i < n; i++) {
                pp[i] = pm[i] = 0.;
                if (m->omega[i] == 0.) continue;
                const double vgt = -(gx * m->vx[i] + gy * m->vy[i]);
                const double p = std::fabs(vgt * h_be_kernel(m->omega[i], B.Teq));
                acc += p;
                (vgt >= 0. ? pp : pm)[i] = p;
            }
            int cls = 0;
            for (int sgn = 0; sgn < 2; sgn++) {
                if (build_alias((sgn == 0 ? pp : pm).data(), n, th.data(), al.data())) cls |= 1 << sgn;
                for (int i = 0; i < n; i++) gt.push_back(make_uint2(th[i], al[i]));
            }
            gbox.push_back(b);
            gclass.push_back(cls);
            gE.push_back(B.area() * cfg->thickness / vuc * kB * acc / m->nq);
        }
    }
    double Egrad = 0;
    for (double w : gE) Egrad += w;
    const double Etot = Ewall + Egrad;
    if (!(Etot > 0)) throw Error(BTE_EINVAL, "no isothermal walls or gradient sources");
    const double Eeff = Etot / (double)cfg->nparticles;
    std::vector<uint32_t> sth, sal;
    DevBuf<RtaGen> d_gens;
    if (!gens.empty()) {
        sth.resize(gw.size());
        sal.resize(gw.size());
        build_alias(gw.data(), (int)gw.size(), sth.data(), sal.data());
        upload_alias(d_gen_sel, sth, sal, s);
        d_gens.upload(gens, s);
        d_gen_tab.upload(gtab, s);
    }
    DevBuf<int32_t> d_gbox, d_gclass, d_perm, d_mirror;
    if (!gbox.empty()) {
        sth.resize(gE.size());
        sal.resize(gE.size());
        build_alias(gE.data(), (int)gE.size(), sth.data(), sal.data());
        upload_alias(d_gbox_sel, sth, sal, s);
        d_gbox.upload(gbox, s);
        d_gclass.upload(gclass, s);
        d_gtab.upload(gt, s);
    }
    std::vector<int4> info;
    build_lambert(*m, cfg->sigma_bounce > 0 ? cfg->sigma_bounce : 0.25, g->normals, info, d_lam_tab, d_perm, s);
    DevBuf<int4> d_lam_info;
    d_lam_info.upload(info, s);
    const uint64_t cap = cfg->nparticles;
    DevBuf<RtaSPart> d_parts;
    d_parts.alloc(2 * cap);
    DevBuf<double> d_acc, d_phi;
    d_acc.alloc(3 * (size_t)nbox);
    d_phi.alloc(nbox);
    DevBuf<uint64_t> d_regen;
    d_regen.alloc(nbox + 1);
    DevBuf<unsigned long long> d_cnt;
    d_cnt.alloc(4);
    HIPCHECK(hipMemsetAsync(d_acc.p, 0, 3 * (size_t)nbox * sizeof(double), s));
    RtaSteadyParams P{};
    P.modes = d_modes.p;
    P.ivel = d_ivel.p;
    P.scat = d_scat.p;
    P.boxes = g->d_boxes.p;
    P.cts = g->d_contacts.p;
    P.cseg = g->d_cseg.p;
    P.cross = g->d_cross.p;
    P.ptrans = g->d_ptrans.p;
    P.sides = g->d_sides.p;
    P.srange = g->d_srange.p;
    std::vector<double2> centre(nbox);
    for (int i = 0; i < nbox; i++) centre[i] = make_double2(g->boxes[i].cx(), g->boxes[i].cy());
    DevBuf<double2> d_centre;
    d_centre.upload(centre, s);
    P.center = d_centre.p;
    P.lam_info = d_lam_info.p;
    P.lam_tab = d_lam_tab.p;
    P.perm = d_perm.p;
    P.gens = d_gens.p;
    P.gen_sel = d_gen_sel.p;
    P.gen_tab = d_gen_tab.p;
    P.gbox = d_gbox.p;
    P.gbox_sel = d_gbox_sel.p;
    P.gtab = d_gtab.p;
    P.gclass = d_gclass.p;
    P.regen = d_regen.p;
    P.acc = d_acc.p;
    P.phi = d_phi.p;
    P.counters = d_cnt.p;
    P.seed = cfg->seed;
    P.pwall = Ewall / Etot;
    P.max_iters = 1ULL << 26;
    P.n = n;
    P.nbox = nbox;
    P.ngen = (int)gens.size();
    P.ngbox = (int)gbox.size();
    P.lds_tally = nbox <= 1024 ? 1 : 0;
    const size_t lds = P.lds_tally ? 4 * (size_t)nbox * sizeof(double) : 0;
    const int blocks = c->cu_count * 8;
    RtaSPart* buf[2] = {d_parts.p, d_parts.p + cap};
    int cur = 0;
    P.pout = buf[cur];
    hipLaunchKernelGGL(g->poly ? rta_steady_init_kernel<true> : rta_steady_init_kernel<false>, dim3(blocks), dim3(256),
                       0, s, P, cap);
    HIPCHECK(hipGetLastError());
    uint64_t nin = cap;
    std::vector<double> acc(3 * (size_t)nbox, 0.), old(3 * (size_t)nbox), phi(nbox);
    std::vector<uint64_t> pre(nbox + 1, 0);
    int gen = 0;
    bool converged = false;
    unsigned long long flights = 0;
    hipEvent_t e0, e1;
    HIPCHECK(hipEventCreate(&e0));
    HIPCHECK(hipEventCreate(&e1));
    struct EvG {
        hipEvent_t a, b;
        ~EvG() { (void)hipEventDestroy(a); (void)hipEventDestroy(b); }
    } evg{e0, e1};
    double kms = 0;
    const int maxgen = cfg->max_generations > 0 ? cfg->max_generations : 1000000;
    while (nin > 0 && !converged && gen < maxgen) {
        P.pin = buf[cur];
        P.pout = buf[cur ^ 1];
        P.nin = nin;
        uint64_t z = cfg->seed + 0x9e3779b97f4a7c15ULL * (uint64_t)(gen + 1);
        P.key = mix64(z ^ 0x57ead7ULL);
        HIPCHECK(hipMemsetAsync(d_phi.p, 0, nbox * sizeof(double), s));
        HIPCHECK(hipMemsetAsync(d_cnt.p, 0, 4 * sizeof(unsigned long long), s));
        HIPCHECK(hipEventRecord(e0, s));
        hipLaunchKernelGGL(g->poly ? rta_steady_flight_kernel<true> : rta_steady_flight_kernel<false>, dim3(blocks),
                           dim3(256), lds, s, P);
        HIPCHECK(hipGetLastError());
        HIPCHECK(hipEventRecord(e1, s));
        unsigned long long cnt[4];
        old = acc;
        HIPCHECK(hipMemcpyAsync(acc.data(), d_acc.p, acc.size() * sizeof(double), hipMemcpyDeviceToHost, s));
        HIPCHECK(hipMemcpyAsync(phi.data(), d_phi.p, nbox * sizeof(double), hipMemcpyDeviceToHost, s));
        HIPCHECK(hipMemcpyAsync(cnt, d_cnt.p, sizeof(cnt), hipMemcpyDeviceToHost, s));
        HIPCHECK(hipStreamSynchronize(s));
        float ms = 0;
        HIPCHECK(hipEventElapsedTime(&ms, e0, e1));
        kms += ms;
        if (cnt[2]) throw Error(BTE_EGEOM, "a flight exceeded the iteration budget");
        if (cnt[3]) throw Error(BTE_EGEOM, "Error in translation, no box found");
        flights += cnt[1];
        // re-emission counts (RTA_MC2D.cpp:2637-2654); pre outlives the copy
        pre[0] = 0;
        for (int b = 0; b < nbox; b++) {
            const double a = std::fabs(phi[b]);
            pre[b + 1] = pre[b] + (almost_equal(phi[b], 0.) ? 0 : (uint64_t)(a + 1.0e-9));
        }
        const uint64_t nb = cnt[0], nre = pre[nbox];
        if (nb + nre > cap) throw Error(BTE_ECAPACITY, "steady generation larger than the first");
        if (nre) {
            d_regen.upload(pre.data(), nbox + 1, s);
            hipLaunchKernelGGL(g->poly ? rta_steady_regen_kernel<true> : rta_steady_regen_kernel<false>, dim3(blocks),
                               dim3(256), 0, s, P, nb, nre);
            HIPCHECK(hipGetLastError());
        }
        // convergence (RTA_MC2D.cpp:2660-2692)
        auto rel = [&](int q) {
            double d = 0, sq = 0;
            for (int b = 0; b < nbox; b++) {
                const double o = old[(size_t)q * nbox + b], v = acc[(size_t)q * nbox + b];
                d += (o - v) * (o - v);
                sq += v * v;
            }
            return std::sqrt(d) / std::sqrt(sq);
        };
        const double rgz = rel(0), rjx = rel(1), rjy = rel(2);
        if (almost_equal(gx, 0.)) converged = rgz < cfg->eps_energy && rjy < cfg->eps_flux;
        else if (almost_equal(gy, 0.)) converged = rgz < cfg->eps_energy && rjx < cfg->eps_flux;
        else converged = rgz < cfg->eps_energy && rjx < cfg->eps_flux && rjy < cfg->eps_flux;
        nin = nb + nre;
        cur ^= 1;
        gen++;
    }
    HIPCHECK(hipStreamSynchronize(s));
    // post-processing (RTA_MC2D.cpp:2696-2728)
    const double vcorr = cfg->thickness / m->lattz, cv = h_calc_cv(*m, cfg->T0);
    for (int b = 0; b < nbox; b++) {
        const double vbox = g->boxes[b].area() * cfg->thickness;
        T_out[b] = acc[b] / vbox * Eeff / (cv / vcorr) + cfg->T0;
        jx_out[b] = acc[nbox + b] / vbox * Eeff * 1e30;
        jy_out[b] = acc[2 * nbox + b] / vbox * Eeff * 1e30;
    }
    if (rep) {
        rep->generations = gen;
        rep->flights = flights;
        rep->Eeff = Eeff;
        rep->kernel_ms = kms;
        rep->converged = converged ? 1 : 0;
    }
    BTE_GUARD_END
}
