// trk_mc.h -- device layouts of the event transport shared by the host
// driver (trk_mc.hip) and the two compilations of the event code
// (trk_mc_fp64.hip, trk_mc_mx.hip).
#pragma once

#include <hip/hip_runtime.h>
#include "trk_ctx.h"
#include "trk_delta.h"
#include "trk_beb.h"

namespace trk {

// ---------------------------------------------------------------- layouts
// A particle list: one record of 4-byte words per particle, back to back.  A
// wave appends 64 records as one contiguous range, a lane that takes a single
// particle touches one or two cache lines instead of one per field, and the
// event code keeps one address per list in scalar registers.
struct PList {
    uint32_t *w;
};

// Bytes allocated per particle: the FP64 record without and with the fields
// of holes and ions (the mixed path's records are shorter).
constexpr size_t kRecordBytes = 92, kHoleRecordBytes = 112;
inline size_t list_bytes(size_t n, int hole) { return n * (hole ? kHoleRecordBytes : kRecordBytes); }

struct Tally {            // fixed-point difference arrays, replicated R times
    int Nt, NR, nsh, R;
    unsigned long long *cnt_e, *E_e;               // [R][Nt][NR], [R][Nt][NR][2]
    unsigned long long *cnt_h, *E_h, *Ek_h;        // [R][Nt][NR][nsh] (x2 for energies)
    unsigned long long *cnt_p, *E_p;               // [R][Nt][NR]
    unsigned long long *Elat;                      // [R][Nt][NR][2] (not differenced)
};

// Per-iteration snapshot histograms for the tallies the reference normalises
// inside each iteration (Out_Ee_vs_E, Out_Eh_vs_E, Out_theta, Out_theta_h by
// that iteration's particle counts, Out_diff_coeff by its VB-hole count),
// difference arrays over time like the Tally arrays.  b = iteration - iter0.
struct Spec {
    int on, B, ND, iter0;
    int *nel, *nvb, *dcn;          // [B][Nt]
    int *eve;                      // [B][Nt][NR]   electron spectrum, bins of Out_R
    int *ehve;                     // [B][Nt][ND]   VB-hole spectrum, bins of the DOS grid
    int *th, *thh;                 // [B][Nt][180]  polar angle of electrons / moving holes
    unsigned long long *dcs;       // [B][Nt][2]    sum of v*L/3 of mobile holes, fixed point
};

// tables staged in each transport workgroup's LDS (see stage_tables)
constexpr int kStaged = 34;

// The ion of one impact: its parameters and its own tables (SHI_MFP, the
// fused SHI_path, diff_SHI_MFP at its initial energy and the mixed path's
// per-shell transfer constants).  A context has one; a batch keeps one per
// impact in device memory, read by the lanes that run an ion's collision.
struct IonDev {
    double mass, E0, Zeff0, fixed_zeff;   // [proton masses], [eV], charge at E0, fixed charge
    int Z, kind_zeff, nS, pad_;
    const double *ES, *LSsh, *shi_path, *lnES, *ln_LSsh, *ln_shi_path;
    const int *sd_n; const int64_t *sd_off; const double *sd_E, *sd_L, *sd_inv; const int *sd_nonmono;
    const int *sd_M; const double *sd_c; const int *sd_bk;
};

// Round state of one material group of a batch (device memory): particles
// of the current round by kind, the next round's allocation counters by list
// parity, the shared cursor and the parity of the current round's lists.
struct GroupCtl {
    int n_in[4];
    int out_cnt[2][4];
    int cursor;
    int cur;
    int overflow;
    int ion_cursor;
};

// Control of a batch launch (device memory): the grid barrier, the round
// number, the end flag, and the error bits (barrier time-out).
struct BatchCtl {
    unsigned bar_count, bar_gen;
    int done, err;
    int round, n_groups;
    unsigned long long deadline_ticks;   // wall-clock ticks a barrier may wait
};
constexpr int kBatchErrBarrier = 1;
constexpr int kMaxGroups = 8;

struct McDev {
    MatDev m;
    // tables
    int nE; const double *E, *Lsh, *el_imfp; const int64_t *roff; const double *rhw, *rlam;
    int nEel; const double *Eel, *Lel; const int64_t *roff_el; const double *rhw_el, *rlam_el;
    int nH; const double *EH, *LHsh, *hole_imfp; const int64_t *roff_h; const double *rhw_h, *rlam_h;
    int nHel; const double *EHel, *LHel; const int64_t *roff_hel; const double *rhw_hel, *rlam_hel;
    // 1 per cumulative row whose lam never increases (counted search)
    const unsigned char *rmono, *rmono_h, *rmono_el, *rmono_hel;
    int nP; const double *EP, *LPsh, *phot_imfp;
    int nS; const double *ES, *LSsh, *shi_path;
    const int *sd_n; const int64_t *sd_off; const double *sd_E, *sd_L, *sd_inv; const int *sd_nonmono;
    // logs of grids and fused tables (interpolation without per-node logs)
    const double *lnE, *ln_el_imfp, *lnEel, *ln_Lel, *lnEH, *ln_hole_imfp, *lnEHel, *ln_LHel;
    // logs of the per-shell paths and of the cumulative transfer rows
    const double *ln_Lsh, *ln_LHsh;
    const double *ln_rhw, *ln_rlam, *ln_rhw_h, *ln_rlam_h, *ln_rhw_el, *ln_rlam_el, *ln_rhw_hel, *ln_rlam_hel;
    // run
    uint64_t seed;
    double T_last, Tim, cutoff_eff;
    int Nt; const double *tim_glob;
    double inv_dt;                      // 1/dt of a linear time grid, 0 otherwise
    int hints;                          // 1: the electron and hole energy grids, the time grid and Out_R are strictly increasing
    // tables copied into each transport workgroup's LDS (count and offset in
    // doubles; count 0 = read from global memory), see kStage* below
    int lds_n[kStaged], lds_off[kStaged];
    int NR; const double *R;
    int include_photons;
    // lists, by kind: electrons, holes, photons, ions
    PList in[4], out[4];
    int n_in[4];                        // particles of the current round
    int cap[4];                         // capacity of each list
    int *out_cnt;                       // [4] allocation counters of the next round
    int *cursor;                        // next item of the current round
    int *overflow;
    unsigned long long *counters;       // [16] event counters
    double *trace; unsigned long long *trace_n; long long trace_cap;
    Tally T;
    Spec S;
    // the ion's collisions: per-shell constants of its transfer's draw
    // (k_shi_consts) with the index of its rows by draw (k_shi_buckets), logs
    // of the SHI grid, of its per-shell paths and of the fused path
    const int *sd_M; const double *sd_c; const int *sd_bk;
    const double *lnES, *ln_LSsh, *ln_shi_path;
    // batch runs only: the impacts' ions (indexed by iteration - iter0), this
    // group's round state
    const IonDev *ions;
    const int *plane_of;        // tally plane of each impact in its group
    uint32_t iter0;
    int round_events;           // events a particle may take per round (round_budget)
    GroupCtl *gctl;
    // emission through the surface Z = 0 (em_W, the work function, > 0): the
    // barrier height, the E1 and gamma of its logistic transmission, and the
    // per-iteration tallies of the emitted electrons while S.on (indexed like
    // S): counts [B][Nt], kinetic energies [B][Nt][2] (fixed point) and
    // spectrum [B][Nt][NR] on the energy grid RE = Out_R/10, all difference
    // arrays over time
    double em_W, em_H, em_E1, em_gamma;
    const double *RE;
    int *em_n, *em_h;
    unsigned long long *em_e;
    // the oscillators' Delta-CDF weights (kind_of_DR = 4), indexed like m.oE0;
    // per shell, the electron and hole cross section (2: BEB) and the mean
    // kinetic energy of the shell's electrons (both read by the general
    // transport kernel only)
    const double *delta_alpha;
    const int *beb_kocs;
    const double *beb_Ek;
    // DSF elastic scattering (kind_of_EMFP = 2) of electrons [0] and holes [1]
    DsfDev dsf[2];
    // the next ion of the current round and the collisions an ion may take in it
    int *ion_cursor;
    int ion_events;
    // lanes of a wave that take particles (run_items)
    int lane_cap;
};

enum { EV_SHI = 0, EV_E_INEL, EV_E_EL, EV_H_INEL, EV_H_EL, EV_AUGER, EV_RAD, EV_PHOT };

// d.overflow bits: list capacities, the per-particle event limit, NaN state.
constexpr int kFlagPairs = 1, kFlagPhotons = 2, kFlagEvents = 4, kFlagNaN = 8;
// Events one particle may take over all rounds.  A history needs a few
// thousand at most, an ion 10^5; the limit only guarantees that every run ends.
constexpr uint32_t kMaxEvents = 1u << 22;

enum { K_EL = 0, K_HO = 1, K_PH = 2, K_ION = 3 };

enum { C_E_EL = 0, C_E_INEL, C_H_EL, C_H_INEL, C_DEEP, C_PHOT, C_COUNT };

// A wave runs a category of events only when at least this many of its lanes
// want it (or when it is the most wanted one); the other lanes wait with
// their state untouched.  Rare, long branches (ionisation, decays) then run
// for many lanes at once instead of stalling the wave at almost every step.
constexpr int kBatchLanes = 16;
constexpr int kMaxWait = 16;

// A moving particle's flight over more nodes than this is tallied by its whole
// wave.  One lane needs about 2800 cycles a node (shared with the wave's other
// long flights), the wave about 2000 cycles a flight.
constexpr int kWaveNodes = 3;

// Events one particle may take in one round.  A particle with more left is
// written to the next round's list; this bounds the tail of every launch by
// the cost of kRoundEvents events instead of the longest history.
constexpr uint32_t kRoundEvents = 512;

// The budget of a round of n particles on `lanes` lanes.  A round lasts until
// its longest history has used the budget, and children wait for its end:
// with few particles a lane, a smaller budget starts them earlier.  Below 128
// the rounds' own cost (a launch, the staging, a read of the counts) shows;
// with eight budgets' worth of particles a lane the end of a round does not.
// Budgets of 512 against this rule: 25 oxide iterations 16.7 -> 11.9 ms, 1000
// of them in FP64 240 -> 217, the track target 42 -> 37; 128 for every round
// made 4001 oxide iterations slower (430 -> 490).  free: only where the lists are
// long (the ions may run on beyond the budget), since particles that wait
// between rounds take room in them.
TRK_HD int round_budget(long long n, long long lanes, int budget, bool free)
{
    const long long b = 8 * n / lanes;
    if (!free || b >= budget) return budget;
    return b > 128 ? (int)b : (budget < 128 ? budget : 128);
}

extern __shared__ double lds_tab[];

// The sources a path's kernels are spread over (TRK_PART): the transport of
// single runs with its set-up kernels, the ions and the general transfers, and
// the batch kernels.
#define TRK_PART_RUN 0
#define TRK_PART_GENERAL 1
#define TRK_PART_BATCH 2

// Transport workgroup of each path: one per CU (the staged tables fill most
// of the LDS), 12 waves, 3 per SIMD (168 VGPRs).  At 16 waves the mixed
// path would have to spill to scratch, which costs more than the fourth
// wave gains.
constexpr int kTransportBlockFp64 = 768;
constexpr int kTransportBlockMx = 768;

// Workgroup of the ion kernel: 8 waves, each with one ion, 2 per SIMD.
constexpr int kIonBlock = 512;

// The ions' workgroups of a batch: those of group g start at first[g], each
// with waves[g] ions at a time.
struct BatchIons {
    int first[kMaxGroups + 1], waves[kMaxGroups];
};

// Waves per workgroup for n ions and at most `groups` workgroups: one ion per CU
// while there are few, up to the workgroup's eight.
inline int ion_waves(int64_t n, int64_t groups)
{
    const int64_t per = (n + groups - 1) / groups;
    return (int)(per < kIonBlock / 64 ? per : kIonBlock / 64);
}

// The event code is compiled twice, into namespaces fp64 (deterministic
// FP64, replays the oracle bit for bit) and mx (mixed precision); these are
// the kernels the host driver launches from each.
#define TRK_MC_KERNELS                                                          \
    template <bool kAll, bool kGeneral> __global__ void k_transport(McDev din); \
    template <bool kAll> __global__ void k_ions(McDev din, int waves);       \
    __global__ void k_ion_init(McDev d, int nb, uint32_t first_iter);        \
    __global__ void k_shi_consts(IonDev iv, const double *Ip, int nsh, int *sd_M, double *sd_c); \
    __global__ void k_shi_buckets(IonDev iv, int nsh, const int *sd_M, const double *sd_c, int *sd_bk); \
    template <bool kAll> __global__ void k_batch(BatchCtl *ctl, int n_groups); \
    template <bool kAll> __global__ void k_batch_ions(BatchIons bi, int n_groups); \
    __global__ void k_ion_init_batch(int g, int nb, const int *idx);        \
    hipError_t batch_upload(const McDev *mc, int n_groups, hipStream_t st);
namespace fp64 { TRK_MC_KERNELS }
namespace mx { TRK_MC_KERNELS }
#undef TRK_MC_KERNELS

// The ion view of a context's own ion (host side).
IonDev ion_view_host(const trk_ctx *c);
hipError_t launch_shi_consts(const trk_ctx *c, const IonDev &iv, bool mixed, hipStream_t st);
// Transport descriptor of a context's tables (trk_mc.hip).
void fill_mcdev(const trk_ctx *c, McDev &d);
// LDS layout of the staged tables (trk_mc.hip); true when all are staged.
bool plan_lds(McDev &d, int Nt, int NR, int n_dos, int nsh, size_t limit_doubles, size_t *bytes);
// Collisions an ion may take in one round: all of them while the pairs they
// make (expected number) take a quarter of the lists at most, else as many as
// do, and never fewer than the other particles' budget (deep = false: just
// that).  A run whose lists overflow is repeated with deep = false, so that
// no list has to be longer than with one budget for all.
static inline int ion_round_events(double pairs, int n_ions, int cap, int round_events, bool deep)
{
    if (!deep) return round_events;
    if (pairs <= 0.25 * cap) return 1 << 30;
    const int n = (int)(0.25 * cap / n_ions);
    return n > round_events ? n : round_events;
}
// BEB shells or the Delta-CDF model: the transport kernel's general instantiation
bool uses_general_kernel(const HostMat &h);
// The running sums over time of the tally planes of T, energies as split words
// (split) or as 128-bit integers.
hipError_t launch_time_prefix(const Tally &T, int planes, bool split, hipStream_t st);
// Staging of one plane's finished tallies: device and page-locked host values.
// The device values lie in memory that the object (context or batch) has
// anyway and does not use between a run's transport and the next run, its
// particle lists; only lists shorter than the results need a buffer of their
// own.  Reserved before the transport, so that a run which cannot have its
// memory fails before it has done its work; the host values and the buffer are
// kept by the object and grown to the largest plane it was asked for.
struct FinStage {
    double *dev = nullptr, *pin = nullptr;
    unsigned long long *node_sums = nullptr;   // [Nt][4]: lattice energy of the node, the rest of tot_E
    hipEvent_t done = nullptr;                 // the values are in pin
    size_t n = 0, node_n = 0;                  // what dev and node_sums hold
    void *own = nullptr;
    size_t own_bytes = 0, pin_n = 0;
    bool locked = false;                       // pin is page-locked
    int reserve(size_t values, size_t nodes, void *room, size_t room_bytes);
    void release();
};
// values already on the device that a run adds to another of the caller's arrays
struct FinExtra {
    const double *dev;
    double *dst;
    size_t n;
};
// Values that the finished tallies of a run with these Out_* arrays hold.
size_t finish_values(const trk_ctx *c, int NR, const trk_tallies *out, const std::vector<FinExtra> *extra = nullptr);
// One tally plane converted on the device and copied to the reserved stage, and then
// added into the caller's Out_* arrays (trk_mc.hip).  d_V: Out_V on the device.
int finish_begin(trk_ctx *c, FinStage &fs, const Tally &T, int plane_index, const double *d_V, int NR,
                 const trk_tallies *out, hipStream_t st, const std::vector<FinExtra> *extra = nullptr);
int finish_end(trk_ctx *c, FinStage &fs, int NR, trk_tallies *out, const std::vector<FinExtra> *extra = nullptr);

// 128-bit tally words: (low, high) 64-bit halves of an exact integer
TRK_DEV __int128 fx_read(const unsigned long long *p)
{
    return (__int128)(long long)p[1] * ((__int128)1 << 32) + (__int128)p[0];
}

TRK_DEV void i128_store(unsigned long long *p, __int128 v)
{
    p[0] = (unsigned long long)v;
    p[1] = (unsigned long long)(v >> 64);
}

TRK_DEV __int128 i128_load(const unsigned long long *p)
{
    return (__int128)(((unsigned __int128)p[1] << 64) | (unsigned __int128)p[0]);
}

}  // namespace trk
