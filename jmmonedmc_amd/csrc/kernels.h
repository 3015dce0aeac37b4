// kernels.h -- device data layout and the gfx950 kernels of the engine.
//
// HBM layout (one engine):
//   x        double[sum N]     chain positions, sorted, chains in bundle order
//   chains   DevChain[n]       read-only per-chain constants
//   states   DevState[n]       L, U, sweep counter, cumulative counters
//   sU, sL   double[cap][n]    per-sweep samples, one row per sweep (coalesced)
//   sA       uint2[cap][n]     accepted displacements / box-length trials
//   sW, sH   double[cap][n]    virial and hypervirial after each sweep (optional)
//   bundles  DevBundle[m]      work items: chains packed into one workgroup
//   slots    DevSlot[...]      chain -> lane range and LDS offset in a bundle
//
// Sweep schedule (shared with the oracle): chain c's N particles form B_c
// blocks (B_c a power of two or whole waves, every block at least M_min
// particles); in phase t every block updates its t-th particle.  Trials in
// one phase are at least M_min apart in index order, and M_min is chosen so
// that no two of them can interact or read each other's particle: every
// neighbour gap stays at least the hard core g_min (moves that would break
// it are rejected), so a partner within the cutoff rc is at most
// w = floor(rc/g_min) places away, and M_min = w + 1 (or NBN + 1, and at
// least 2 because the hard-core test reads both nearest partners).  A phase
// is therefore equivalent to running its trials one after another in any
// order.
//
// LDS layout of a chain inside a bundle (batched forms): ghost-left (wg),
// B blocks at an odd stride Sp, ghost-right (wg); see LdsChain.
#pragma once

#include "jmm_device.h"

namespace jmm {

enum : uint32_t { F_PERIODIC = 1u, F_NPT = 2u, F_VOLLOG = 4u };

struct DevChain {
    uint64_t seed;
    uint64_t x_off;   // first position of this chain in x[]
    uint64_t log_off; // first byte of this chain's accept log
    uint32_t N, B, w, smax;
    uint32_t chain_id, eci, flags, kind;
    uint32_t wg, Sp;  // LDS layout: ghost width max(w, 1), odd block stride >= smax
    uint32_t lds_len; // LDS doubles of the chain's region: 2 wg + B Sp
    uint32_t nbn_lim;  // NBN partner limit (UINT32_MAX: none)
    double beta, P, max_step, max_dv, gmin, Lmin;
    double sh[3];  // shifted form at the cutoff: E, dE/dtheta0, dE/dtheta1
    Pot pot;
    float betaf, pad[3];
};

struct DevState {
    double L, U;
    uint64_t sweep;
    uint64_t cnt[8];  // trials, acc_d, wall, core, pair_terms, vol_trials, acc_v, recomputes
    double max_drift;
};

struct DevBundle {
    uint32_t slot0, nslots, lanes, smax;
    uint32_t lds_doubles, kind, global_x, pad;
    uint64_t x_off;
};

struct DevSlot {
    uint32_t chain, lane_off, B, lds_off;
};

struct Ctrl {
    uint32_t queue, sample_off, next_off, pad;
};

struct SweepArgs {
    const DevChain *chains;
    DevState *states;
    double *x;
    const DevBundle *bundles;
    const DevSlot *slots;
    const uint32_t *plain_list;  // plain form: chains of this launch
    Ctrl *ctrl;
    double *sU, *sL;
    uint2 *sA;
    double *sW, *sH;  // nullable: per-sweep virial and hypervirial rows
    uint8_t *acclog;
    uint32_t n_items, n_sweeps, n_chains, cap;
};

// A tile of a chain's configuration: its part-th run of a tile's particles.
struct Tile {
    uint32_t chain, part;
};

// Configurations of up to OBS_ONE particles are one workgroup's (a particle
// per lane, nothing to add afterwards); longer ones are cut into tiles of
// OBS_TILE, summed by a second launch (about 3 us, against 30 us saved per
// 1024 particles of a configuration that one workgroup walks in turn).  Tiles
// of 512 rather than 256 halve the pairs evaluated again at their edges: FP32
// Yukawa of 65,536 with gradients, both launches, 12 configurations 54 against
// 56 us, one 21.4 against 22.8 us.
constexpr uint32_t OBS_ONE = 1024, OBS_TILE = 512;

struct ObsArgs {
    const DevChain *chains;  // engine form (nullable)
    const DevState *states;  // engine form: the chains' lengths
    DevChain one;            // standalone form
    const double *x;
    const double *L;         // standalone form
    const Tile *tiles;       // engine form, nullable: tiles of all chains in chain order
    const uint32_t *first;   // engine form with tiles: [n + 1], first tile of each chain
    const double *Lnew;      // engine form, nullable: evaluate at x * Lnew/L, length Lnew
    double *part;            // nullable: [tile][6] partial sums, for k_obs_sum
    double *obs;
    double *grad;
    const uint32_t *row;     // engine form, nullable: output row of each chain (else its index)
    const uint64_t *goff;    // engine form, nullable: gradient offset of each chain (else x_off)
    uint32_t tile, parts;    // particles per workgroup; standalone form: workgroups per configuration
    uint32_t standalone;
    uint32_t group0;         // first workgroup of this launch
};

// A chain too large for one workgroup's LDS is split into S segments of Bs
// consecutive blocks, one workgroup each (one launch, all resident).
struct DevSeg {
    uint32_t chain;  // internal chain index
    uint32_t s, S;   // segment index, segments of the chain
    uint32_t Bs;     // blocks (lanes) in each segment
    uint32_t first;  // index of the chain's segment 0 in the per-segment arrays
    uint32_t pad[3];
};

// Per-segment partial sums: [segment][sweep parity][field][wave of the
// segment's workgroup], fields dU, box-length dU, accepts, overlaps,
// recomputed U, final counters, virial, hypervirial, the FP32 form's
// configuration energy from the box-length pass.
constexpr uint32_t SEG_FIELDS = 9, SEG_WAVES = 4;

struct SegArgs {
    SweepArgs a;
    const DevSeg *segs;
    double *pub_head, *pub_tail;  // [segment][wgmax]: first / last wg positions
    unsigned long long *ctr;      // [segment]: synchronisation points passed
    double *part;                 // [segment][2][SEG_FIELDS][SEG_WAVES]
    uint32_t *err;                // set when a wait times out
    uint32_t wgmax, n_segs;
};

// Histogram kernel: lanes of a workgroup (HIST_TILE of them without g(x), which
// has one count a particle), particles of a tile (short chains: fewer, with more
// lanes a particle), 32-bit counters in LDS (64 KB: two workgroups per CU), and
// the longest chain whose tiles cannot overflow them (HIST_TILE particles, N - 1
// partners, both members).
constexpr uint32_t HIST_T = 1024, HIST_TILE = 256, HIST_WORDS = 16384, HIST_N_LDS = 1u << 22;

__host__ __device__ inline uint32_t hist_tile(uint32_t N) { return N <= 64 ? 64u : N <= 128 ? 128u : HIST_TILE; }

// rho(x) and g(x) histograms of every chain's current configuration.
struct HistArgs {
    const DevChain *chains;
    const DevState *states;
    const double *x;
    const Tile *tiles;        // of all chains
    unsigned long long *rho;  // [chain][rhonb]
    unsigned long long *g;    // [chain][gns][gnb]
    double rbw, gsw, gbw;
    uint32_t n_tiles, rhonb, gns, gnb;
    uint32_t group0;          // first workgroup of this launch
};

}  // namespace jmm

namespace jmm {
// Where a block's box-length sums are cut in two: sums over the block
// positions [0, h) and [h, size) are formed apart and added, so that two lanes
// can share a block (the split kernel) and one lane gives the same bits.
// Short blocks are not cut: the second walk would cost more than half of one
// (the 20 sigma Yukawa chains, which the cut is for, have blocks of at least 41).
constexpr uint32_t HALF_MIN = 40;

hipError_t launch_begin(Ctrl *c, uint32_t n, hipStream_t s);
// waves: per SIMD, 2 or (T = 256 in LDS) 3
const void *batched_kernel(int fp32, int T, int gx, int waves);
hipError_t launch_batched(const SweepArgs &a, int fp32, int T, int gx, int waves, uint32_t grid, size_t lds,
                          hipStream_t s);
// Cooperative form: one chain per workgroup of at most COOP_T lanes (512: two
// waves per SIMD, so 256 registers; 1024 lanes with 128 spilled), 16, 4 or 2
// lanes per block; chains with at most COOP_W partners per side and COOP_B
// blocks.
constexpr uint32_t COOP_W = 8, COOP_B = 256, COOP_T = 512;
__host__ __device__ inline uint32_t coop_lanes(uint32_t B) { return B <= 32 ? 16u : B <= 128 ? 4u : 2u; }
size_t coop_lds(const DevChain &c);
uint32_t coop_threads(const DevChain &c);
const void *coop_kernel(int fp32);
hipError_t launch_coop(const SweepArgs &a, int fp32, uint32_t grid, uint32_t threads, size_t lds, hipStream_t s);
const void *plain_kernel(int gx);
hipError_t launch_plain(const SweepArgs &a, int gx, uint32_t grid, size_t lds, hipStream_t s);
hipError_t launch_observables(const ObsArgs &a, int fp32, uint32_t n_tiles, uint32_t n_configs, int threads,
                              hipStream_t s);
// Samples in the caller's layout (jmm_sample): out[ext[k] * n_sweeps + s]
// from the engine's [sweep][chain] arrays.
struct SampleRec {
    double U, L;
    uint32_t acc_d, acc_v;
};
static_assert(sizeof(SampleRec) == 24, "SampleRec must match jmm_sample");
hipError_t launch_pack_samples(const double *sU, const double *sL, const uint2 *sA, const uint32_t *ext,
                               uint32_t n_chains, uint32_t n_sweeps, SampleRec *out, Ctrl *ctrl, uint32_t n_ctrl,
                               hipStream_t s);
// Virial rows to the caller's layout: out[(ext[k] * n_sweeps + s) * 2 + {0, 1}]
// = (W, HV) of sweep s.
hipError_t launch_pack_virials(const double *sW, const double *sH, const uint32_t *ext, uint32_t n_chains,
                               uint32_t n_sweeps, double *out, hipStream_t s);
hipError_t launch_hist(const HistArgs &a, hipStream_t s);
// tw: workgroup width (256 or 512); lpb: lanes per block (1 or 2; 512 only with 2)
const void *segmented_kernel(int fp32, int tw, int lpb);
hipError_t launch_segmented(const SegArgs &a, int fp32, int tw, int lpb, size_t lds, hipStream_t s);
hipError_t launch_rescale(const DevChain *chains, const DevState *st, double *x, const double *Lnew,
                          uint32_t n_chains, uint32_t parts, hipStream_t s);
}  // namespace jmm
