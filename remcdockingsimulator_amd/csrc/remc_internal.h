// remc_internal.h -- device data layout shared by the kernels and the C-ABI
// implementation.  Everything lives in HBM as structure-of-arrays:
//
//   static, per bead (all systems concatenated, index sys.bead_off + b):
//     tc   int    type | crowder<<8
//     q    float  charge
//     sig  float  vdW radius
//     body int    body index local to the system
//   static, per body (index sys.body_off + m): bstart, bend (local bead
//     indices), bcrow (crowder flag)
//   dynamic, per replica bead (index rep.bead_off + b): px,py,pz positions,
//     rx,ry,rz positions relative to the body centre
//   dynamic, per replica body (index rep.body_off + m): cx,cy,cz centre,
//     quat[4*(...)] rotation (w,x,y,z) in FP64
//   dynamic, per replica: E (FP64, kcal/mol), T (FP64), step (RNG counter),
//     cnt[3] accept/accept_boltz/reject
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "remc.h"

namespace remc {

struct DevSys {
    int bead_off, n_beads, body_off, n_bodies;
    int max_body, rep_first, n_rep, slot_off;
    float box, inv_box;
    int grp_off; // groups of 16 beads of the systems before it
    int n_multi; // bodies of several beads
    double unit; // units of contact distances per Angstrom: 2^32 / box where they are fractions of it, else 1
};

// Boxes whose coordinates the all-pairs kernels take as 32-bit fractions
constexpr float FIX_BOX_MAX = 1024.0f;
__host__ __device__ inline bool box_in_fractions(float box) { return box > 0.0f && box <= FIX_BOX_MAX; }
// Boxes in whose units the MC kernel forms the distances of its large moves:
// there must be one, and the crowder term's sixth powers must be normal numbers
// (in a box of 1e6 A the constant is above 1e-33 and the power below 1e38 beyond
// 0.4 A; at 1e7 A both leave single precision).
constexpr float UNIT_BOX_MAX = 1.0e6f;
__host__ __device__ inline bool box_is_unit(float inv_box) { return inv_box >= 1.0f / UNIT_BOX_MAX; }

struct DevRep {
    int sys, bead_off, body_off;
    uint32_t rng_id;
    float tstep;
    int grp_off; // groups of 16 beads of the replicas before it
    double rot_ch, rot_sh;
    double rstep; // rotate step (rad)
};

// prescaled force field: etab[i*20+j] = lambda*(table-e0)*lj_cf*kbt_cf
struct DevFF {
    float c_crow;    // lj_cf*kbt_cf (crowder term coefficient)
    float crow_s2;   // crowder sigma^2
    float crow_cut2; // crowder cutoff^2
    float c_dh;      // dh_cf*kbt_cf
    float k_dh;      // -log2(e)/xi, exp(-r/xi) = exp2(r*k_dh)
    float eps_r;     // 1e-38 added to r
    float crow_k;    // c_crow * crow_s2^3: crowder term = crow_k / r^6
    float crow_cut;  // crowder cutoff
};

// One workgroup of the MC kernel: member c of the coop workgroups of replica r
// (r < 0: none), and where its copy of the replica's state begins in the dynamic
// arrays (member 0's is the canonical one).
struct McWg {
    int r, c, coop, pad;
    long long bead, body;
};

struct KParams {
    // static
    const int *tc;
    const float *q;
    const float *sig;
    const int *body;
    const int *bstart;
    const int *bend;
    const int *bcrow;
    const int *border; // the system's bodies (local), those of several beads first
    const int *grp; // per group of 16 beads (sys.grp_off + g): first body, last body, kinds of beads | beads << 8, mask of charged beads
    const DevSys *sys;
    const DevRep *rep;
    const float *etab;
    const float *sstab; // per system: (0.5 (sigma_i + sigma_j))^2 of type pairs, over box^2 and as it is (when sigtab)
    int sigtab;         // 1: every non-crowder bead's sigma is its type's
    DevFF ff;
    // dynamic
    float *px, *py, *pz, *rx, *ry, *rz, *cx, *cy, *cz;
    double *quat;
    double *E, *T;
    unsigned long long *step;
    unsigned long long *cnt;
    // exchange ladder
    int *slot_rep;          // per system slots: slot_rep[sys.slot_off + k]
    double *ladder;         // ladder[sys.slot_off + k]
    unsigned long long *ex_round;  // per system
    int *ex_offset;         // per system
    unsigned long long *ex_swaps;  // per system cumulative
    // cooperative MC: private state copies and partial-dE slots
    int n_rep;
    int coop_min_pairs;     // moves with fewer pair terms are not split across members
    size_t copy_beads;      // stride between state copies (beads)
    size_t copy_bodies;     // stride between state copies (bodies)
    unsigned long long *slots; // n_rep x 2 banks of REMC_SLOT_K x slot_row tagged partial sums
    int slot_row;           // entries of a row: REMC_MAX_COOP, or REMC_MAX_MEMBERS where a replica has more members
    const McWg *wg;         // the launch's workgroups
    int *err;               // set when a member waited too long
    // MC dynamic LDS: moved-body staging size and partner-bead/body caches
    int lds_mb;             // largest body (beads)
    int lds_cl;             // cached partner beads per workgroup (0 = no cache)
    int lds_nbody;          // cached bodies per workgroup (0 = none)
    int cache_slice;        // 1: each member caches only its partner slice
    int cache_bodies;       // 1: body ranges and centres cached
    int cache_rel;          // 1: relative positions cached (full partner cache only)
    int cache_quat;         // 1: body rotations cached (with the body table)
    int spec;               // 1: speculative windows of small moves (needs the full caches)
    int draw2;              // 1: a second draw batch in dynamic LDS, formed ahead
    // recording
    remc_step_record *rec;
    unsigned long long *rec_start;
    int rec_max;
    uint32_t key0, key1;
};

// launchers (remc_kernels.hip)
// p.wg holds grid workgroups; shared: some replica has several members
hipError_t launch_mc(const KParams &p, int grid, bool shared, int nsteps, int block, hipStream_t s);
// copies every replica's canonical state to the copies of its other members
hipError_t launch_copy_state(const KParams &p, int grid, hipStream_t s);
size_t mc_dynamic_lds(const KParams &p);
// static LDS of the MC kernel at this block size (its largest variant), or -1
int mc_static_lds(int block);
size_t mc_draw_batch_bytes(); // LDS of one batch of MC step draws
hipError_t launch_mc_fb(const KParams &p, int n_rep, int nsteps, int block, int coop, hipStream_t s);
hipError_t mc_fb_max_active_per_cu(const KParams &p, int block, int *out);
size_t mc_fb_dynamic_lds(const KParams &p);
hipError_t mc_max_active_per_cu(const KParams &p, int block, int *out);
// How the host learns that a kernel's results are in pinned memory: the last workgroup
// (counted in *count, which is left at 0) writes ticket to *flag.
struct Signal {
    uint32_t *count, *flag;
    uint32_t ticket;
};
// A result's store to pinned memory: written through to the host, so that its
// completion (counted by the wave) is its visibility, with no cache to flush.
template <typename T>
__device__ __forceinline__ void host_store(T *ptr, T v)
{
    __hip_atomic_store(ptr, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Called by every thread of every workgroup after its host_store's (no flag:
// nobody waits for it).  Every wave waits for its own stores, so the last
// workgroup to count itself stores the ticket after all of them.  (A system
// fence here writes back the L2 for every wave: 25 us in a gather of 476 KB.)
__device__ __forceinline__ void signal_done(const Signal &sig)
{
    if (!sig.flag) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        // wraps to 0 with the last workgroup
        const uint32_t before = atomicInc(sig.count, gridDim.x - 1);
        if (before == gridDim.x - 1) host_store(sig.flag, sig.ticket);
    }
}

// full energies of n_rep replicas of at most max_beads beads: fix holds
// fix_ints(...) ints (scratch), partials n_rep x full_units(...) doubles
hipError_t launch_energy_full(const KParams &p, int n_rep, int max_beads, int *fix, double *partials, double *out,
                              int noncrowder_only, int write_E, hipStream_t s, const Signal &sig = Signal{});
int full_units(int n_rep, int max_beads);
constexpr int GROUP = 16;                          // beads of a column group of the all-pairs kernels
constexpr int GROUP_CHAIN = 1, GROUP_CROWDER = 2; // kinds of beads present (KParams::grp)
__host__ __device__ inline int full_groups(int beads) { return (beads + GROUP - 1) / GROUP; }
// k_fix's output: coordinates as fractions of the box of all replicas, then
// (16-byte aligned) the groups' ranges
__host__ __device__ inline size_t fix_centres(size_t beads) { return (3 * beads + 3) / 4 * 4; }
inline size_t fix_ints(size_t beads, size_t groups) { return fix_centres(beads) + 4 * groups; }
hipError_t launch_energy_plain(const KParams &p, int replica, int n_beads, int block, float *partials, hipStream_t s);
hipError_t launch_exchange(const KParams &p, int n_sys, hipStream_t s);
// adjoint launch plan for n_rep replicas of at most max_beads beads whose
// beads span bead_stride entries of the replica arrays: row tiles, partner
// sub-ranges and the scratch they need (per-sub-range bead gradients, then
// per-workgroup parameter partials)
struct AdjPlan {
    int tiles, split, sub_len;
    size_t part_doubles, param_doubles;
};
// target_wg: the workgroups a launch aims at (0: the size rule's 2048);
// sub-ranges are cut only while the launch holds fewer
AdjPlan adjoint_plan(int n_rep, int max_beads, size_t bead_stride, int target_wg = 0);
hipError_t launch_adjoint(const KParams &p, const void *adj_ff, const AdjPlan &a, int rep_first, int n_rep,
                          int max_beads, int body_waves, int bead_base, size_t bead_stride, int body_base, int *fix,
                          double *scratch, double *force_torque, double *dparams, hipStream_t s);
hipError_t launch_drms(const KParams &p, int sys_id, int n_beads, int n_rep, const float *rx, const float *ry,
                       const float *rz, double *partials, double inv_pairs, double *out, const Signal &sig, hipStream_t s);
size_t drms_units(int n_beads, int n_rep); // partials of launch_drms per replica
// part: hist_workgroups(...) x nh 32-bit counts; the result goes to gr when it
// is given, else to counts
int hist_workgroups(int n_bodies, int n_rep, int nh);
hipError_t launch_centre_hist(const KParams &p, int sys_id, int n_bodies, int n_rep, const int *btype, const int *site,
                              int n_types, int nbin, double lo, double dr, unsigned int *part, const int *type_count,
                              double frames_over_volume, unsigned long long *counts, double *gr, const Signal &sig, hipStream_t s);
// Up to GATHER_MAX device arrays read back by one launch: array k's words go to
// dst[at[k]] .. dst[at[k + 1]) (32-bit words, packed without gaps), dst being
// pinned host memory.
constexpr int GATHER_MAX = 10;
struct Gather {
    const uint32_t *src[GATHER_MAX];
    uint32_t at[GATHER_MAX + 1];
    int n;
};
hipError_t launch_gather(const Gather &g, uint32_t *dst, const Signal &sig, hipStream_t s);
// One replica's state as rows: double quat[n_bodies][4], then float pos[n_beads][3],
// rel[n_beads][3], centre[n_bodies][3], from the arrays at bead / body
struct StateRows {
    const float *p[6], *c[3];
    const uint32_t *quat;
    int n_beads, n_bodies;
};
hipError_t launch_state_rows(const StateRows &g, uint32_t *dst, const Signal &sig, hipStream_t s);
size_t adjoint_ff_size();
void adjoint_ff_fill(void *dst, const float *table, double lambda, double e0, double xi, double c_lj, double c_dh);

// full energy: tiles of 64 beads; column tiles of a workgroup (at most),
// workgroups a launch aims at
__host__ __device__ inline int full_tiles(int beads) { return (beads + 63) / 64; }
constexpr int FULL_PER_MAX = 32;
constexpr int FULL_WG = 2048;
constexpr int SPEC_MAX = 16;     // largest body (beads) a speculative window slot takes
static_assert(SPEC_MAX > 1, "a window slot's thread 1 forms its rotation");
constexpr int REMC_MAX_COOP = 8; // workgroups per replica where all replicas have as many
constexpr int REMC_MAX_MEMBERS = 32; // workgroups of one replica where they follow its system's cost
constexpr int REMC_SLOT_K = 64;  // partial sums per member and exchange (MC window slots, force-biased window values)
static_assert(REMC_MAX_MEMBERS <= 64 && REMC_MAX_MEMBERS % REMC_MAX_COOP == 0, "a lane per member, rows of whole polls");
static_assert(REMC_SLOT_K >= 64, "every lane of a polling wave reads a slot row of its own");

} // namespace remc
