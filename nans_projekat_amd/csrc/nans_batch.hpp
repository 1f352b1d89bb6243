// nans_batch.hpp -- the device-resident world batch shared by the step
// (nans_step.hip) and its adjoint (nans_adjoint.hip).
#pragma once

#include "nans_common.hpp"
#include "nans_world.hpp"

#include <vector>

struct nans_worlds;

namespace nans {

constexpr int PLAIN_MAX_BODIES = 16384;  // solver head[] lives in LDS (64 KiB)
constexpr int BATCH_MAX_BODIES = 512;    // bodies of one world kept in LDS by the batched path
constexpr int SCAN_THREADS = 1024;
constexpr int SOLVE_THREADS = 1024;
// The plain step's solve for worlds of at most PLAIN_SMALL_BODIES bodies: 256
// threads, with lists, bodies and as many contact terms as a CU's LDS holds.
constexpr int PLAIN_SMALL_THREADS = 256;
constexpr int PLAIN_SMALL_BODIES = 512;
constexpr size_t PLAIN_SMALL_LDS = 156 * 1024;
// head[], two counters, list[2 n], body planes
constexpr size_t plain_small_fixed_bytes(int n)
{
    return sizeof(int) * ((size_t)(3 + F_NLDS) * ((n + 3) & ~3) + 4);
}
constexpr int CULL_CHUNK = 4096;          // canonical pairs per block of the plain cull at most,
constexpr int CULL_BLOCKS = 512;          // fewer where this many blocks then suffice

enum : int {
    CNT_EPA_OVERFLOW = 0,
    CNT_CAND_OVERFLOW,
    CNT_CON_OVERFLOW,
    CNT_CANDIDATES,
    CNT_CONTACTS,
    CNT_GJK_FOUND,
    CNT_PAIR_TESTS,
    CNT_N
};

// A kept state: planes P V W A (the first F_SX fields), then force and torque.
constexpr int STATE_FIELDS = F_SX + 6;

// Arguments of k_batched_step (one persistent launch = nsteps steps of every world).
struct BatchArgs {
    float *planes;          // [F_NFIELDS][N]
    int64_t N;
    const int *offsets;     // [nw+1]
    const int *nboxes;      // [nw]
    const int *order;       // largest world first
    int nworlds;
    int nbig;               // order[0, nbig) run by a whole workgroup, the rest one per wave
    int nmax;               // LDS stride of a workgroup's world (>= largest world)
    int wrows;              // LDS stride of a wave's world (>= largest of order[nbig, nworlds))
    int lds_floats;         // floats of world LDS before the polytope LDS (a multiple of 4)
    int nsteps;
    int *queue;             // this launch's work counters: [0] workgroup worlds, [1] wave worlds
    int *queue_next;        // the next launch's counters, cleared by this one
    StepConsts k;
    const FloorDev *fl;
    const float *wfric, *wrest;  // per-world coefficients (may be null)
    int *cand;              // per-workgroup scratch, cap entries each
    ContactRec *rec;
    int *flag;
    int *qidx;
    SimplexRec *qsim;
    int cap;                // entries per workgroup
    int wcap;               // entries per wave in the wave phase (cap / waves)
    float *corners;         // per-workgroup box corners, corner_stride floats each
    int64_t corner_stride;
    float *state_out;       // [nsteps + 1][STATE_FIELDS][N]: slot k + 1 receives the state after step k (may be null)
    ContactRec *rec_out;    // recording (may be null): step k's contacts of world w at
    int64_t rec_stride;     // k * rec_stride + rec_off[w], their number at
    const int64_t *rec_off; // rec_count[k * rec_count_stride + w]
    int *rec_count;
    int rec_count_stride;
    unsigned long long *rec_pos;  // or, if set, the lists one after another as they come:
    int *rec_start;               // step k's of world w at rec_start[k * rec_count_stride + w],
    int rec_total;                // rec_total records in all (those beyond are only counted)
    const int *rec_cap;
    unsigned long long *cnt;
};

// The batched step's arguments; the warm-started instantiation adds, per world w,
// the previous and this step's contact lists (canonical pair index, three
// accumulators; ascending) at warm_off[w], warm_cap[w] entries each.  The cold
// step's arguments stay BatchArgs exactly.
template <bool WARM>
struct BatchArgsT : BatchArgs {};
template <>
struct BatchArgsT<true> : BatchArgs {
    int *warm_p0 = nullptr, *warm_p1 = nullptr;  // step k reads the lists of buffer (warm_flip + k) & 1
    float *warm_s0 = nullptr, *warm_s1 = nullptr;  // and writes the other's
    int *warm_n0 = nullptr, *warm_n1 = nullptr;
    int warm_flip = 0;
    const int64_t *warm_off = nullptr;
    const int *warm_cap = nullptr;
};

struct AdjointTape;  // nans_adjoint.hip
void adjoint_release(nans_worlds *W);

template <typename T>
inline int dmalloc(T **p, size_t n)
{
    *p = nullptr;
    if (n == 0) n = 1;
    NANS_HIP(hipMalloc((void **)p, n * sizeof(T)));
    return NANS_OK;
}

void wfree(void *p);
StepConsts step_consts(const nans_params &p, int orientation);
int warm_reset(nans_ctx *ctx);
int setup_floor(nans_ctx *ctx, hipStream_t s);
int check_overflow(nans_ctx *ctx);
// Saves the state a stepping call starts from; step_finish checks the call for a
// capacity overflow and, if it overflowed, restores that state and the counters
// (and empties the warm-start lists) before returning NANS_ERR_CAPACITY.
int snapshot_take(nans_ctx *ctx, hipStream_t s);
int step_finish(nans_ctx *ctx);
// nsteps batched steps (warm-started if the context is)
int batched_run(nans_ctx *ctx, int nsteps, int block);
// threads per world of the batched step (the autotuner's choice or the default)
int batched_block(nans_ctx *ctx);
// Where a run of cold batched steps keeps every step's state and contact lists
// (BatchArgs' recording fields).
struct BatchRecord {
    float *state;
    ContactRec *rec;
    int64_t rec_stride;
    const int64_t *rec_off;
    int *rec_count;  // nworlds per step
    const int *rec_cap;
    // set: lists one after another instead, rec_total records of room
    unsigned long long *pos = nullptr;
    int *start = nullptr;  // nworlds per step
    int rec_total = 0;
};
int batched_run_recorded(nans_ctx *ctx, int nsteps, hipStream_t s, const BatchRecord &rec);

}  // namespace nans

struct nans_worlds {
    int nworlds = 0;
    int64_t N = 0;
    int nmax = 0;
    int64_t max_pairs = 0;
    std::vector<int> h_off, h_nb;
    std::vector<float> h_fric, h_rest;
    std::vector<float> quat_angles;  // nans_set_state's angles while their quaternions are not made
    float *planes = nullptr;
    float *verts = nullptr;
    float *brad = nullptr;
    int *offsets = nullptr;
    int *nboxes = nullptr;
    int *order = nullptr;
    float *wfric = nullptr;
    float *wrest = nullptr;
    nans::FloorDev *floor = nullptr;
    unsigned long long *cnt = nullptr;
    // plain scratch
    int cand_cap = 0;
    int *cand = nullptr;
    nans::ContactRec *rec = nullptr;
    int *flag = nullptr;
    nans::ContactRec *con = nullptr;
    int *done = nullptr;
    int *qidx = nullptr;
    nans::SimplexRec *qsim = nullptr;
    int *blk_counts = nullptr;
    int *blk_offsets = nullptr;
    int *ncand = nullptr;
    int max_blk = 0;
    // Further lanes of the plain step for batches of several worlds: world w runs on
    // lane w % lanes (lane 0 is the context's stream with the scratch above; a world
    // that takes the grid broadphase always runs on lane 0, the grid's only user).
    struct PlainLane {
        hipStream_t s = nullptr;
        hipEvent_t ev = nullptr;
        int *cand = nullptr;
        nans::ContactRec *rec = nullptr;
        int *flag = nullptr;
        nans::ContactRec *con = nullptr;
        int *done = nullptr;
        int *qidx = nullptr;
        nans::SimplexRec *qsim = nullptr;
        int *blk_counts = nullptr;
        int *blk_offsets = nullptr;
        int *ncand = nullptr;
        int *warm_cp = nullptr;
        float *warm_sums = nullptr;
    };
    std::vector<PlainLane> plain_lanes;  // lanes 1.. (lane 0 is not stored)
    hipEvent_t plain_ev0 = nullptr;
    // hierarchical-grid broadphase of the plain step (sized for the largest world)
    int bp_buckets = 0;          // power of two >= 2 * nmax
    long long *bp_cell = nullptr;  // [3][nmax] cell coordinates
    int *bp_hslot = nullptr;     // [3][nmax] bucket, slot in bucket, level
    int *bp_sorted = nullptr;    // [nmax] bodies grouped by bucket
    int *bp_bcnt = nullptr;      // [bp_buckets]
    int *bp_boff = nullptr;      // [bp_buckets]
    int *bp_counts = nullptr;    // [3 nmax] row counts
    int *bp_offsets = nullptr;   // [3 nmax]
    int *bp_tmp = nullptr;       // [cand_cap] unsorted rows
    int *bp_stash = nullptr;     // [2 nmax][32] first pairs of each row
    int *bp_ovf = nullptr;       // a row overflowed its stash
    // opt-in warm start of the plain and batched steps: two contact lists per world
    int warm_ready = 0, warm_flip = 0;
    std::vector<int64_t> h_warm_off;
    std::vector<int> h_warm_cap;
    int64_t *warm_offd = nullptr;           // [nworlds] h_warm_off on the device
    int *warm_capd = nullptr;               // [nworlds] h_warm_cap on the device
    int *warm_p[2] = {nullptr, nullptr};    // canonical pair indices
    float *warm_s[2] = {nullptr, nullptr};  // [3] accumulators per contact
    int *warm_n[2] = {nullptr, nullptr};    // [nworlds] list lengths
    int *warm_cp = nullptr;                 // [cand_cap] pair index per contact of the world being solved
    float *warm_sums = nullptr;             // [3 cand_cap] its accumulators
    void *bp_grid = nullptr;     // nans::BpGrid
    // batched scratch
    int b_grid = 0;
    int b_cap = 0;
    int *b_cand = nullptr;
    nans::ContactRec *b_rec = nullptr;
    int *b_flag = nullptr;
    int *b_qidx = nullptr;
    nans::SimplexRec *b_qsim = nullptr;
    float *b_corners = nullptr;    // box corners of the batched step's worlds in flight
    int64_t b_corner_floats = 0;   // its size
    int *queue = nullptr;
    int queue_len = 0;
    int queue_flip = 0;  // which half of queue[] the next batched launch uses
    // recording
    int record = 0;
    nans::ContactRec *rec_buf = nullptr;
    int64_t *rec_off = nullptr;
    int *rec_count = nullptr;
    int *rec_cap = nullptr;
    std::vector<int64_t> h_rec_off;
    std::vector<int> h_rec_cap;
    hipEvent_t ev_t0 = nullptr, ev_t1 = nullptr;
    // shape of the last batched launch
    int shape_block = 0, shape_grid = 0, shape_lds = 0;
    int shape_wave = -1;     // worlds of at most this many bodies ran one per wave
    int shape_nwave = 0;     // and there were this many of them
    int timed_steps = 0;
    float timed_ms = 0.0f;
    int tuned_block = 0;   // autotuner's choice of threads per world (0: not tuned)
    int tuned_wave = -1;   // autotuner's or caller's wave-world bound in bodies (-1: default)
    nans::AdjointTape *adj = nullptr;  // checkpoints and scratch of the differentiable rollout
    float *snap = nullptr;             // state at the start of a stepping call (snapshot_take)
};
