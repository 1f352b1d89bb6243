// nans_adjoint.hip -- differentiable rollout of the batched step: forward with
// checkpoints, and the hand-written adjoint (nans_adjoint.hpp) run backwards
// step by step.
//
// nans_rollout keeps every step's state (P, V, W, angles, force, torque) and ordered
// contact list where memory allows (the dense tape), else the state every
// checkpoint_every steps.  nans_adjoint runs k_adjoint_steps over the tape, or walks
// the checkpoint segments from the last one: it restores the segment's checkpoint,
// recomputes the segment's steps with the batched step kernel (bit-identical to the
// rollout) while keeping each step's state and contacts, then runs k_adjoint_steps
// over the segment's steps in reverse, one world per workgroup: it replays a step's RK4 and SolveConstraints from the
// kept state and contact list (the same routines as the step, so the velocities
// after the solve equal the next kept state's, which is checked), recording the
// velocities each contact read and its dependency round, then propagates the
// adjoint back through IntegrateVelocities, the contacts in reverse round order
// (contacts of one round touch disjoint bodies), and RK4.  Per-body mass and
// moment-of-inertia adjoints accumulate in place; per-world friction and
// restitution adjoints are summed over the contacts in a fixed order, so a run
// is deterministic and independent of checkpoint_every.
#include "nans_adjoint.hpp"
#include "nans_batch.hpp"

#include <algorithm>
#include <climits>
#include <vector>

namespace nans {

// World-steps with more contacts than are kept; whose replay differs from the kept state;
// whose kept state and replay are both not a number.  Of the last two the first one, as the
// complement of step << 32 | world (a maximum, so that zero means none).
enum : int {
    ADJ_CNT_OVERFLOW = 0,
    ADJ_CNT_REPLAY,
    ADJ_CNT_NAN,
    ADJ_FIRST_REPLAY,
    ADJ_FIRST_NAN,
    ADJ_CNT_N
};

struct AdjArgs {
    const float *state;   // [nsteps + 1][STATE_FIELDS][N]: slot k the state before step k
    int nsteps;
    int step0;            // number of step 0 in the rollout
    const float *planes;  // the batch's planes (scale, mass, moi)
    int64_t N;
    const int *offsets;
    int nmax;
    StepConsts k;
    const FloorDev *fl;
    const float *wfric, *wrest;
    const ContactRec *rec;  // step k's contacts of world w at k * rec_stride + rec_off[w]
    int64_t rec_stride;     // (or, if rec_start is set, at rec_start[k][w])
    const int64_t *rec_off;
    const int *rec_start;   // [nsteps][nworlds] or null
    const int *rec_count;   // [nsteps][nworlds]
    const int *rec_cap;
    AdjTape *tape;          // per contact, one step, at rec_off[w]
    float *adj;             // [12][N]: adjoints of P V W A, in: after the steps, out: before
    float *g_mass, *g_moi;  // [N], accumulated
    float *g_fric, *g_rest; // [nworlds], accumulated
    unsigned long long *cnt;
};

// LDS planes: bodies (F_NLDS fields), adjoints gP gV gW (9) and gm gI (2) of the
// step, the sums of gm and gI over the steps (2), head[] of the dependency rounds.
constexpr int ADJ_LDS_PLANES = 13;
// Per thread besides: its first contact's position-only terms and the velocities the
// contact read (an odd number of words each: no bank conflicts across the lanes).
struct AdjOwn {
    ContactTerms t;
    ContactVel v;
    int pad;
};
constexpr int ADJ_OWN_FLOATS = (int)(sizeof(AdjOwn) / sizeof(float));
static_assert(ADJ_OWN_FLOATS % 2 == 1, "odd stride in words");

// A thread's iteration history in LDS: word it of lane-interleaved sums, then codes.
template <int BLOCK>
struct LdsHistory {
    float *s;
    __device__ void put(int it, float sum, int code)
    {
        s[2 * it * BLOCK] = sum;
        s[(2 * it + 1) * BLOCK] = __int_as_float(code);
    }
    __device__ float sum(int it) const { return s[2 * it * BLOCK]; }
    __device__ int code(int it) const { return __float_as_int(s[(2 * it + 1) * BLOCK]); }
};

__device__ inline ContactVel contact_velocities(const Planes &B, int sa, int sb)
{
    const V3 zero = mk3(0.0f, 0.0f, 0.0f);
    ContactVel v;
    v.V1 = B.get3(F_VX, sa);
    v.W1 = B.get3(F_WX, sa);
    v.two_sided = sb >= 0;
    v.V2 = sb >= 0 ? B.get3(F_VX, sb) : zero;
    v.W2 = sb >= 0 ? B.get3(F_WX, sb) : zero;
    return v;
}

// Adjoint planes of the step around one contact's reverse.
template <class History>
__device__ inline void contact_reverse(const Planes &Gd, int sa, int sb, const ContactTerms &t,
                                       const ContactReplay &p, const StepConsts &k, float Cf, float Cr,
                                       const History &h, float &gcf, float &gcr)
{
    ContactGrad g;
    g.gV1 = Gd.get3(3, sa);
    g.gW1 = Gd.get3(6, sa);
    g.gV2 = g.gW2 = mk3(0.0f, 0.0f, 0.0f);
    if (sb >= 0) {
        g.gV2 = Gd.get3(3, sb);
        g.gW2 = Gd.get3(6, sb);
    }
    constraint_adjoint(t, p, sb >= 0, k, Cf, Cr, h, g);
    Gd.set3(3, sa, g.gV1);
    Gd.set3(6, sa, g.gW1);
    Gd.set3(0, sa, add(Gd.get3(0, sa), g.gPA));
    Gd.at(9, sa) += g.gmA;
    Gd.at(10, sa) += g.gIA;
    if (sb >= 0) {
        Gd.set3(3, sb, g.gV2);
        Gd.set3(6, sb, g.gW2);
        Gd.set3(0, sb, add(Gd.get3(0, sb), g.gPB));
        Gd.at(9, sb) += g.gmB;
        Gd.at(10, sb) += g.gIB;
    }
    gcf = g.gCf;
    gcr = g.gCr;
}

// Steps nsteps - 1 .. 0 of one world per workgroup, its adjoints kept in LDS from
// step to step.  A step's cost is its chain of dependency rounds, forward and back,
// so all that does not hang on the chain leaves it: a thread's first contact keeps
// its position-only terms in LDS and its place in registers, and once the forward rounds have told the
// velocities each contact read, its forward values and impulse iterations are
// replayed for all contacts at once, their history in LDS (HL; else, where that does
// not fit, every contact replays in its round through scratch).  A launch per step,
// each round holding its contacts' whole arithmetic, took 126 us a step of 1024 worlds
// of 16 bodies; rollout and gradient of 240 steps 68.3 -> 43 ms, 24 worlds of 9
// bodies, 50 steps 9.3 -> 6.2 ms.
template <int BLOCK, bool HL>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2))) void k_adjoint_steps(AdjArgs a)
{
    extern __shared__ float smem[];
    __shared__ float red[2][BLOCK];
    const int w = blockIdx.x, tid = threadIdx.x, nmax = a.nmax;
    const int b0 = a.offsets[w];
    const int n = a.offsets[w + 1] - b0;
    const FloorDev &fl = *a.fl;
    const Planes Lb{smem, nmax};
    float *ga = smem + F_NLDS * nmax;
    const Planes Gd{ga, nmax};  // 0..2 gP, 3..5 gV, 6..8 gW, 9 gm, 10 gI, 11 12 their sums
    unsigned *hk = (unsigned *)(ga + ADJ_LDS_PLANES * nmax);
    AdjOwn &mine = reinterpret_cast<AdjOwn *>(ga + (ADJ_LDS_PLANES + 1) * nmax)[tid];
    ContactTerms &t = mine.t;
    ContactVel &v = mine.v;
    LdsHistory<BLOCK> hist{ga + (ADJ_LDS_PLANES + 1) * nmax + ADJ_OWN_FLOATS * BLOCK + tid};
    const Planes G{const_cast<float *>(a.planes) + b0, (int)a.N};
    const Planes Ad{a.adj + b0, (int)a.N};
    AdjTape *tape = a.tape + a.rec_off[w];
    const float dt = a.k.dt;
    const float Cf = a.wfric ? a.wfric[w] : a.k.friction;
    const float Cr = a.wrest ? a.wrest[w] : a.k.restitution;

    for (int i = tid; i < n; i += BLOCK) {
#pragma unroll
        for (int f = F_SX; f < F_NLDS; ++f) Lb.at(f, i) = G.at(f, i);
#pragma unroll
        for (int f = 0; f < 9; ++f) Gd.at(f, i) = Ad.at(f, i);
        Gd.at(11, i) = a.g_mass[b0 + i];
        Gd.at(12, i) = a.g_moi[b0 + i];
    }
    float tot_f = a.g_fric[w], tot_r = a.g_rest[w];
    for (int step = a.nsteps - 1; step >= 0; --step) {
        const Planes S{const_cast<float *>(a.state) + (int64_t)step * STATE_FIELDS * a.N + b0, (int)a.N};
        const Planes Nx{S.base + (int64_t)STATE_FIELDS * a.N, (int)a.N};
        const int64_t kw = (int64_t)step * gridDim.x + w;
        const ContactRec *con = a.rec + (a.rec_start ? a.rec_start[kw] : step * a.rec_stride + a.rec_off[w]);
        const int ncon = a.rec_count[kw];
        if (ncon > a.rec_cap[w]) {  // uniform over the workgroup; the call then fails
            if (tid == 0) atomicAdd(&a.cnt[ADJ_CNT_OVERFLOW], 1ull);
            return;
        }
        // state at the start of the step, RK4, and the adjoint through IntegrateVelocities
        for (int i = tid; i < n; i += BLOCK) {
#pragma unroll
            for (int f = 0; f < F_SX; ++f) Lb.at(f, i) = S.at(f, i);
            integrate_forces_body(Lb, i, S.get3(12, i), S.get3(15, i), a.k);
            // P' = P + dt V, A' = A + dt W (V, W after the solve)
            Gd.set3(3, i, add(Gd.get3(3, i), mul(Gd.get3(0, i), dt)));
            Gd.set3(6, i, add(Gd.get3(6, i), mul(Ad.get3(9, i), dt)));
            Gd.at(9, i) = 0.0f;
            Gd.at(10, i) = 0.0f;
            hk[i] = 0u;
        }
        for (int c = tid + BLOCK; c < ncon; c += BLOCK) tape[c].round = -1;
        __syncthreads();
        // this thread's first contact
        const bool own = tid < ncon;
        int sa = 0, sb = -1, myround = -1;
        if (own) {
            const ContactRec rc = con[tid];
            sa = rc.slot_a;
            sb = rc.slot_b;
            contact_terms(Lb, rc, fl, a.k, t);
        }

        // forward SolveConstraints by dependency rounds (solve_team's keys), keeping
        // what each contact read
        int rounds = 0;
        unsigned key_round = 0;
        bool pend = own;
        int pending = ncon;
        while (pending > 0) {
            if (++key_round == 2048u) {
                for (int i = tid; i < n; i += BLOCK) hk[i] = 0u;
                __syncthreads();
                key_round = 1;
            }
            const unsigned rk = (key_round << 21) | 0x1FFFFFu;
            auto key = [rk](int c) { return rk - (unsigned)c; };
            if (pend) {
                atomicMax(&hk[sa], key(tid));
                if (sb >= 0) atomicMax(&hk[sb], key(tid));
            }
            for (int c = tid + BLOCK; c < ncon; c += BLOCK) {
                if (tape[c].round < 0) {
                    atomicMax(&hk[con[c].slot_a], key(c));
                    const int s2 = con[c].slot_b;
                    if (s2 >= 0) atomicMax(&hk[s2], key(c));
                }
            }
            __syncthreads();
            int left = 0;
            if (pend) {
                const unsigned kc = key(tid);
                if (hk[sa] == kc && (sb < 0 || hk[sb] == kc)) {
                    v = contact_velocities(Lb, sa, sb);
                    ContactRec r;
                    r.slot_a = sa;
                    r.slot_b = sb;
                    contact_apply(Lb, r, t, a.k, Cf, Cr);
                    myround = rounds;
                    pend = false;
                } else {
                    left = 1;
                }
            }
            for (int c = tid + BLOCK; c < ncon; c += BLOCK) {
                if (tape[c].round < 0) {
                    const int s1 = con[c].slot_a, s2 = con[c].slot_b;
                    if (hk[s1] == key(c) && (s2 < 0 || hk[s2] == key(c))) {
                        AdjTape &q = tape[c];
                        const ContactVel u = contact_velocities(Lb, s1, s2);
                        q.v1[0] = u.V1.x; q.v1[1] = u.V1.y; q.v1[2] = u.V1.z;
                        q.w1[0] = u.W1.x; q.w1[1] = u.W1.y; q.w1[2] = u.W1.z;
                        q.v2[0] = u.V2.x; q.v2[1] = u.V2.y; q.v2[2] = u.V2.z;
                        q.w2[0] = u.W2.x; q.w2[1] = u.W2.y; q.w2[2] = u.W2.z;
                        q.round = rounds;
                        ContactRec r = con[c];
                        constraint(Lb, r, fl, a.k, Cf, Cr);
                    } else {
                        left = 1;
                    }
                }
            }
            pending = __syncthreads_count(left);
            ++rounds;
        }

        // the replay must land on the kept next state
        int bad = 0;
        for (int i = tid; i < n; i += BLOCK) {
            const V3 vi = Lb.get3(F_VX, i), wi = Lb.get3(F_WX, i);
            const V3 p = add(Lb.get3(F_PX, i), mul(vi, dt));
            bad |= !veq(vi, Nx.get3(3, i)) || !veq(wi, Nx.get3(6, i)) || !veq(p, Nx.get3(0, i));
        }
        if (__syncthreads_count(bad)) {  // uniform; the call then fails
            // a NaN on both sides is no difference, though no comparison says so
            int differs = 0;
            for (int i = tid; i < n; i += BLOCK) {
                for (int f = F_PX; f < F_AX; ++f) {  // P, V, W
                    const float x = f < F_VX ? Lb.at(f, i) + Lb.at(F_VX + f, i) * dt : Lb.at(f, i), y = Nx.at(f, i);
                    differs |= !(x == y || (x != x && y != y));
                }
            }
            differs = __syncthreads_count(differs);
            const unsigned long long at = ((unsigned long long)(a.step0 + step) << 32) | (unsigned)w;
            if (tid == 0) {
                atomicAdd(&a.cnt[differs ? ADJ_CNT_REPLAY : ADJ_CNT_NAN], 1ull);
                atomicMax(&a.cnt[differs ? ADJ_FIRST_REPLAY : ADJ_FIRST_NAN], ~at);
            }
        }

        // reverse SolveConstraints, latest round first
        ContactReplay rp;
        float gcf = 0.0f, gcr = 0.0f;
        if (HL && own) contact_replay(t, v, a.k, Cf, Cr, rp, hist);
        for (int r = rounds - 1; r >= 0; --r) {
            if (HL && myround == r) contact_reverse(Gd, sa, sb, t, rp, a.k, Cf, Cr, hist, gcf, gcr);
            for (int c = HL ? tid + BLOCK : tid; c < ncon; c += BLOCK) {
                if ((!HL && c == tid ? myround : tape[c].round) != r) continue;
                LocalHistory h;
                ContactTerms tc;
                ContactReplay rc;
                const ContactRec rec = con[c];
                contact_terms(Lb, rec, fl, a.k, tc);
                ContactVel u = v;
                if (HL || c != tid) {
                    const AdjTape &q = tape[c];
                    u.V1 = mk3(q.v1[0], q.v1[1], q.v1[2]);
                    u.W1 = mk3(q.w1[0], q.w1[1], q.w1[2]);
                    u.V2 = mk3(q.v2[0], q.v2[1], q.v2[2]);
                    u.W2 = mk3(q.w2[0], q.w2[1], q.w2[2]);
                }
                contact_replay(tc, u, a.k, Cf, Cr, rc, h);
                float cf = 0.0f, cr = 0.0f;
                contact_reverse(Gd, rec.slot_a, rec.slot_b, tc, rc, a.k, Cf, Cr, h, cf, cr);
                if (!HL && c == tid) {
                    gcf = cf;
                    gcr = cr;
                } else {
                    tape[c].gcf = cf;
                    tape[c].gcr = cr;
                }
            }
            __syncthreads();
        }

        // reverse RK4
        for (int i = tid; i < n; i += BLOCK) {
            float gm = Gd.at(9, i), gI = Gd.at(10, i);
            const float m = Lb.at(F_MASS, i), I = Lb.at(F_MOI, i);
            Gd.set3(3, i, rk4_adjoint<false>(dt, S.get3(3, i), S.get3(12, i), m, a.k, Gd.get3(3, i), gm));
            Gd.set3(6, i, rk4_adjoint<true>(dt, S.get3(6, i), S.get3(15, i), I, a.k, Gd.get3(6, i), gI));
            Gd.at(11, i) += gm;
            Gd.at(12, i) += gI;
        }
        // friction / restitution adjoints of the world: strided partial sums, fixed tree
        float sf = 0.0f, sr = 0.0f;
        if (own) {
            sf += gcf;
            sr += gcr;
        }
        for (int c = tid + BLOCK; c < ncon; c += BLOCK) {
            sf += tape[c].gcf;
            sr += tape[c].gcr;
        }
        if constexpr (BLOCK > 64) {
            red[0][tid] = sf;
            red[1][tid] = sr;
            __syncthreads();
            for (int q = BLOCK / 2; q >= 64; q >>= 1) {
                if (tid < q) {
                    sf += red[0][tid + q];
                    sr += red[1][tid + q];
                    red[0][tid] = sf;
                    red[1][tid] = sr;
                }
                __syncthreads();
            }
        }
        for (int q = 32; q > 0; q >>= 1) {
            sf += __shfl_down(sf, q, 64);
            sr += __shfl_down(sr, q, 64);
        }
        tot_f += sf;  // thread 0's are the world's
        tot_r += sr;
    }
    for (int i = tid; i < n; i += BLOCK) {
#pragma unroll
        for (int f = 0; f < 9; ++f) Ad.at(f, i) = Gd.at(f, i);
        a.g_mass[b0 + i] = Gd.at(11, i);
        a.g_moi[b0 + i] = Gd.at(12, i);
    }
    if (tid == 0) {
        a.g_fric[w] = tot_f;
        a.g_rest[w] = tot_r;
    }
}

__global__ void k_fill_f32(float *p, int64_t n, float v)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_adj_zero_u64(unsigned long long *p, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

struct AdjointTape {
    int steps = 0, every = 0, ncp = 0;
    nans_params params;
    // states the rollout kept: every step's (dense: its contacts too), or every
    // checkpoint's
    bool dense = false;
    float *states = nullptr;    // [nslots][STATE_FIELDS][N]
    size_t nslots = 0;
    float *last = nullptr;      // [STATE_FIELDS][N] after the rollout
    ContactRec *rec = nullptr;  // [rec_total], as the worlds' steps came
    int rec_total = 0;
    size_t rec_need = 0;        // records the next tape has room for at least
    int *rec_start = nullptr, *rec_cnt = nullptr;  // [rec_steps][nworlds]
    int rec_steps = 0;
    unsigned long long *pos = nullptr;
    // backward scratch
    int seg_len = 0;
    float *seg = nullptr;       // [seg_len + 1][STATE_FIELDS][N]
    ContactRec *seg_rec = nullptr;  // [seg_len][total]
    int *seg_cnt = nullptr;     // [seg_len][nworlds]
    AdjTape *tape = nullptr;    // [total]
    int64_t total = 0;          // contact capacity summed over worlds
    int64_t *rec_off = nullptr;
    int *rec_cap = nullptr;
    float *adj = nullptr;       // [12][N]
    float *g_mass = nullptr, *g_moi = nullptr, *g_fric = nullptr, *g_rest = nullptr;
    unsigned long long *cnt = nullptr;
};

// The dense tape: a rollout keeps every step's state and contacts while that takes at
// most the context's tape_bytes and a quarter of the free memory, so that the adjoint need not
// step the batch a second time (1024 worlds of 16 bodies, 240 steps, 1.5 GB: rollout
// and gradient 43 -> 21.7 ms; 24 of 9, 50 steps: 6.2 -> 3.5).  Room for
// ADJ_TAPE_CONTACTS contacts per body and step; a rollout with more is differentiated
// through its checkpoints, as is one past the bounds, and the next one gets the room
// it needed.
constexpr int ADJ_TAPE_CONTACTS = 4;

static void free_dense(AdjointTape *T)
{
    for (void *p : {(void *)T->rec, (void *)T->rec_start, (void *)T->rec_cnt}) wfree(p);
    T->rec = nullptr;
    T->rec_start = T->rec_cnt = nullptr;
    T->rec_total = T->rec_steps = 0;
}

static int need_states(AdjointTape *T, size_t slots, size_t slot_floats)
{
    if (T->states && T->nslots == slots) return NANS_OK;
    wfree(T->states);
    T->states = nullptr;
    T->nslots = 0;
    NANS_TRY(dmalloc(&T->states, slots * slot_floats));
    T->nslots = slots;
    return NANS_OK;
}

static size_t tape_bytes(const nans_worlds *W, size_t slots, size_t recs, size_t steps)
{
    return sizeof(float) * STATE_FIELDS * W->N * slots + sizeof(ContactRec) * recs +
           2 * sizeof(int) * (size_t)W->nworlds * steps;
}

// Room for a dense tape of nsteps steps; false where it does not fit, with what is there
// left to the checkpoints.  A tape with room to spare is kept (rollouts of alternating
// lengths otherwise free and allocate it on every call: 1024 worlds of 16 bodies, 200 to
// 250 steps, 0.5 ms each), unless more than three quarters of it lie idle.
static bool dense_prepare(nans_worlds *W, AdjointTape *T, int nsteps, int64_t limit)
{
    const size_t slot = (size_t)STATE_FIELDS * W->N, lists = (size_t)W->nworlds * nsteps;
    const size_t recs = std::max((size_t)ADJ_TAPE_CONTACTS * W->N * nsteps, T->rec_need);
    if (recs == 0 || recs > INT_MAX) return false;
    const size_t bytes = tape_bytes(W, (size_t)nsteps + 1, recs, nsteps);
    const size_t held = tape_bytes(W, T->nslots, T->rec_total, T->rec_steps);
    if (bytes > (size_t)limit) return false;
    if (T->rec && (size_t)T->rec_total >= recs && T->rec_steps >= nsteps && T->nslots > (size_t)nsteps &&
        held <= (size_t)limit && held / 4 <= bytes)
        return true;
    size_t avail = 0, all = 0;
    if (hipMemGetInfo(&avail, &all) != hipSuccess || bytes > (avail + held) / 4) return false;
    free_dense(T);
    wfree(T->states);
    T->states = nullptr;
    T->nslots = 0;
    if (dmalloc(&T->rec, recs) || dmalloc(&T->rec_start, lists) || dmalloc(&T->rec_cnt, lists) ||
        need_states(T, (size_t)nsteps + 1, slot)) {
        (void)hipGetLastError();  // an allocation refused is no error of the rollout
        free_dense(T);
        return false;
    }
    T->rec_total = (int)recs;
    T->rec_steps = nsteps;
    return true;
}

static void free_segment(AdjointTape *T)
{
    for (void *p : {(void *)T->seg, (void *)T->seg_rec, (void *)T->seg_cnt}) wfree(p);
    T->seg = nullptr;
    T->seg_rec = nullptr;
    T->seg_cnt = nullptr;
    T->seg_len = 0;
}

void adjoint_release(nans_worlds *W)
{
    AdjointTape *T = W->adj;
    if (!T) return;
    free_segment(T);
    free_dense(T);
    for (void *p : {(void *)T->states, (void *)T->pos, (void *)T->last, (void *)T->tape, (void *)T->rec_off, (void *)T->rec_cap,
                    (void *)T->adj, (void *)T->g_mass, (void *)T->g_moi, (void *)T->g_fric, (void *)T->g_rest,
                    (void *)T->cnt})
        wfree(p);
    delete T;
    W->adj = nullptr;
}

// state planes <-> a kept slot [STATE_FIELDS][N]
static int save_state(nans_worlds *W, float *dst, hipStream_t s)
{
    const size_t N = (size_t)W->N;
    NANS_HIP(hipMemcpyAsync(dst, W->planes, sizeof(float) * 12 * N, hipMemcpyDeviceToDevice, s));
    NANS_HIP(hipMemcpyAsync(dst + 12 * N, W->planes + (size_t)F_FX * N, sizeof(float) * 6 * N,
                            hipMemcpyDeviceToDevice, s));
    return NANS_OK;
}

static int load_state(nans_worlds *W, const float *src, hipStream_t s)
{
    const size_t N = (size_t)W->N;
    NANS_HIP(hipMemcpyAsync(W->planes, src, sizeof(float) * 12 * N, hipMemcpyDeviceToDevice, s));
    NANS_HIP(hipMemcpyAsync(W->planes + (size_t)F_FX * N, src + 12 * N, sizeof(float) * 6 * N,
                            hipMemcpyDeviceToDevice, s));
    return NANS_OK;
}

// LDS of a workgroup's history at BLOCK threads.
static size_t history_bytes(const StepConsts &k, int block)
{
    return 2 * sizeof(float) * (size_t)std::max(adj_iterations(k), 0) * block;
}

// The history is kept in LDS while four 64-thread workgroups, or two of 256 threads,
// still share a CU's 160 KB.
constexpr size_t ADJ_LDS_64 = 40 * 1024, ADJ_LDS_256 = 80 * 1024;

template <int BLOCK, bool HL>
static int adjoint_launch(nans_ctx *ctx, AdjArgs &a, hipStream_t s)
{
    nans_worlds *W = ctx->worlds;
    const size_t lds = sizeof(float) * (size_t)((F_NLDS + ADJ_LDS_PLANES + 1) * W->nmax + ADJ_OWN_FLOATS * BLOCK) +
                       (HL ? history_bytes(a.k, BLOCK) : 0);
    if (!HL && lds + history_bytes(a.k, BLOCK) + 4096 <= (BLOCK == 64 ? ADJ_LDS_64 : ADJ_LDS_256))
        return adjoint_launch<BLOCK, true>(ctx, a, s);
    NANS_HIP(hipFuncSetAttribute((const void *)k_adjoint_steps<BLOCK, HL>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    k_adjoint_steps<BLOCK, HL><<<W->nworlds, BLOCK, lds, s>>>(a);
    NANS_HIP(hipGetLastError());
    return NANS_OK;
}

}  // namespace nans

using namespace nans;

extern "C" {

int nans_set_rollout_memory(nans_ctx *ctx, int64_t max_bytes)
{
    NANS_REQUIRE(ctx, NANS_ERR_INVALID, "ctx is NULL");
    ctx->tape_bytes = max_bytes < 0 ? ADJ_TAPE_BYTES : max_bytes;
    return NANS_OK;
}

int nans_rollout(nans_ctx *ctx, int32_t nsteps, int32_t checkpoint_every)
{
    NANS_REQUIRE(ctx && ctx->worlds, NANS_ERR_STATE, "no worlds uploaded");
    NANS_REQUIRE(ctx->orientation == NANS_ORIENT_EULER, NANS_ERR_STATE,
                 "the differentiable rollout follows the reference's Euler orientation only");
    NANS_REQUIRE(!ctx->warm, NANS_ERR_STATE, "the differentiable rollout does not warm-start contacts");
    NANS_REQUIRE(nsteps >= 1 && checkpoint_every >= 1, NANS_ERR_INVALID,
                 "nsteps and checkpoint_every must be >= 1 (got %d, %d)", nsteps, checkpoint_every);
    NANS_REQUIRE(ctx->p.solver_iterations <= ADJ_MAX_ITERS, NANS_ERR_INVALID,
                 "the adjoint records at most %d impulse iterations (solver_iterations = %d)", ADJ_MAX_ITERS,
                 ctx->p.solver_iterations);
    nans_worlds *W = ctx->worlds;
    NANS_REQUIRE(W->nmax <= BATCH_MAX_BODIES, NANS_ERR_CAPACITY,
                 "the differentiable rollout uses the batched step: at most %d bodies per world (largest: %d)",
                 BATCH_MAX_BODIES, W->nmax);
    NANS_HIP(hipSetDevice(ctx->p.device));
    hipStream_t s = ctx->stream;
    NANS_HIP(hipStreamSynchronize(s));
    if (!W->adj) W->adj = new AdjointTape();
    AdjointTape *T = W->adj;
    const size_t slot = (size_t)STATE_FIELDS * W->N;
    const int ncp = (nsteps + checkpoint_every - 1) / checkpoint_every;
    if (!T->last) NANS_TRY(dmalloc(&T->last, slot));
    if (!T->pos) NANS_TRY(dmalloc(&T->pos, 1));
    T->steps = 0;
    T->ncp = ncp;
    // (a batch that records its contacts keeps them in its own buffers)
    T->dense = !W->record && dense_prepare(W, T, nsteps, ctx->tape_bytes);
    if (!T->dense) {
        free_dense(T);
        NANS_TRY(need_states(T, ncp, slot));
    }
    NANS_TRY(snapshot_take(ctx, s));
    unsigned long long used = 0;
    if (T->dense) {
        k_adj_zero_u64<<<1, 64, 0, s>>>(T->pos, 1);
        NANS_TRY(save_state(W, T->states, s));
        NANS_TRY(setup_floor(ctx, s));
        BatchRecord r{T->states, T->rec, 0, nullptr, T->rec_cnt, nullptr, T->pos, T->rec_start, T->rec_total};
        NANS_TRY(batched_run_recorded(ctx, nsteps, s, r));
        NANS_HIP(hipMemcpyAsync(&used, T->pos, sizeof(used), hipMemcpyDeviceToHost, s));
        // nans_batched_timing answers after any batched launch; without an
        // nans_step_batched call before, as after the last checkpoint's launch
        if (W->timed_steps == 0) W->timed_steps = nsteps - (ncp - 1) * checkpoint_every;
    } else {
        const int block = batched_block(ctx);
        for (int j = 0; j < ncp; ++j) {
            const int len = std::min(checkpoint_every, nsteps - j * checkpoint_every);
            NANS_TRY(save_state(W, T->states + slot * j, s));
            NANS_TRY(batched_run(ctx, len, block));
        }
    }
    NANS_TRY(save_state(W, T->last, s));
    NANS_HIP(hipStreamSynchronize(s));
    NANS_TRY(step_finish(ctx));
    T->steps = nsteps;
    T->every = checkpoint_every;
    if (T->dense && used > (unsigned long long)T->rec_total) {  // the kept states still hold the checkpoints
        T->rec_need = (size_t)(used + used / 4);
        free_dense(T);
    }
    T->params = ctx->p;
    return NANS_OK;
}

int nans_adjoint(nans_ctx *ctx, const nans_adjoint_io *io)
{
    NANS_REQUIRE(ctx && ctx->worlds, NANS_ERR_STATE, "no worlds uploaded");
    NANS_REQUIRE(io, NANS_ERR_INVALID, "io is NULL");
    nans_worlds *W = ctx->worlds;
    AdjointTape *T = W->adj;
    NANS_REQUIRE(T && T->steps > 0, NANS_ERR_STATE, "no rollout to differentiate (call nans_rollout first)");
    NANS_REQUIRE(memcmp(&T->params, &ctx->p, sizeof(nans_params)) == 0, NANS_ERR_STATE,
                 "the parameters changed since nans_rollout");
    NANS_HIP(hipSetDevice(ctx->p.device));
    hipStream_t s = ctx->stream;
    NANS_HIP(hipStreamSynchronize(s));
    const int64_t N = W->N;
    const int nw = W->nworlds;
    const size_t slot = (size_t)STATE_FIELDS * N;
    // contact capacity per world and step, as the contact recording of the step
    if (!T->rec_off) {
        std::vector<int64_t> off(nw + 1, 0);
        std::vector<int> cap(nw);
        for (int w = 0; w < nw; ++w) {
            cap[w] = 16 * (W->h_off[w + 1] - W->h_off[w]) + 64;
            off[w + 1] = off[w] + cap[w];
        }
        T->total = off[nw];
        NANS_TRY(dmalloc(&T->rec_off, (size_t)nw));
        NANS_TRY(dmalloc(&T->rec_cap, (size_t)nw));
        NANS_HIP(hipMemcpy(T->rec_off, off.data(), sizeof(int64_t) * nw, hipMemcpyHostToDevice));
        NANS_HIP(hipMemcpy(T->rec_cap, cap.data(), sizeof(int) * nw, hipMemcpyHostToDevice));
        NANS_TRY(dmalloc(&T->tape, (size_t)T->total));
        NANS_TRY(dmalloc(&T->adj, (size_t)12 * N));
        NANS_TRY(dmalloc(&T->g_mass, (size_t)N));
        NANS_TRY(dmalloc(&T->g_moi, (size_t)N));
        NANS_TRY(dmalloc(&T->g_fric, (size_t)nw));
        NANS_TRY(dmalloc(&T->g_rest, (size_t)nw));
        NANS_TRY(dmalloc(&T->cnt, ADJ_CNT_N));
    }
    const bool whole = T->dense && T->rec;  // every step's contacts are on the tape
    const int L = std::min(T->every, T->steps);
    if (whole) {
        free_segment(T);
    } else if (T->seg_len != L) {
        free_segment(T);
        NANS_TRY(dmalloc(&T->seg, slot * (L + 1)));
        NANS_TRY(dmalloc(&T->seg_rec, (size_t)T->total * L));
        NANS_TRY(dmalloc(&T->seg_cnt, (size_t)nw * L));
        T->seg_len = L;
    }
    // initial adjoint: dL/d(final state)
    {
        std::vector<float> h((size_t)12 * N, 0.0f);
        const float *src[4] = {io->dl_pos, io->dl_vel, io->dl_angvel, io->dl_angles};
        for (int f = 0; f < 4; ++f)
            if (src[f]) std::copy(src[f], src[f] + 3 * N, h.begin() + (size_t)3 * f * N);
        NANS_HIP(hipMemcpy(T->adj, h.data(), sizeof(float) * h.size(), hipMemcpyHostToDevice));
    }
    auto fill = [&](float *p, int64_t n) { k_fill_f32<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(p, n, 0.0f); };
    fill(T->g_mass, N);
    fill(T->g_moi, N);
    fill(T->g_fric, nw);
    fill(T->g_rest, nw);
    k_adj_zero_u64<<<1, 64, 0, s>>>(T->cnt, ADJ_CNT_N);
    NANS_HIP(hipGetLastError());
    // the recomputation must not count in the step statistics
    unsigned long long saved[CNT_N];
    NANS_HIP(hipMemcpy(saved, W->cnt, sizeof(saved), hipMemcpyDeviceToHost));

    AdjArgs a;
    a.planes = W->planes;
    a.N = N;
    a.offsets = W->offsets;
    a.nmax = W->nmax;
    a.k = step_consts(ctx->p, NANS_ORIENT_EULER);
    a.fl = W->floor;
    a.wfric = W->wfric;
    a.wrest = W->wrest;
    a.state = whole ? T->states : T->seg;
    a.rec = whole ? T->rec : T->seg_rec;
    a.rec_stride = T->total;
    a.rec_off = T->rec_off;
    a.rec_start = whole ? T->rec_start : nullptr;
    a.rec_count = whole ? T->rec_cnt : T->seg_cnt;
    a.rec_cap = T->rec_cap;
    a.tape = T->tape;
    a.adj = T->adj;
    a.g_mass = T->g_mass;
    a.g_moi = T->g_moi;
    a.g_fric = T->g_fric;
    a.g_rest = T->g_rest;
    a.cnt = T->cnt;
    NANS_TRY(setup_floor(ctx, s));
    int rc = NANS_OK;
    auto reverse = [&](int first, int nsteps) {
        a.step0 = first;
        a.nsteps = nsteps;
        return W->nmax <= 64 ? adjoint_launch<64, false>(ctx, a, s) : adjoint_launch<256, false>(ctx, a, s);
    };
    if (whole) rc = reverse(0, T->steps);
    for (int j = whole ? -1 : T->ncp - 1; j >= 0 && rc == NANS_OK; --j) {
        const int t0 = j * T->every;
        const int len = std::min(T->every, T->steps - t0);
        rc = load_state(W, T->states + slot * (T->dense ? t0 : j), s);
        if (rc == NANS_OK) rc = save_state(W, T->seg, s);
        if (rc == NANS_OK)
            rc = batched_run_recorded(ctx, len, s,
                                      BatchRecord{T->seg, T->seg_rec, T->total, T->rec_off, T->seg_cnt, T->rec_cap});
        if (rc == NANS_OK) rc = reverse(t0, len);
    }
    // back to the state after the rollout, and the statistics before this call
    if (rc == NANS_OK) rc = load_state(W, T->last, s);
    NANS_HIP(hipStreamSynchronize(s));
    NANS_HIP(hipMemcpy(W->cnt, saved, sizeof(saved), hipMemcpyHostToDevice));
    if (rc != NANS_OK) return rc;
    unsigned long long c[ADJ_CNT_N];
    NANS_HIP(hipMemcpy(c, T->cnt, sizeof(c), hipMemcpyDeviceToHost));
    NANS_REQUIRE(c[ADJ_CNT_OVERFLOW] == 0, NANS_ERR_CAPACITY,
                 "a world had more contacts in one step than the adjoint keeps (16 per body + 64)");
    auto step_of = [&](int k) { return (int)(~c[k] >> 32); };
    auto world_of = [&](int k) { return (int)(unsigned)~c[k]; };
    NANS_REQUIRE(c[ADJ_CNT_REPLAY] == 0, NANS_ERR_STATE,
                 "the adjoint's replay of a step did not reproduce the rollout (%llu world-steps, the first: step %d "
                 "of world %d)",
                 c[ADJ_CNT_REPLAY], step_of(ADJ_FIRST_REPLAY), world_of(ADJ_FIRST_REPLAY));
    NANS_REQUIRE(c[ADJ_CNT_NAN] == 0, NANS_ERR_STATE,
                 "the rollout's state is not a number in %llu world-steps, from step %d of world %d on: no gradient",
                 c[ADJ_CNT_NAN], step_of(ADJ_FIRST_NAN), world_of(ADJ_FIRST_NAN));
    // outputs
    std::vector<float> h((size_t)12 * N);
    NANS_HIP(hipMemcpy(h.data(), T->adj, sizeof(float) * h.size(), hipMemcpyDeviceToHost));
    float *dst[4] = {io->dl_pos0, io->dl_vel0, io->dl_angvel0, io->dl_angles0};
    for (int f = 0; f < 4; ++f)
        if (dst[f]) std::copy(h.begin() + (size_t)3 * f * N, h.begin() + (size_t)3 * (f + 1) * N, dst[f]);
    if (io->dl_mass) NANS_HIP(hipMemcpy(io->dl_mass, T->g_mass, sizeof(float) * N, hipMemcpyDeviceToHost));
    if (io->dl_moi) NANS_HIP(hipMemcpy(io->dl_moi, T->g_moi, sizeof(float) * N, hipMemcpyDeviceToHost));
    if (io->dl_friction)
        NANS_HIP(hipMemcpy(io->dl_friction, T->g_fric, sizeof(float) * nw, hipMemcpyDeviceToHost));
    if (io->dl_restitution)
        NANS_HIP(hipMemcpy(io->dl_restitution, T->g_rest, sizeof(float) * nw, hipMemcpyDeviceToHost));
    return check_overflow(ctx);
}

}  // extern "C"
