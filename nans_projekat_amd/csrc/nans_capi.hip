// nans_capi.hip -- context management and the narrowphase entry point of the
// C ABI declared in include/nans_gpu.h.
#include "nans_common.hpp"

#include <algorithm>
#include <mutex>
#include <new>

namespace nans {

static thread_local char g_error[1024];

void set_error(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_error, sizeof(g_error), fmt, ap);
    va_end(ap);
}

struct NarrowIn {
    const int32_t *type;
    const float *pos, *quat, *half;
};

struct NarrowOutDev {
    int32_t *gjk, *contact, *status;
    float *normal, *pa, *pb;
    double *depth;
};

__device__ inline Shape load_shape(const NarrowIn &s, int64_t i, int64_t n)
{
    Shape sh;
    sh.vm = nullptr;
    sh.kind = s.type[i];
    sh.c = mk3(s.pos[i], s.pos[n + i], s.pos[2 * n + i]);
    V3 h = mk3(s.half[i], s.half[n + i], s.half[2 * n + i]);
    sh.r = h.x;
    if (sh.kind == SHAPE_BOX) {
        box_from_quat(sh.c, s.quat[i], s.quat[n + i], s.quat[2 * n + i], s.quat[3 * n + i], h, sh.v);
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) sh.v[k] = mk3(0.0f, 0.0f, 0.0f);
    }
    return sh;
}

__device__ inline void write_pair(const NarrowOutDev &o, int64_t i, int64_t n, int g, int status, V3 nrm, V3 pa,
                                  V3 pb, double depth)
{
    if (o.gjk) o.gjk[i] = g;
    if (o.contact) o.contact[i] = status == EPA_CONTACT ? 1 : 0;
    if (o.status) o.status[i] = status;
    if (o.normal) { o.normal[i] = nrm.x; o.normal[n + i] = nrm.y; o.normal[2 * n + i] = nrm.z; }
    if (o.pa) { o.pa[i] = pa.x; o.pa[n + i] = pa.y; o.pa[2 * n + i] = pa.z; }
    if (o.pb) { o.pb[i] = pb.x; o.pb[n + i] = pb.y; o.pb[2 * n + i] = pb.z; }
    if (o.depth) o.depth[i] = depth;
}

// Candidates of one wave: pairs [first, first + count) of its group's (pair()).
struct PairSrc {
    NarrowIn a, b;
    int64_t first, n;
    int groups, group, shift;
    NarrowOutDev o;
    unsigned long long *overflow;
    SimplexRec *simplex;
    __device__ SimplexRec &sim(int c) const { return simplex[c]; }
    __device__ int key(int c) const { return c; }
    // shares of 2^shift pairs go to the groups in turn
    __device__ int64_t pair(int c) const
    {
        const int64_t u = first + c, s = u >> shift;
        return ((s * groups + group) << shift) + (u - (s << shift));
    }
    __device__ void shapes(int key, Shape &A, Shape &B) const
    {
        const int64_t i = pair(key);
        A = load_shape(a, i, n);
        B = load_shape(b, i, n);
    }
    __device__ void gjk_result(int c, int g) const
    {
        const V3 z = mk3(0.0f, 0.0f, 0.0f);
        write_pair(o, pair(c), n, g, EPA_NONE, z, z, z, 0.0);
    }
    __device__ void epa_result(int c, int key, const EpaResult &r) const
    {
        write_pair(o, pair(c), n, GJK_FOUND, r.status, r.n, r.pa, r.pb, r.depth);
        if (r.status == EPA_OVERFLOW) atomicAdd(overflow, 1ull);
    }
};

// The narrowphase entry point: every wave takes shares of the pairs on its own
// (narrow_wave), so a small call is spread over the whole chip and no wave waits
// for the slowest pair of its workgroup.  With 256 pairs per workgroup, 777 random
// pairs ran on four workgroups as a chain of EPA passes (716 us a call, now 123),
// 30011 on 117 of the chip's 256 CUs (859 us, now 306); 1M pairs 4.62 -> 3.68 ms.
// A share is a power of two: a quarter of a wave's part of the call, down to one
// pair, and at most 32, so that the last ones end together (1M pairs at 16, 32, 64:
// 4.10, 3.90, 3.96 ms; 200k in the islands mode 1.19, 1.24, 1.36 ms).  Three waves per
// SIMD (168 VGPRs; two take 5.37 ms where three take 4.82).
constexpr int NP_SHARE = 32;
constexpr int NP_WAVES_PER_CU = 12;
// The shares go in turn to as many groups of workgroups, each of which hands out its
// own from a counter in its own 128-byte line; a wave's first share is its place in
// the group, without a claim.  One counter for all serialised the claims at some 15 ns
// each, and a call whose pairs mostly miss is nothing but claims: pairs that all miss,
// 30011 / 200k / 1M a call, 249 / 219 / 445 us, now 59 / 47 / 69 (8, 16, 32, 64 groups
// alike within 5 %).
constexpr int NP_GROUPS = 32;
constexpr int NP_CNT_STRIDE = 16;
constexpr int NP_CNT_WORDS = NP_CNT_STRIDE * NP_GROUPS;
constexpr int NP_CNT_OVERFLOW = 1;  // the word of the overflow count, beside the first counter
// A wave that has seen this many pairs in a row miss takes twice as many with its next
// claim, up to 64, until a pair hits: one share fills few lanes of GJK, and only hits
// make a share long (all miss, 200k / 1M: 60 / 101 -> 47 / 69 us; at 32 in a row 52 / 69;
// at 8, 60000 pairs with 1 % overlaps take 154 us instead of 132).
constexpr int NP_RUN = 16;

// ISL: the FP64-islands mode (grouped EPA tiers with a binary64 final face).
template <bool ISL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NP_WAVES_PER_CU / 4))) void k_narrowphase(
    int64_t n, int shift, NarrowIn a, NarrowIn b, NarrowParams p, NarrowOutDev o, unsigned long long *cnt, int *list,
    SimplexRec *sim)
{
    __shared__ EpaLds lds[4];
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int groups = min(NP_GROUPS, (int)gridDim.x);
    const int g = (int)blockIdx.x % groups;
    const int waves = 4 * (((int)gridDim.x - g + groups - 1) / groups);  // of this group
    // the group's pairs, and how many the groups before it have
    const int64_t cycle = (int64_t)groups << shift, q = n / cycle, r = n - q * cycle;
    const int64_t mine = (q << shift) + min((int64_t)1 << shift, max((int64_t)0, r - ((int64_t)g << shift)));
    const int64_t before = (q << shift) * g + min(r, (int64_t)g << shift);
    const int64_t started = (int64_t)waves << shift;
    int take = 1 << shift, run = 0;
    int64_t first = (int64_t)(4 * ((int)blockIdx.x / groups) + wv) << shift;  // a wave's first share is its own
    while (first < mine) {
        const int count = (int)min((int64_t)take, mine - first);
        PairSrc src{a, b, first, n, groups, g, shift, o, &cnt[NP_CNT_OVERFLOW], sim + before + first};
        run = narrow_wave<ISL>(src, count, p, lds[wv], list + before + first) ? 0 : run + count;
        if (started >= mine) break;  // the first shares were all
        take = run >= NP_RUN ? min(64, 2 * take) : 1 << shift;
        unsigned long long c = 0;
        wave_sync();  // the wave meets on both sides of the claim
        if (lane_id() == 0) c = atomicAdd(&cnt[NP_CNT_STRIDE * g], (unsigned long long)take);
        wave_sync();
        first = started + (int64_t)(((unsigned long long)__builtin_amdgcn_readfirstlane((int)(c >> 32)) << 32) |
                                    (unsigned)__builtin_amdgcn_readfirstlane((int)c));
    }
}

__global__ void k_fill_u64(unsigned long long *p, int n, unsigned long long v)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Scratch of nans_narrowphase_noalloc, one copy per device for the life of the
// process: k_narrowphase's counters, then its hit list -- a candidate index and a GJK
// simplex per pair -- for up to NANS_NARROWPHASE_NOALLOC_MAX_PAIRS pairs (27 MiB in
// all).
constexpr size_t NA_CNT_BYTES = (sizeof(unsigned long long) * NP_CNT_WORDS + 255) / 256 * 256;
constexpr size_t NA_QIDX_BYTES = sizeof(int) * (size_t)NANS_NARROWPHASE_NOALLOC_MAX_PAIRS;
constexpr size_t NA_QSIM_BYTES = sizeof(SimplexRec) * (size_t)NANS_NARROWPHASE_NOALLOC_MAX_PAIRS;
constexpr size_t NA_BYTES = NA_CNT_BYTES + NA_QIDX_BYTES + NA_QSIM_BYTES;
static_assert(NA_QIDX_BYTES % 256 == 0, "the simplex records start 256-byte aligned");
static __device__ __align__(256) unsigned char scratch[NA_BYTES];

// Device address of each device's copy of scratch[], looked up once per device
// (with that device current) by nans_create.  The name scratch is a host-side
// stand-in in host code; only these addresses are passed to kernels.
constexpr int NA_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_dev[NA_MAX_DEVICES];

static int noalloc_scratch_init(int device, void **out)
{
    NANS_REQUIRE(device >= 0 && device < NA_MAX_DEVICES, NANS_ERR_INVALID, "device %d beyond %d", device,
                 NA_MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[device]) {
        void *ptr = nullptr;
        NANS_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        NANS_REQUIRE(ptr, NANS_ERR_HIP, "hipGetSymbolAddress returned no address for the scratch array");
        g_scratch_dev[device] = ptr;
    }
    *out = g_scratch_dev[device];
    return NANS_OK;
}

}  // namespace nans

using namespace nans;

extern "C" {

const char *nans_last_error(void) { return g_error; }

void nans_default_params(nans_params *p)
{
    if (!p) return;
    memset(p, 0, sizeof(*p));
    p->solver_iterations = 70;
    p->beta = 0.3f;
    p->restitution = (float)0.1;
    p->friction = 0.1f;
    p->damping = 1.5f;
    p->gravity = 9.81f;
    p->dt = 1.0f / 60.0f;
    p->max_gjk_iterations = 64;
    p->max_epa_iterations = 64;
    p->epa_tolerance = 0.001f;
    p->fp64_islands = 0;
    p->floor_pos[0] = 1.2f;
    p->floor_pos[1] = -0.5f;
    p->floor_pos[2] = 1.0f;
    p->floor_scale[0] = 100.0f;
    p->floor_scale[1] = 1.0f;
    p->floor_scale[2] = 100.0f;
    p->floor_mass = 100000.0f;
    p->floor_moi = (p->floor_mass / 12.0f) * (2.0f * 100.0f * 100.0f);
    p->device = 0;
}

static int check_params(const nans_params *p)
{
    NANS_REQUIRE(p, NANS_ERR_INVALID, "params is NULL");
    NANS_REQUIRE(p->solver_iterations >= 0 && p->solver_iterations <= 100000, NANS_ERR_INVALID,
                 "solver_iterations out of range");
    NANS_REQUIRE(p->max_gjk_iterations >= 0 && p->max_gjk_iterations <= 100000, NANS_ERR_INVALID,
                 "max_gjk_iterations out of range");
    NANS_REQUIRE(p->max_epa_iterations >= 0 && p->max_epa_iterations <= 100000, NANS_ERR_INVALID,
                 "max_epa_iterations out of range");
    NANS_REQUIRE(p->fp64_islands == 0 || p->fp64_islands == 1, NANS_ERR_INVALID, "fp64_islands must be 0 or 1");
    NANS_REQUIRE(p->floor_mass > 0.0f && p->floor_moi > 0.0f, NANS_ERR_INVALID, "floor mass/moi must be positive");
    return NANS_OK;
}

int nans_create(nans_ctx **out, const nans_params *p)
{
    NANS_REQUIRE(out, NANS_ERR_INVALID, "out is NULL");
    *out = nullptr;
    nans_params q;
    if (p) q = *p;
    else nans_default_params(&q);
    int rc = check_params(&q);
    if (rc) return rc;
    int ndev = 0;
    NANS_HIP(hipGetDeviceCount(&ndev));
    NANS_REQUIRE(q.device >= 0 && q.device < ndev, NANS_ERR_INVALID, "device %d not present (%d devices)", q.device, ndev);
    NANS_HIP(hipSetDevice(q.device));
    nans_ctx *c = new (std::nothrow) nans_ctx();
    NANS_REQUIRE(c, NANS_ERR_CAPACITY, "out of host memory");
    c->p = q;
    c->stream = nullptr;
    c->worlds = nullptr;
    c->np_cap = 0;
    c->np_qidx = nullptr;
    c->np_qsim = nullptr;
    c->na_scratch = nullptr;
    c->tape_bytes = ADJ_TAPE_BYTES;
    rc = noalloc_scratch_init(q.device, &c->na_scratch);
    if (rc) {
        delete c;
        return rc;
    }
    hipError_t e = hipMalloc((void **)&c->d_counters, NP_CNT_WORDS * sizeof(unsigned long long));
    if (e != hipSuccess) {
        delete c;
        set_error("hipMalloc: %s", hipGetErrorString(e));
        return NANS_ERR_HIP;
    }
    *out = c;
    return NANS_OK;
}

int nans_destroy(nans_ctx *ctx)
{
    if (!ctx) return NANS_OK;
    NANS_HIP(hipSetDevice(ctx->p.device));
    NANS_HIP(hipDeviceSynchronize());
    worlds_release(ctx);
    hipFree(ctx->d_counters);
    if (ctx->np_qidx) hipFree(ctx->np_qidx);
    if (ctx->np_qsim) hipFree(ctx->np_qsim);
    delete ctx;
    return NANS_OK;
}

int nans_set_params(nans_ctx *ctx, const nans_params *p)
{
    NANS_REQUIRE(ctx, NANS_ERR_INVALID, "ctx is NULL");
    int rc = check_params(p);
    if (rc) return rc;
    NANS_REQUIRE(p->device == ctx->p.device, NANS_ERR_INVALID, "the device of a context cannot change");
    ctx->p = *p;
    return NANS_OK;
}

int nans_set_stream(nans_ctx *ctx, void *hip_stream)
{
    NANS_REQUIRE(ctx, NANS_ERR_INVALID, "ctx is NULL");
    ctx->stream = (hipStream_t)hip_stream;
    return NANS_OK;
}

int nans_set_broadphase(nans_ctx *ctx, int32_t mode)
{
    NANS_REQUIRE(ctx, NANS_ERR_INVALID, "ctx is NULL");
    NANS_REQUIRE(mode == NANS_BROADPHASE_AUTO || mode == NANS_BROADPHASE_ALL_PAIRS || mode == NANS_BROADPHASE_GRID,
                 NANS_ERR_INVALID, "broadphase mode %d is not one of NANS_BROADPHASE_*", (int)mode);
    ctx->broadphase = mode;
    return NANS_OK;
}

}  // extern "C"

namespace nans {

static int narrow_check(const nans_ctx *ctx, int64_t n, const nans_shapes_soa *a, const nans_shapes_soa *b,
                        const nans_narrow_out *out)
{
    NANS_REQUIRE(ctx, NANS_ERR_INVALID, "ctx is NULL");
    NANS_REQUIRE(n >= 0, NANS_ERR_INVALID, "n < 0");
    NANS_REQUIRE(n <= (int64_t)1 << 31, NANS_ERR_CAPACITY, "n = %lld exceeds 2^31 pairs", (long long)n);
    NANS_REQUIRE(a && b && out, NANS_ERR_INVALID, "shape or output descriptor is NULL");
    NANS_REQUIRE(n == 0 || (a->type && a->pos && a->quat && a->half && b->type && b->pos && b->quat && b->half),
                 NANS_ERR_INVALID, "a shape array is NULL");
    return NANS_OK;
}

// k_narrowphase over n pairs on the context's stream with the given overflow
// counter and EPA queue (n entries), then the counter to the host.
static int narrow_launch(nans_ctx *ctx, int64_t n, const nans_shapes_soa *a, const nans_shapes_soa *b,
                         const nans_narrow_out *out, unsigned long long *cnt, int *qidx, SimplexRec *qsim,
                         int64_t *n_overflow)
{
    hipStream_t s = ctx->stream;
    k_fill_u64<<<(NP_CNT_WORDS + 255) / 256, 256, 0, s>>>(cnt, NP_CNT_WORDS, 0ull);
    NANS_HIP(hipGetLastError());
    if (n > 0) {
        NarrowIn ia{a->type, a->pos, a->quat, a->half};
        NarrowIn ib{b->type, b->pos, b->quat, b->half};
        NarrowOutDev o{out->gjk, out->contact, out->status, out->normal, out->point_a, out->point_b, out->depth};
        int cus = 0;
        NANS_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->p.device));
        const int64_t waves = NP_WAVES_PER_CU * (int64_t)cus;
        int shift = 0;  // of a share
        while (2 << shift <= NP_SHARE && (2 << shift) * 4 * waves <= n) ++shift;
        const int64_t shares = (n + (1 << shift) - 1) >> shift;
        unsigned grid = (unsigned)std::min<int64_t>((shares + 3) / 4, waves / 4);
        // as many workgroups to every group: 200 pairs on 50 left some groups a claim short
        if (grid > NP_GROUPS) grid = (grid + NP_GROUPS - 1) / NP_GROUPS * NP_GROUPS;
        const NarrowParams np = narrow_params(ctx->p);
        if (ctx->p.fp64_islands)
            k_narrowphase<true><<<grid, 256, 0, s>>>(n, shift, ia, ib, np, o, cnt, qidx, qsim);
        else
            k_narrowphase<false><<<grid, 256, 0, s>>>(n, shift, ia, ib, np, o, cnt, qidx, qsim);
        NANS_HIP(hipGetLastError());
    }
    unsigned long long ov = 0;
    NANS_HIP(hipMemcpyAsync(&ov, cnt + NP_CNT_OVERFLOW, sizeof(ov), hipMemcpyDeviceToHost, s));
    NANS_HIP(hipStreamSynchronize(s));
    if (n_overflow) *n_overflow = (int64_t)ov;
    return NANS_OK;
}

}  // namespace nans

extern "C" {

int nans_narrowphase(nans_ctx *ctx, int64_t n, const nans_shapes_soa *a, const nans_shapes_soa *b,
                     const nans_narrow_out *out, int64_t *n_overflow)
{
    NANS_TRY(narrow_check(ctx, n, a, b, out));
    NANS_HIP(hipSetDevice(ctx->p.device));
    if (n > ctx->np_cap) {
        hipFree(ctx->np_qidx);
        hipFree(ctx->np_qsim);
        ctx->np_qidx = nullptr;
        ctx->np_qsim = nullptr;
        ctx->np_cap = 0;
        NANS_HIP(hipMalloc((void **)&ctx->np_qidx, sizeof(int) * (size_t)n));
        NANS_HIP(hipMalloc((void **)&ctx->np_qsim, sizeof(SimplexRec) * (size_t)n));
        ctx->np_cap = n;
    }
    return narrow_launch(ctx, n, a, b, out, ctx->d_counters, ctx->np_qidx, (SimplexRec *)ctx->np_qsim, n_overflow);
}

int nans_narrowphase_noalloc(nans_ctx *ctx, int64_t n, const nans_shapes_soa *a, const nans_shapes_soa *b,
                             const nans_narrow_out *out, int64_t *n_overflow)
{
    NANS_TRY(narrow_check(ctx, n, a, b, out));
    NANS_REQUIRE(n <= NANS_NARROWPHASE_NOALLOC_MAX_PAIRS, NANS_ERR_CAPACITY,
                 "n = %lld exceeds the %d pairs of the no-allocation scratch; split the call",
                 (long long)n, NANS_NARROWPHASE_NOALLOC_MAX_PAIRS);
    NANS_REQUIRE(ctx->na_scratch, NANS_ERR_STATE, "the context has no scratch address");
    NANS_HIP(hipSetDevice(ctx->p.device));
    unsigned char *base = static_cast<unsigned char *>(ctx->na_scratch);
    return narrow_launch(ctx, n, a, b, out, reinterpret_cast<unsigned long long *>(base),
                         reinterpret_cast<int *>(base + NA_CNT_BYTES),
                         reinterpret_cast<SimplexRec *>(base + NA_CNT_BYTES + NA_QIDX_BYTES), n_overflow);
}

}  // extern "C"
