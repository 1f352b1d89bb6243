// nans_epa.hpp -- EPA (ResolveCollision, code/nans.cpp:787-904) by one wavefront
// per pair, by groups of 16 or 32 lanes and by single lanes, and the narrowphase
// drivers (GJK per lane, then EPA) of a workgroup and of a wave.
//
// Layout of the whole wave's polytope:
//   vertices   registers: lane l holds vertex l (and lane l < 8 vertex 64 + l): its
//              P and its equality class (the first vertex with the same P, 255 if
//              P has a NaN: never equal); LDS keeps P, SupA, SupB for gathers;
//   faces      registers: lane l owns faces l, l+64, l+128 and keeps for each its
//              stored normal N, first vertex A, distance |dot(n, A)| and the packed
//              ids and classes of its three vertices;
//   edges      registers: horizon edge e lives in lane e;
//   shapes     registers: lanes 0-7 hold corner (lane) of box A, lanes 8-15 corner
//              (lane - 8) of box B; sphere centres and radii in every lane.
// One iteration of the reference's loop (code/nans.cpp:804-902):
//   closest face   the first face holding the minimum of the distances below face
//                  0's (the strict '<' scan from face 0, code/nans.cpp:807-822):
//                  DPP row minimum + ballots, the winner's data by readlane;
//   new support    along the winner's stored normal (code/nans.cpp:824-825): one
//                  corner dot product per lane and a DPP argmax over each group of
//                  8 lanes with the first-index tie rule of the strict '>' scan;
//   visibility     each lane tests its faces against the new point, ballots;
//   horizon        the visible faces' edges in face order with the exact
//                  reversed-edge cancellation of PushEdge (code/nans.cpp:232-266):
//                  when no edge key occurs twice, an edge survives iff its reverse
//                  is not among the pushed edges, which every lane checks at once;
//                  otherwise (or beyond 64 pushes) the pushes run one at a time;
//   compaction     survivors keep their order (std::vector::erase), new faces
//                  follow in edge order: one pass through an LDS staging area.
// A face's distance and flipped normal never change once it is made, so they are
// computed once, with the expression the reference re-evaluates every iteration.
#pragma once

#include "nans_narrow.hpp"

namespace nans {

constexpr int EPA_MAXV = 72;   // 4 + 65 vertices at most (one per iteration)
constexpr int EPA_MAXF = 192;  // alive faces: a closed triangulation of V <= 69 points has 2V-4 <= 134
constexpr int EPA_FSLOTS = EPA_MAXF / 64;
constexpr int CLS_NAN = 255;

struct EpaLds {
    float vp[EPA_MAXV][3];
    float va[EPA_MAXV][3];
    float vb[EPA_MAXV][3];
    float sfn[EPA_MAXF][3];  // compaction staging: stored normal
    float sfd[EPA_MAXF];     //                     distance
    int sfid[EPA_MAXF];      //                     a | b << 8 | c << 16
    int sfcl[EPA_MAXF];      //                     classes of a, b, c
    int ekey[128];           // horizon: pushed edges' classes (0..63), survivors (64..127)
    int eids[128];           //          and vertex ids, a | b << 8
};

struct EpaResult {
    int status;  // EPA_*
    V3 pa, pb, n;
    double depth;
    int iters, max_faces, nverts;
};

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63); }
__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

// The threads that run one world's step or one narrowphase: the whole workgroup,
// or one wave of it.  whole must be uniform over the workgroup (made from
// constants or readfirstlane values), so that sync()'s barrier is reached by
// every wave or by none.  A wave team's sync orders its global and LDS accesses
// at workgroup scope (the memory it shares is the workgroup's), with no barrier.
struct Team {
    int rank;    // the thread's index in the team
    int size;    // threads in the team: the workgroup's, or 64
    bool whole;  // the whole workgroup

    __device__ static Team block(int threads) { return Team{(int)threadIdx.x, threads, true}; }
    __device__ static Team wave() { return Team{(int)(threadIdx.x & 63), 64, false}; }
    __device__ int waves() const { return size >> 6; }
    __device__ __forceinline__ void sync() const
    {
        if (whole) {
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        }
    }
    // sync() that also returns the number of threads with p set
    __device__ __forceinline__ int sync_count(bool p) const
    {
        if (whole) return __syncthreads_count(p);
        const int c = __popcll(__ballot(p));
        sync();
        return c;
    }
};
__device__ __forceinline__ int ffs64(uint64_t m) { return __builtin_ctzll(m); }

__device__ __forceinline__ V3 ld3(const float (*a)[3], int i) { return mk3(a[i][0], a[i][1], a[i][2]); }
__device__ __forceinline__ void st3(float (*a)[3], int i, V3 v)
{
    a[i][0] = v.x;
    a[i][1] = v.y;
    a[i][2] = v.z;
}

// DPP move of a 32-bit value (GFX9 encodings: quad_perm 0x00-0xff, row_mirror
// 0x140, row_half_mirror 0x141; gfx90a and later: row_newbcast 0x150-0x15f,
// lane n of each 16-lane row to the whole row); every source lane of these
// patterns exists.
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

__device__ __forceinline__ float readlane_f(float v, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

__device__ __forceinline__ int readlane_i(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }

// Minimum over the 64 lanes (no NaN inputs): quad and row reductions by DPP, then
// the four row results through readlane.
__device__ __forceinline__ float wave_min(float v)
{
    v = fminf(v, dpp_f<0xB1>(v));   // quad_perm [1,0,3,2]
    v = fminf(v, dpp_f<0x4E>(v));   // quad_perm [2,3,0,1]
    v = fminf(v, dpp_f<0x141>(v));  // row_half_mirror
    v = fminf(v, dpp_f<0x140>(v));  // row_mirror
    return fminf(fminf(readlane_f(v, 0), readlane_f(v, 16)), fminf(readlane_f(v, 32), readlane_f(v, 48)));
}

// Wave argmin over (value, index) among candidates; ties -> lowest index.
template <typename T>
__device__ inline void wave_argmin(bool &valid, T &v, int &i)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        bool ov = __shfl_xor((int)valid, off, 64) != 0;
        T ovv = __shfl_xor(v, off, 64);
        int oi = __shfl_xor(i, off, 64);
        bool take = ov && (!valid || ovv < v || (ovv == v && oi < i));
        if (take) {
            valid = true;
            v = ovv;
            i = oi;
        }
    }
}


template <int CTRL>
__device__ __forceinline__ int dpp_i(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false);
}

// The two shapes of a pair as one wave holds them for EPA.
struct EpaShapes {
    int kind_a, kind_b;  // uniform
    V3 ca, cb;           // centres (spheres)
    float ra, rb;        // radii (spheres)
    V3 k;                // lanes 0-7: corner (lane) of A; lanes 8-15: corner (lane - 8) of B
};

__device__ __forceinline__ V3 pick_corner(const Shape &s, int k)
{
    V3 v = s.v[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) {
        const bool t = k == j;
        v.x = t ? s.v[j].x : v.x;
        v.y = t ? s.v[j].y : v.y;
        v.z = t ? s.v[j].z : v.z;
    }
    return v;
}

__device__ __forceinline__ EpaShapes epa_shapes(const Shape &A, const Shape &B)
{
    const int lane = lane_id();
    EpaShapes e;
    e.kind_a = A.kind;
    e.kind_b = B.kind;
    e.ca = A.c;
    e.cb = B.c;
    e.ra = A.r;
    e.rb = B.r;
    const V3 ka = pick_corner(A, lane & 7), kb = pick_corner(B, lane & 7);
    const bool onb = lane >= 8;
    e.k = mk3(onb ? kb.x : ka.x, onb ? kb.y : ka.y, onb ? kb.z : ka.z);
    return e;
}

// Supports of the boxes held as corners in lanes 0-7 (A, along d) and 8-15 (B,
// along -d), both at once: in each group of 8 lanes, the first corner of greatest
// dot(v, dir) among those above -FLT_MAX, else (0,0,0) -- GetCubeSupport's strict
// '>' scan from -FLT_MAX (code/nans.cpp:409-430).
__device__ __forceinline__ void box_supports(V3 kv, V3 d, V3 nd, V3 &sa, V3 &sb, int lane)
{
    const float dist = dot(kv, lane >= 8 ? nd : d);
    float key = dist > -FLT_MAX ? dist : -__builtin_inff();
    int idx = lane & 7;
    auto step = [&](float ok, int oi) {
        const bool take = ok > key || (ok == key && oi < idx);
        key = take ? ok : key;
        idx = take ? oi : idx;
    };
    step(dpp_f<0xB1>(key), dpp_i<0xB1>(idx));    // quad_perm [1,0,3,2]
    step(dpp_f<0x4E>(key), dpp_i<0x4E>(idx));    // quad_perm [2,3,0,1]
    step(dpp_f<0x141>(key), dpp_i<0x141>(idx));  // row_half_mirror: the other quad of the 8
    const float ka = readlane_f(key, 0), kb = readlane_f(key, 8);
    const int wa = readlane_i(idx, 0), wb = 8 + readlane_i(idx, 8);
    sa = ka == -__builtin_inff() ? mk3(0.0f, 0.0f, 0.0f)
                                 : mk3(readlane_f(kv.x, wa), readlane_f(kv.y, wa), readlane_f(kv.z, wa));
    sb = kb == -__builtin_inff() ? mk3(0.0f, 0.0f, 0.0f)
                                 : mk3(readlane_f(kv.x, wb), readlane_f(kv.y, wb), readlane_f(kv.z, wb));
}

// CalculateSupport (code/nans.cpp:463-519): S_A(d) and S_B(-d); every lane calls.
__device__ __forceinline__ Vtx wave_support(const EpaShapes &s, V3 d, int lane)
{
    const V3 nd = mul(d, -1.0f);
    Vtx v;
    V3 ga = mk3(0.0f, 0.0f, 0.0f), gb = mk3(0.0f, 0.0f, 0.0f);
    if (s.kind_a == SHAPE_BOX || s.kind_b == SHAPE_BOX) box_supports(s.k, d, nd, ga, gb, lane);
    v.A = s.kind_a == SHAPE_BOX ? ga : sphere_support(s.ca, s.ra, d);
    v.B = s.kind_b == SHAPE_BOX ? gb : sphere_support(s.cb, s.rb, nd);
    v.P = sub(v.A, v.B);
    return v;
}

// Position of the n-th set bit of m (n < __popc(m)).
__device__ __forceinline__ int nth_set_bit(uint64_t m, int n)
{
    int pos = 0;
#pragma unroll
    for (int w = 32; w >= 1; w >>= 1) {
        const uint64_t low = m & ((1ull << w) - 1ull);
        const int c = __popcll(low);
        if (n >= c) {
            n -= c;
            pos += w;
            m >>= w;
        } else {
            m = low;
        }
    }
    return pos;
}

// Equality class of a new vertex with id nv and point P against the vertices in
// registers (vertex == compares P, code/nans.h:251-254): the first earlier vertex
// with the same P, CLS_NAN if P has a NaN.  Every lane calls.
__device__ __forceinline__ int vertex_class_reg(V3 v0, V3 v1, int nv, V3 P, int lane)
{
    if (has_nan(P)) return CLS_NAN;
    const uint64_t m0 = ballot(lane < nv && veq(v0, P));
    if (m0) return ffs64(m0);
    const uint64_t m1 = ballot(lane + 64 < nv && veq(v1, P));
    return m1 ? 64 + ffs64(m1) : nv;
}

__device__ __forceinline__ float pick3f(int k, float a, float b, float c) { return k == 0 ? a : (k == 1 ? b : c); }
__device__ __forceinline__ int pick3i(int k, int a, int b, int c) { return k == 0 ? a : (k == 1 ? b : c); }

// A face in registers.
struct FaceR {
    float nx, ny, nz;  // stored normal (flipped away from the origin)
    float ax, ay, az;  // first vertex A
    float d;           // |dot(unflipped normal, A)| with glm's abs
    int id;            // a | b << 8 | c << 16
    int cl;            // classes of a, b, c
};

// PushTriangle (code/nans.cpp:291-322) of vertices (A, B, C) = (a, b, c).
__device__ __forceinline__ FaceR make_face(V3 A, V3 B, V3 C, int a, int b, int c, int ca, int cb, int cc)
{
    V3 n = normalize(cross(sub(B, A), sub(C, A)));
    FaceR f;
    f.d = gabs(dot(n, A));
    if (dot(A, n) < 0.0f) n = mul(n, -1.0f);
    f.nx = n.x; f.ny = n.y; f.nz = n.z;
    f.ax = A.x; f.ay = A.y; f.az = A.z;
    f.id = a | (b << 8) | (c << 16);
    f.cl = ca | (cb << 8) | (cc << 16);
    return f;
}

// Binary64 distance of the plane of A, B, C to the origin (FP64-islands final choice).
__device__ inline double face_plane64(V3 A, V3 B, V3 C)
{
    const double ax = A.x, ay = A.y, az = A.z;
    const double ux = (double)B.x - ax, uy = (double)B.y - ay, uz = (double)B.z - az;
    const double vx = (double)C.x - ax, vy = (double)C.y - ay, vz = (double)C.z - az;
    const double nx = uy * vz - vy * uz, ny = uz * vx - vz * ux, nz = ux * vy - vx * uy;
    const double inv = 1.0 / __builtin_sqrt((nx * nx + ny * ny) + nz * nz);
    const double d = ((nx * inv) * ax + (ny * inv) * ay) + (nz * inv) * az;
    return d >= 0.0 ? d : -d;
}

// The same for a face of the whole-wave polytope.
__device__ inline double face_dist64(const EpaLds &L, const FaceR &f)
{
    return face_plane64(mk3(f.ax, f.ay, f.az), ld3(L.vp, (f.id >> 8) & 255), ld3(L.vp, (f.id >> 16) & 255));
}

// ResolveCollision (code/nans.cpp:787-904) executed by one full wavefront.  The
// caller has written the GJK simplex to L.vp / L.va / L.vb[0..3], passes vertex
// (lane)'s P in p0 for lanes 0-3, and has called wave_sync().  Every lane returns
// the same result.
__device__ __forceinline__ EpaResult epa_wave(EpaLds &L, const EpaShapes &sh, V3 p0, const NarrowParams &p, int lane)
{
    EpaResult r;
    r.status = EPA_ITER;
    r.pa = r.pb = r.n = mk3(0.0f, 0.0f, 0.0f);
    r.depth = 0.0;
    r.iters = 0;
    r.max_faces = 4;
    r.nverts = 4;

    // vertices in registers: v0 = vertex (lane), v1 = vertex (64 + lane)
    V3 v0 = lane < 4 ? p0 : mk3(0.0f, 0.0f, 0.0f);
    V3 v1 = mk3(0.0f, 0.0f, 0.0f);
    int c0 = 0;
    {
        // classes of the simplex vertices: the first earlier vertex with the same P
        int cls = lane;
        bool found = false;
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            const V3 pu = mk3(readlane_f(v0.x, u), readlane_f(v0.y, u), readlane_f(v0.z, u));
            if (!found && u < lane && veq(pu, v0)) {
                cls = u;
                found = true;
            }
        }
        c0 = has_nan(v0) ? CLS_NAN : cls;
    }
    FaceR F[EPA_FSLOTS];
#pragma unroll
    for (int k = 0; k < EPA_FSLOTS; ++k) F[k] = FaceR{0, 0, 0, 0, 0, 0, 0, 0, 0};
    {
        // ABC, ACD, ADB, BDC (code/nans.cpp:799-802)
        const int a = lane == 3 ? 1 : 0;
        const int b = lane == 0 ? 1 : (lane == 1 ? 2 : 3);
        const int c = lane == 0 ? 2 : (lane == 1 ? 3 : (lane == 2 ? 1 : 2));
        const int ca = __shfl(c0, a, 64), cb = __shfl(c0, b, 64), cc = __shfl(c0, c, 64);
        if (lane < 4) F[0] = make_face(ld3(L.vp, a), ld3(L.vp, b), ld3(L.vp, c), a, b, c, ca, cb, cc);
    }
    int nf = 4, nv = 4;
    int iter = 0;
    while (iter++ <= p.max_epa_iterations) {
        r.iters += 1;
        if (nf == 0) {
            r.status = EPA_EMPTY;
            break;
        }
        // closest face
        const float d0 = readlane_f(gabs(dot(mk3(F[0].nx, F[0].ny, F[0].nz), mk3(F[0].ax, F[0].ay, F[0].az))), 0);
        float key[EPA_FSLOTS];
        float kmin = __builtin_inff();
#pragma unroll
        for (int k = 0; k < EPA_FSLOTS; ++k) {
            const int f = lane + 64 * k;
            key[k] = (f < nf && F[k].d < d0) ? F[k].d : __builtin_inff();
            kmin = fminf(kmin, key[k]);
        }
        const float m = wave_min(kmin);
        int best = 0;
        if (m != __builtin_inff()) {
#pragma unroll
            for (int k = EPA_FSLOTS - 1; k >= 0; --k) {
                uint64_t b = ballot(key[k] == m);
                if (b) best = 64 * k + ffs64(b);
            }
        }
        int owner = best & 63, ks = best >> 6;
        V3 N = mk3(readlane_f(pick3f(ks, F[0].nx, F[1].nx, F[2].nx), owner),
                   readlane_f(pick3f(ks, F[0].ny, F[1].ny, F[2].ny), owner),
                   readlane_f(pick3f(ks, F[0].nz, F[1].nz, F[2].nz), owner));
        float cur = m == __builtin_inff() ? d0 : readlane_f(pick3f(ks, F[0].d, F[1].d, F[2].d), owner);
        // new support along the stored normal
        const Vtx ns = wave_support(sh, N, lane);
        if (dot(N, ns.P) - cur < p.epa_tolerance) {
            double depth = (double)cur;
            if (p.fp64_islands) {
                wave_sync();
                double d64[EPA_FSLOTS];
#pragma unroll
                for (int k = 0; k < EPA_FSLOTS; ++k) d64[k] = (lane + 64 * k < nf) ? face_dist64(L, F[k]) : 0.0;
                const double f0 = __shfl(d64[0], 0, 64);
                bool v64 = false;
                double bd = 0.0;
                int bi64 = 0x7fffffff;
#pragma unroll
                for (int k = 0; k < EPA_FSLOTS; ++k) {
                    const int f = lane + 64 * k;
                    if (f < nf && d64[k] < f0 && (!v64 || d64[k] < bd)) {
                        v64 = true;
                        bd = d64[k];
                        bi64 = f;
                    }
                }
                wave_argmin(v64, bd, bi64);
                const int sel = v64 ? bi64 : 0;
                depth = v64 ? bd : f0;
                if (sel != best) {
                    best = sel;
                    owner = best & 63;
                    ks = best >> 6;
                    N = mk3(readlane_f(pick3f(ks, F[0].nx, F[1].nx, F[2].nx), owner),
                            readlane_f(pick3f(ks, F[0].ny, F[1].ny, F[2].ny), owner),
                            readlane_f(pick3f(ks, F[0].nz, F[1].nz, F[2].nz), owner));
                    cur = sel == 0 ? d0 : readlane_f(pick3f(ks, F[0].d, F[1].d, F[2].d), owner);
                }
            }
            const int id = readlane_i(pick3i(ks, F[0].id, F[1].id, F[2].id), owner);
            const int a = id & 255, b = (id >> 8) & 255, c = (id >> 16) & 255;
            wave_sync();
            V3 PA = ld3(L.vp, a), PB = ld3(L.vp, b), PC = ld3(L.vp, c);
            // Barycentric (code/nans.cpp:771-785) of N * d
            V3 P = mul(N, cur);
            V3 e0 = sub(PB, PA), e1 = sub(PC, PA), e2 = sub(P, PA);
            float d00 = dot(e0, e0), d01 = dot(e0, e1), d11 = dot(e1, e1);
            float d20 = dot(e2, e0), d21 = dot(e2, e1);
            float denom = d00 * d11 - d01 * d01;
            float V = (d11 * d20 - d01 * d21) / denom;
            float W = (d00 * d21 - d01 * d20) / denom;
            float U = 1.0f - V - W;
            if (fabsf(U) > 1.0f || fabsf(V) > 1.0f || fabsf(W) > 1.0f) {
                r.status = EPA_BARY;
            } else if (!isfinite(U) || !isfinite(V) || !isfinite(W)) {
                r.status = EPA_NONFINITE;
            } else {
                r.pa = add(add(mul(ld3(L.va, a), U), mul(ld3(L.va, b), V)), mul(ld3(L.va, c), W));
                r.n = mul(N, -1.0f);
                r.pb = add(add(mul(ld3(L.vb, a), U), mul(ld3(L.vb, b), V)), mul(ld3(L.vb, c), W));
                r.depth = depth;
                r.status = EPA_CONTACT;
            }
            break;
        }
        if (nv >= EPA_MAXV) {
            r.status = EPA_OVERFLOW;
            break;
        }
        // append the vertex
        const int vnew = nv;
        const int ncls = vertex_class_reg(v0, v1, vnew, ns.P, lane);
        if (lane == (vnew & 63)) {
            if (vnew < 64) v0 = ns.P;
            else v1 = ns.P;
        }
        if (lane == 0) {
            st3(L.vp, vnew, ns.P);
            st3(L.va, vnew, ns.A);
            st3(L.vb, vnew, ns.B);
        }
        nv += 1;
        r.nverts = nv;
        // visibility (code/nans.cpp:869-891): the recomputed flipped normal is the stored one
        uint64_t vis[EPA_FSLOTS];
        int nvis = 0;
#pragma unroll
        for (int k = 0; k < EPA_FSLOTS; ++k) {
            const int f = lane + 64 * k;
            const bool vv = f < nf && dot(mk3(F[k].nx, F[k].ny, F[k].nz),
                                          sub(ns.P, mk3(F[k].ax, F[k].ay, F[k].az))) > 0.0f;
            vis[k] = ballot(vv);
            nvis += __popcll(vis[k]);
        }
        // horizon edges in face order (PushEdge), edge e in lane e
        int ne = 0, ea = 0, eb = 0, eca = 0, ecb = 0;
        // fast path (all faces in one slot, at most 64 pushes): an edge survives iff
        // its reverse is not among the pushed edges, provided no key occurs twice
        bool sequential = nf > 64 || 3 * nvis > 64;
        if (!sequential) {
            const bool mine = (vis[0] >> lane) & 1ull;
            const int cl = F[0].cl;
            int key[3], rev[3], nsame[3] = {0, 0, 0}, nrev[3] = {0, 0, 0};
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                const int ca = (cl >> (8 * e)) & 255, cb = (cl >> (8 * ((e + 1) % 3))) & 255;
                key[e] = ca | (cb << 8);
                rev[e] = (ca == CLS_NAN || cb == CLS_NAN) ? -1 : (cb | (ca << 8));
            }
            uint64_t mk = vis[0];
            while (mk) {
                const int o = ffs64(mk);
                mk &= mk - 1;
                const int co = readlane_i(cl, o);
#pragma unroll
                for (int t = 0; t < 3; ++t) {
                    const int kt = ((co >> (8 * t)) & 255) | (((co >> (8 * ((t + 1) % 3))) & 255) << 8);
#pragma unroll
                    for (int e = 0; e < 3; ++e) {
                        nsame[e] += kt == key[e];
                        nrev[e] += kt == rev[e];
                    }
                }
            }
            bool dup = false;
#pragma unroll
            for (int e = 0; e < 3; ++e) dup |= rev[e] >= 0 && (nsame[e] > 1 || nrev[e] > 1);
            sequential = ballot(mine && dup) != 0ull;
            if (!sequential) {
                // kept edges of this lane's face, placed after those of earlier visible faces
                int keep = 0;
#pragma unroll
                for (int e = 0; e < 3; ++e) keep |= (rev[e] < 0 || nrev[e] == 0) ? (1 << e) : 0;
                const int cnt = mine ? __popc(keep) : 0;
                const uint64_t lower = (1ull << lane) - 1ull;
                const uint64_t b0 = ballot(cnt & 1), b1 = ballot(cnt & 2);
                int o = __popcll(b0 & lower) + 2 * __popcll(b1 & lower);
                ne = __popcll(b0) + 2 * __popcll(b1);
                if (mine) {
                    const int id = F[0].id;
#pragma unroll
                    for (int e = 0; e < 3; ++e) {
                        if ((keep >> e) & 1) {
                            const int s0 = 8 * e, s1 = 8 * ((e + 1) % 3);
                            L.eids[o] = ((id >> s0) & 255) | (((id >> s1) & 255) << 8);
                            L.ekey[o] = key[e];
                            ++o;
                        }
                    }
                }
                wave_sync();
                if (lane < ne) {
                    const int k2 = L.ekey[lane], i2 = L.eids[lane];
                    ea = i2 & 255;
                    eb = (i2 >> 8) & 255;
                    eca = k2 & 255;
                    ecb = (k2 >> 8) & 255;
                }
                wave_sync();
            }
        }
        bool overflow = false;
        if (sequential) {
            ne = 0;
#pragma unroll
            for (int k = 0; k < EPA_FSLOTS; ++k) {
                uint64_t mk = vis[k];
                while (mk) {
                    const int o = ffs64(mk);
                    mk &= mk - 1;
                    const int id = readlane_i(F[k].id, o), cl = readlane_i(F[k].cl, o);
                    const int fv[3] = {id & 255, (id >> 8) & 255, (id >> 16) & 255};
                    const int fc[3] = {cl & 255, (cl >> 8) & 255, (cl >> 16) & 255};
#pragma unroll
                    for (int e = 0; e < 3; ++e) {
                        const int A = fv[e], B = fv[(e + 1) % 3];
                        const int cA = fc[e], cB = fc[(e + 1) % 3];
                        const bool match = lane < ne && eca != CLS_NAN && eca == cB && ecb != CLS_NAN && ecb == cA;
                        const uint64_t mm = ballot(match);
                        if (mm) {
                            const int j = ffs64(mm);
                            const int na = __shfl_down(ea, 1, 64), nb = __shfl_down(eb, 1, 64);
                            const int nca = __shfl_down(eca, 1, 64), ncb = __shfl_down(ecb, 1, 64);
                            if (lane >= j) {
                                ea = na; eb = nb; eca = nca; ecb = ncb;
                            }
                            ne -= 1;
                        } else if (ne < 64) {
                            if (lane == ne) {
                                ea = A; eb = B; eca = cA; ecb = cB;
                            }
                            ne += 1;
                        } else {
                            overflow = true;
                        }
                    }
                }
            }
        }
        if (overflow) {
            r.status = EPA_OVERFLOW;
            break;
        }
        // ordered removal of the visible faces, then the new ones
        int nsurv = 0;
        int dst[EPA_FSLOTS];
        uint64_t am0 = 0ull;
#pragma unroll
        for (int k = 0; k < EPA_FSLOTS; ++k) {
            const int f = lane + 64 * k;
            const bool alive = f < nf && !((vis[k] >> lane) & 1ull);
            const uint64_t am = ballot(alive);
            if (k == 0) am0 = am;
            dst[k] = alive ? nsurv + __popcll(am & ((1ull << lane) - 1ull)) : -1;
            nsurv += __popcll(am);
        }
        if (nsurv + ne > EPA_MAXF) {
            r.status = EPA_OVERFLOW;
            break;
        }
        // PushTriangle(NewSupport, e.A, e.B) (code/nans.cpp:894-899) in lane e
        FaceR g = FaceR{0, 0, 0, 0, 0, 0, 0, 0, 0};
        wave_sync();  // lane 0's vertex stores before other lanes read L.vp
        if (lane < ne) g = make_face(ns.P, ld3(L.vp, ea), ld3(L.vp, eb), vnew, ea, eb, ncls, eca, ecb);
        const int nfn = nsurv + ne;
        if (nf <= 64 && nfn <= 64) {
            // lane f takes survivor f from its lane, or new face f - nsurv from its edge lane
            const bool old = lane < nsurv;
            const int src = old ? nth_set_bit(am0, lane) : lane - nsurv;
            const int adr = 4 * (src & 63);
            auto pull = [&](float a_, float b_) {
                const float x = __int_as_float(__builtin_amdgcn_ds_bpermute(adr, __float_as_int(a_)));
                const float y = __int_as_float(__builtin_amdgcn_ds_bpermute(adr, __float_as_int(b_)));
                return old ? x : y;
            };
            auto pulli = [&](int a_, int b_) {
                const int x = __builtin_amdgcn_ds_bpermute(adr, a_);
                const int y = __builtin_amdgcn_ds_bpermute(adr, b_);
                return old ? x : y;
            };
            FaceR h;
            h.nx = pull(F[0].nx, g.nx);
            h.ny = pull(F[0].ny, g.ny);
            h.nz = pull(F[0].nz, g.nz);
            h.ax = pull(F[0].ax, g.ax);
            h.ay = pull(F[0].ay, g.ay);
            h.az = pull(F[0].az, g.az);
            h.d = pull(F[0].d, g.d);
            h.id = pulli(F[0].id, g.id);
            h.cl = pulli(F[0].cl, g.cl);
            F[0] = h;
            nf = nfn;
            if (nf > r.max_faces) r.max_faces = nf;
            continue;
        }
        // otherwise through the LDS staging area
#pragma unroll
        for (int k = 0; k < EPA_FSLOTS; ++k) {
            if (dst[k] >= 0) {
                L.sfn[dst[k]][0] = F[k].nx;
                L.sfn[dst[k]][1] = F[k].ny;
                L.sfn[dst[k]][2] = F[k].nz;
                L.sfd[dst[k]] = F[k].d;
                L.sfid[dst[k]] = F[k].id;
                L.sfcl[dst[k]] = F[k].cl;
            }
        }
        if (lane < ne) {
            const int s = nsurv + lane;
            L.sfn[s][0] = g.nx;
            L.sfn[s][1] = g.ny;
            L.sfn[s][2] = g.nz;
            L.sfd[s] = g.d;
            L.sfid[s] = g.id;
            L.sfcl[s] = g.cl;
        }
        nf = nfn;
        if (nf > r.max_faces) r.max_faces = nf;
        wave_sync();
#pragma unroll
        for (int k = 0; k < EPA_FSLOTS; ++k) {
            const int f = lane + 64 * k;
            if (f < nf) {
                F[k].nx = L.sfn[f][0];
                F[k].ny = L.sfn[f][1];
                F[k].nz = L.sfn[f][2];
                F[k].d = L.sfd[f];
                F[k].id = L.sfid[f];
                F[k].cl = L.sfcl[f];
                const int a = F[k].id & 255;
                F[k].ax = L.vp[a][0];
                F[k].ay = L.vp[a][1];
                F[k].az = L.vp[a][2];
            }
        }
        wave_sync();
    }
    return r;
}

// ---------------------------------------------------------------------- four EPAs per wave
// ResolveCollision for 64/G pairs at once, one per G-lane group (G = 16: a row
// of the wave; G = 32: half a wave): the same steps as epa_wave, with the
// polytope of each pair held by its group -- face f and vertex v in lane f / v
// (P, SupA, SupB; P also in LDS for gathers) -- group reductions by row-local DPP
// (and one ds_bpermute across the two rows of a 32-lane group) and group
// broadcasts by ds_bpermute.  A polytope that outgrows its group (G+1 vertices,
// G+1 faces, G+1 horizon edges, or an edge key pushed twice) stops with EPA_SPILL
// and is redone from its simplex by the next wider tier (16 -> 32 -> epa_wave),
// so the result is always epa_wave's.
constexpr int EPA_SPILL = 99;

template <int G>
struct EpgLds {
    static_assert(G == 16 || G == 32, "groups of 16 or 32 lanes");
    float vp[64 / G][G][3];   // vertex P per group
    int edge[64];             // horizon edges per group (G each): ids a | b << 8, classes ca << 16 | cb << 24
    // horizon: the directed edges (ca, cb) that the visible faces push, bit cb of
    // word ca
    uint32_t pushed[64 / G][G];
    uint32_t seen[64 / G];      // positions of the visible faces
    uint32_t kept[64 / G][2];   // low and high bit of the number of edges each keeps, by position
};
static_assert(sizeof(EpgLds<16>) <= sizeof(EpaLds), "the grouped EPA reuses the wave's EPA LDS");
static_assert(sizeof(EpgLds<32>) <= sizeof(EpaLds), "the grouped EPA reuses the wave's EPA LDS");
static_assert(16 * 4 * 64 <= sizeof(EpaLds), "GJK keeps 16 words per lane in the EPA LDS");

__device__ __forceinline__ float gpull_f(float v, int src_lane)
{
    return __int_as_float(__builtin_amdgcn_ds_bpermute(src_lane << 2, __float_as_int(v)));
}
__device__ __forceinline__ int gpull_i(int v, int src_lane) { return __builtin_amdgcn_ds_bpermute(src_lane << 2, v); }
__device__ __forceinline__ V3 gpull3(V3 v, int src_lane)
{
    return mk3(gpull_f(v.x, src_lane), gpull_f(v.y, src_lane), gpull_f(v.z, src_lane));
}
// lane U of this lane's G-lane group, in every lane (G = 16: one row broadcast,
// no LDS round trip); the whole wave must be active
template <int G, int U>
__device__ __forceinline__ float gbcast_f(float v)
{
    if constexpr (G == 16) return dpp_f<0x150 + U>(v);
    else return gpull_f(v, (lane_id() & (64 - G)) + U);
}
template <int G, int U>
__device__ __forceinline__ int gbcast_i(int v)
{
    if constexpr (G == 16) return dpp_i<0x150 + U>(v);
    else return gpull_i(v, (lane_id() & (64 - G)) + U);
}
template <int G, int U>
__device__ __forceinline__ V3 gbcast3(V3 v)
{
    return mk3(gbcast_f<G, U>(v.x), gbcast_f<G, U>(v.y), gbcast_f<G, U>(v.z));
}

// this lane's G-lane group bits of a wave ballot
template <int G>
__device__ __forceinline__ uint32_t gbits(uint64_t m, int lane)
{
    return (uint32_t)(m >> (lane & (64 - G))) & (uint32_t)((1ull << G) - 1ull);
}
// minimum over the lane's group of G (no NaN inputs), in every lane of the group:
// a row of 16 by DPP, then the two rows of a 32-lane group through ds_bpermute
template <int G>
__device__ __forceinline__ float group_min(float v)
{
    v = fminf(v, dpp_f<0xB1>(v));
    v = fminf(v, dpp_f<0x4E>(v));
    v = fminf(v, dpp_f<0x141>(v));
    v = fminf(v, dpp_f<0x140>(v));
    if (G == 32) v = fminf(v, gpull_f(v, lane_id() ^ 16));
    return v;
}

// The group's shapes: lanes 0-7 of each row hold the corners of A, 8-15 of B.
// MEM: the shapes carry only Shape::vm (corners in memory, null for a sphere),
// and each lane reads its one corner from there.
template <bool MEM = false>
__device__ __forceinline__ EpaShapes epa_shapes_group(const Shape &A, const Shape &B, int lane = lane_id())
{
    const int j = lane & 15;
    EpaShapes e;
    e.kind_a = A.kind;
    e.kind_b = B.kind;
    e.ca = A.c;
    e.cb = B.c;
    e.ra = A.r;
    e.rb = B.r;
    const bool onb = j >= 8;
    if (MEM) {
        const float *vm = onb ? B.vm : A.vm;
        e.k = vm ? mk3(vm[3 * (j & 7)], vm[3 * (j & 7) + 1], vm[3 * (j & 7) + 2]) : mk3(0.0f, 0.0f, 0.0f);
    } else {
        const V3 ka = pick_corner(A, j & 7), kb = pick_corner(B, j & 7);
        e.k = mk3(onb ? kb.x : ka.x, onb ? kb.y : ka.y, onb ? kb.z : ka.z);
    }
    return e;
}

// CalculateSupport for each group's pair along its d (group-uniform).  Every row
// of 16 lanes holds the corners of A (lanes 0-7) and B (8-15); a butterfly of DPP
// moves inside each 8-lane half carries (dot, corner number, corner) to the first
// corner of greatest dot product -- GetCubeSupport's strict '>' scan in corner
// order -- and a row mirror hands each half the other half's winner.  No
// cross-lane traffic leaves the row, so a 32-lane group's two rows agree.
template <int G>
__device__ __forceinline__ Vtx group_support(const EpaShapes &s, V3 d, int lane)
{
    const int j = lane & 15;
    const V3 nd = mul(d, -1.0f);
    const float dist = dot(s.k, j >= 8 ? nd : d);
    float key = dist > -FLT_MAX ? dist : -__builtin_inff();
    int idx = j & 7;
    V3 cw = s.k;
    auto step = [&](float ok, int oi, float ox, float oy, float oz) {
        const bool take = ok > key || (ok == key && oi < idx);
        key = take ? ok : key;
        idx = take ? oi : idx;
        cw.x = take ? ox : cw.x;
        cw.y = take ? oy : cw.y;
        cw.z = take ? oz : cw.z;
    };
    step(dpp_f<0xB1>(key), dpp_i<0xB1>(idx), dpp_f<0xB1>(cw.x), dpp_f<0xB1>(cw.y), dpp_f<0xB1>(cw.z));
    step(dpp_f<0x4E>(key), dpp_i<0x4E>(idx), dpp_f<0x4E>(cw.x), dpp_f<0x4E>(cw.y), dpp_f<0x4E>(cw.z));
    step(dpp_f<0x141>(key), dpp_i<0x141>(idx), dpp_f<0x141>(cw.x), dpp_f<0x141>(cw.y), dpp_f<0x141>(cw.z));
    // this half's winner and, through the row mirror, the other half's
    const float ko = dpp_f<0x140>(key);
    const V3 co = mk3(dpp_f<0x140>(cw.x), dpp_f<0x140>(cw.y), dpp_f<0x140>(cw.z));
    const bool onb = j >= 8;
    const float ka = onb ? ko : key, kb = onb ? key : ko;
    const V3 ca = mk3(onb ? co.x : cw.x, onb ? co.y : cw.y, onb ? co.z : cw.z);
    const V3 cb = mk3(onb ? cw.x : co.x, onb ? cw.y : co.y, onb ? cw.z : co.z);
    // a sphere's support along -d is c - r n with the n of +d (as in minkowski):
    // one normalize serves both shapes and every group
    const bool sa = s.kind_a != SHAPE_BOX, sb = s.kind_b != SHAPE_BOX;
    V3 n = mk3(0.0f, 0.0f, 0.0f);
    if (sa || sb) n = normalize(d);
    Vtx v;
    v.A = sa ? add(s.ca, mul(n, s.ra)) : (ka == -__builtin_inff() ? mk3(0.0f, 0.0f, 0.0f) : ca);
    v.B = sb ? sub(s.cb, mul(n, s.rb)) : (kb == -__builtin_inff() ? mk3(0.0f, 0.0f, 0.0f) : cb);
    v.P = sub(v.A, v.B);
    return v;
}

// classes (ca | cb << 8) of edge e of a face with packed classes cl
__device__ __forceinline__ int edge_key(int cl, int e)
{
    return ((cl >> (8 * e)) & 255) | (((cl >> (8 * ((e + 1) % 3))) & 255) << 8);
}

// Every lane calls; lanes 0-3 of a group pass the supports of simplex vertex j in
// sa0 / sb0.  act: the group has a pair.  Returns the group's result (EPA_NONE for
// an idle group, EPA_SPILL to redo with the next wider tier).
// Binary64 distance of a group face's plane to the origin (FP64-islands final
// choice), its vertices b and c from the group's vertex LDS.
__device__ inline double group_face_dist64(const float (*vp)[3], const FaceR &f)
{
    return face_plane64(mk3(f.ax, f.ay, f.az), ld3(vp, (f.id >> 8) & 255), ld3(vp, (f.id >> 16) & 255));
}

// Argmin over (value, index) in each G-lane group, ties to the lowest index;
// every lane of the group receives the result.
template <int G>
__device__ __forceinline__ void group_argmin64(bool &valid, double &v, int &i)
{
#pragma unroll
    for (int off = 1; off < G; off <<= 1) {
        const double ov = __shfl_xor(v, off, 64);
        const int oi = __shfl_xor(i, off, 64);
        const int ok = __shfl_xor(valid ? 1 : 0, off, 64);
        const bool take = ok && (!valid || ov < v || (ov == v && oi < i));
        v = take ? ov : v;
        i = take ? oi : i;
        valid = valid || ok;
    }
}

// ISL: the FP64-islands mode, whose final face choice and depth are binary64
// (as epa_wave's).
template <int G, bool ISL = false>
__device__ __forceinline__ EpaResult epa_group(EpgLds<G> &L, const EpaShapes &sh, V3 sa0, V3 sb0, bool act,
                                      const NarrowParams &p, int lane)
{
    const int j = lane & (G - 1), gb = lane & (64 - G), g = lane / G;
    auto gbits = [lane](uint64_t m) { return nans::gbits<G>(m, lane); };
    EpaResult r;
    r.status = act ? EPA_ITER : EPA_NONE;
    r.pa = r.pb = r.n = mk3(0.0f, 0.0f, 0.0f);
    r.depth = 0.0;
    r.iters = 0;
    r.max_faces = 4;
    r.nverts = 4;
    bool run = act;
    const V3 z = mk3(0.0f, 0.0f, 0.0f);
    // vertex j of the group: P, SupA, SupB
    V3 VA = j < 4 ? sa0 : z, VB = j < 4 ? sb0 : z;
    V3 VP = j < 4 ? sub(sa0, sb0) : z;
    if (j < 4) st3(L.vp[g], j, VP);
    // the group's four simplex vertices in every lane of the group
    const V3 P0 = gbcast3<G, 0>(VP), P1 = gbcast3<G, 1>(VP), P2 = gbcast3<G, 2>(VP), P3 = gbcast3<G, 3>(VP);
    int c0;
    {
        int cls = j;
        bool found = false;
        const V3 pu[3] = {P0, P1, P2};
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            if (!found && u < j && veq(pu[u], VP)) {
                cls = u;
                found = true;
            }
        }
        c0 = has_nan(VP) ? CLS_NAN : cls;
    }
    FaceR F = FaceR{0, 0, 0, 0, 0, 0, 0, 0, 0};
    {
        // ABC, ACD, ADB, BDC (code/nans.cpp:799-802)
        const int a = j == 3 ? 1 : 0;
        const int b = j == 0 ? 1 : (j == 1 ? 2 : 3);
        const int c = j == 0 ? 2 : (j == 1 ? 3 : (j == 2 ? 1 : 2));
        const int C0 = gbcast_i<G, 0>(c0), C1 = gbcast_i<G, 1>(c0), C2 = gbcast_i<G, 2>(c0), C3 = gbcast_i<G, 3>(c0);
        V3 Pa = P0, Pb = P1, Pc = P1;
        fsel(Pa, a == 1, P1);
        fsel(Pb, b == 2, P2);
        fsel(Pb, b == 3, P3);
        fsel(Pc, c == 2, P2);
        fsel(Pc, c == 3, P3);
        const int ca = a == 1 ? C1 : C0;
        const int cb = b == 1 ? C1 : (b == 2 ? C2 : C3);
        const int cc = c == 1 ? C1 : (c == 2 ? C2 : C3);
        if (j < 4) F = make_face(Pa, Pb, Pc, a, b, c, ca, cb, cc);
    }
    // A face stays in the lane that made it; pos is its index in the reference's
    // face vector.  Erasing keeps the vector's order and new faces follow in edge
    // order, so a survivor's position falls by the visible faces before it, and the
    // new faces take the free lanes: no face is moved (staging the survivors and the
    // new faces through LDS and reading them back was 27 LDS accesses a trip; 1M
    // random pairs 4.75 -> 4.55 ms, 200k in the islands mode 1.61 -> 1.57 ms).
    bool al = j < 4;
    int pos = j, nf = 4, nv = 4, iter = 0;
    // A group that converges keeps its closest face (and, for the islands choice,
    // that face's lane) and stops: its polytope is frozen from then on, so the
    // contact points are computed once for every group after the loop rather than
    // on each iteration where some group converges.
    bool cv = false;
    V3 cN = z;
    float ccur = 0.0f;
    int cfid = 0, cbest = 0;
    // the horizon's sets (below), empty at the start of every trip
    auto clear_sets = [&]() {
        L.pushed[g][j] = 0u;
        if (j < 3) (j == 0 ? L.seen[g] : L.kept[g][j - 1]) = 0u;
    };
    clear_sets();
    wave_sync();
    for (;;) {
        // while (iter++ <= MAX_EPA_ITERATIONS), per group
        if (run && !(iter <= p.max_epa_iterations)) run = false;  // status stays EPA_ITER
        iter += 1;
        if (run) r.iters += 1;
        if (run && nf == 0) {
            r.status = EPA_EMPTY;
            run = false;
        }
        if (!ballot(run)) break;
        // closest face: the first face (by position) holding the minimum below face
        // 0's distance; F.d is also the scan's |dot(stored normal, A)|: the flip of
        // the normal only negates the dot product
        const uint32_t f0 = gbits(ballot(al && pos == 0));
        const int first = f0 ? ffs64(f0) : 0;
        const float d0 = gpull_f(F.d, gb + first);
        const float k0 = (al && F.d < d0) ? F.d : __builtin_inff();
        const float m = group_min<G>(k0);
        const uint32_t b0 = gbits(ballot(k0 == m));
        int best = (m != __builtin_inff() && b0) ? ffs64(b0) : first;
        if (ballot(m != __builtin_inff() && (b0 & (b0 - 1)))) {  // some group has a tie
            const float kp = k0 == m ? (float)pos : (float)(2 * G);
            const uint32_t bp = gbits(ballot(kp == group_min<G>(kp)));
            if (m != __builtin_inff() && bp) best = ffs64(bp);
        }
        const int owner = gb + best;
        const V3 N = mk3(gpull_f(F.nx, owner), gpull_f(F.ny, owner), gpull_f(F.nz, owner));
        const float cur = m == __builtin_inff() ? d0 : m;
        // new support along the stored normal
        const Vtx ns = group_support<G>(sh, N, lane);
        const bool conv = run && dot(N, ns.P) - cur < p.epa_tolerance;
        if (ballot(conv)) {
            const int fid = gpull_i(F.id, owner);
            if (conv) {
                cv = true;
                cN = N;
                ccur = gpull_f(F.d, owner);
                cfid = fid;
                cbest = best;
                run = false;
            }
        }
        if (run && nv >= G) {
            r.status = EPA_SPILL;
            run = false;
        }
        // append the vertex (its class: the first earlier vertex with the same P)
        const int vnew = nv;
        const uint32_t meq = gbits(ballot(j < nv && veq(VP, ns.P)));
        const int ncls = has_nan(ns.P) ? CLS_NAN : (meq ? ffs64(meq) : nv);
        if (run) {
            if (j == vnew) {
                VP = ns.P;
                VA = ns.A;
                VB = ns.B;
            }
            if (j == 0) st3(L.vp[g], vnew, ns.P);
            nv += 1;
            r.nverts = nv;
        }
        // visibility
        const bool w0 = run && al && dot(mk3(F.nx, F.ny, F.nz), sub(ns.P, mk3(F.ax, F.ay, F.az))) > 0.0f;
        // horizon: edges of the visible faces in face order; an edge survives iff its
        // reverse is not among them, when no key is pushed twice (else spill: a bit of
        // pushed[] found set).  Edges with a NaN class (not < G) never match, as
        // vertex == never holds for them, and enter no set.  The sets are empty here:
        // cleared before the loop and after each trip's last read of them.
        const int cl = F.cl;
        const uint32_t one = 1;
        bool dup = false;
        if (w0) {
            atomicOr(&L.seen[g], one << pos);
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                const int ke = edge_key(cl, e);
                const int ca = ke & 255, cb = ke >> 8;
                if (ca < G && cb < G) dup |= (atomicOr(&L.pushed[g][ca], one << cb) >> cb) & 1u;
            }
        }
        wave_sync();
        int keep = 0;
        if (w0) {
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                const int ke = edge_key(cl, e);
                const int ca = ke & 255, cb = ke >> 8;
                const bool rev = ca < G && cb < G && ((L.pushed[g][cb] >> ca) & 1u);
                keep |= rev ? 0 : 1 << e;
            }
            const int cnt = __popc(keep);
            if (cnt & 1) atomicOr(&L.kept[g][0], one << pos);
            if (cnt & 2) atomicOr(&L.kept[g][1], one << pos);
        }
        wave_sync();
        const uint32_t seen = L.seen[g], kept0 = L.kept[g][0], kept1 = L.kept[g][1];
        const uint32_t before = (one << pos) - 1;  // positions before this face's
        const int ne = __popc(kept0) + 2 * __popc(kept1);
        const int nsurv = nf - __popc(seen);
        if (run && (gbits(ballot(dup)) != 0 || nsurv + ne > G)) {
            r.status = EPA_SPILL;
            run = false;
        }
        if (run && keep) {
            int o = gb + __popc(kept0 & before) + 2 * __popc(kept1 & before);
            const int id = F.id;
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                if ((keep >> e) & 1) L.edge[o++] = edge_key(id, e) | (edge_key(cl, e) << 16);
            }
        }
        wave_sync();
        clear_sets();  // every read of the sets is behind the sync above
        // the visible faces leave, the survivors move up, and free lane number r of
        // the group makes the face of edge r
        if (run) {
            al = al && !w0;
            if (al) pos -= __popc(seen & before);
        }
        const uint32_t idle = gbits(ballot(!al));
        const int rf = __popc(idle & ((one << j) - 1));
        if (run) {
            if (!al && rf < ne) {
                const int ed = L.edge[gb + rf];
                const int ea = ed & 255, eb = (ed >> 8) & 255, eca = (ed >> 16) & 255, ecb = (ed >> 24) & 255;
                F = make_face(ns.P, ld3(L.vp[g], ea), ld3(L.vp[g], eb), vnew, ea, eb, ncls, eca, ecb);
                al = true;
                pos = nsurv + rf;
            }
            nf = nsurv + ne;
            if (nf > r.max_faces) r.max_faces = nf;
        }
        wave_sync();
    }
    if (ballot(cv)) {
        V3 Nc = cN;
        float cc = ccur;
        double depth = (double)ccur;
        int fid = cfid;
        if constexpr (ISL) {
            // the final face by binary64 plane distance: the first of the least
            // below face 0's, else face 0 (epa_wave's islands choice per group)
            wave_sync();
            const double d64 = al ? group_face_dist64(L.vp[g], F) : 0.0;
            const uint32_t m0 = gbits(ballot(al && pos == 0));
            const int first = m0 ? ffs64(m0) : 0;
            const double f0 = __shfl(d64, gb + first, 64);
            bool v64 = cv && al && d64 < f0;
            double bd = v64 ? d64 : 0.0;
            int bi = v64 ? pos : 0x7fffffff;
            group_argmin64<G>(v64, bd, bi);
            depth = v64 ? bd : f0;
            const uint32_t ms = gbits(ballot(al && pos == bi));
            const int sel = v64 && ms ? ffs64(ms) : first;  // its lane
            const int so = gb + sel;
            const V3 Ns = mk3(gpull_f(F.nx, so), gpull_f(F.ny, so), gpull_f(F.nz, so));
            const float ds = gpull_f(F.d, so);
            const int fs = gpull_i(F.id, so);
            if (sel != cbest) {
                Nc = Ns;
                cc = ds;
                fid = fs;
            }
        }
        const int a = fid & 255, b = (fid >> 8) & 255, c = (fid >> 16) & 255;
        const int am = gb + (a & (G - 1)), bm = gb + (b & (G - 1)), cm = gb + (c & (G - 1));
        const V3 PA = gpull3(VP, am), PB = gpull3(VP, bm), PC = gpull3(VP, cm);
        const V3 AA = gpull3(VA, am), AB = gpull3(VA, bm), AC = gpull3(VA, cm);
        const V3 BA = gpull3(VB, am), BB = gpull3(VB, bm), BC = gpull3(VB, cm);
        if (cv) {
            const V3 P = mul(Nc, cc);
            const V3 e0 = sub(PB, PA), e1 = sub(PC, PA), e2 = sub(P, PA);
            const float d00 = dot(e0, e0), d01 = dot(e0, e1), d11 = dot(e1, e1);
            const float d20 = dot(e2, e0), d21 = dot(e2, e1);
            const float denom = d00 * d11 - d01 * d01;
            const float V = (d11 * d20 - d01 * d21) / denom;
            const float W = (d00 * d21 - d01 * d20) / denom;
            const float U = 1.0f - V - W;
            if (fabsf(U) > 1.0f || fabsf(V) > 1.0f || fabsf(W) > 1.0f) {
                r.status = EPA_BARY;
            } else if (!isfinite(U) || !isfinite(V) || !isfinite(W)) {
                r.status = EPA_NONFINITE;
            } else {
                r.pa = add(add(mul(AA, U), mul(AB, V)), mul(AC, W));
                r.n = mul(Nc, -1.0f);
                r.pb = add(add(mul(BA, U), mul(BB, V)), mul(BC, W));
                r.depth = depth;
                r.status = EPA_CONTACT;
            }
        }
    }
    return r;
}

// ---------------------------------------------------------------------- an EPA per lane
// ResolveCollision for one pair of boxes by one lane: the step's contacts are shallow
// and end after a few iterations (of a batch of stacks' GJK hits 34 % after one, 95 %
// after four, 99.3 % after five), so a polytope of at most 8 vertices and 12 faces is
// small enough to keep EPL_LANES of them in a wave's polytope LDS, one lane's words
// EPL_LANES apart.  A trip then costs a wave about 1.3k instructions for up to
// EPL_LANES pairs, where the 16-lane groups spend 1k on four (their lanes past the
// polytope's faces idle, and every gather crosses lanes): 4096 worlds of 8-256 bodies
// 81.0 -> 67.8 ms per 60 steps, 601 with warm start 31.5 -> 25.6 ms per 30.  What outgrows a lane -- a
// ninth vertex, a thirteenth face, a ninth horizon edge, a NaN vertex -- goes to the
// wider tiers, as pairs with a sphere do.
constexpr int EPL_V = 8, EPL_F = 12;
constexpr int EPL_WORDS = 3 * EPL_V + 5 * EPL_F;  // vertices P, then faces: N, distance, vertex ids
constexpr int EPL_LANES = 24;
static_assert(4 * EPL_WORDS * EPL_LANES <= sizeof(EpaLds), "the lane polytopes fit the wave's EPA LDS");

struct EpaLane {
    float *w;            // the lane's words in LDS
    const float *va, *vb;  // the boxes' corners in memory
    int nf, nv, iter;
    unsigned long long ord;  // slot of the face at position i of the vector in bits 4i
    unsigned used;       // the slots that hold a face
    unsigned cls;        // equality class of vertex v in bits 4v
    unsigned sup;        // corners (8: none) of vertex 4 + k: A's in bits 8k, B's in 8k + 4
    int best;            // the closest face's slot, once the pair has converged

    __device__ float &at(int i) const { return w[i * EPL_LANES]; }
    __device__ V3 p(int v) const { return mk3(at(3 * v), at(3 * v + 1), at(3 * v + 2)); }
    __device__ void put(int v, V3 q) const
    {
        at(3 * v) = q.x;
        at(3 * v + 1) = q.y;
        at(3 * v + 2) = q.z;
    }
    static __device__ int face(int f) { return 3 * EPL_V + 5 * f; }
    __device__ V3 normal(int f) const { return mk3(at(face(f)), at(face(f) + 1), at(face(f) + 2)); }
    __device__ float dist(int f) const { return at(face(f) + 3); }
    __device__ int ids(int f) const { return __float_as_int(at(face(f) + 4)); }
    // PushTriangle (code/nans.cpp:291-322) in slot f
    __device__ __forceinline__ void push(int f, V3 A, V3 B, V3 C, int a, int b, int c) const
    {
        float d;
        const V3 n = plane(A, B, C, d);
        store(f, n, d, a | (b << 4) | (c << 8));
    }
    static __device__ __forceinline__ V3 plane(V3 A, V3 B, V3 C, float &dist)
    {
        V3 n = normalize(cross(sub(B, A), sub(C, A)));
        const float d = dot(n, A);
        if (d < 0.0f) n = mul(n, -1.0f);
        dist = gabs(d);
        return n;
    }
    __device__ __forceinline__ void store(int f, V3 n, float d, int ids) const
    {
        const int o = face(f);
        at(o) = n.x;
        at(o + 1) = n.y;
        at(o + 2) = n.z;
        at(o + 3) = d;
        at(o + 4) = __int_as_float(ids);
    }
};

// The corner of a box in memory that box_support picks, 8 for none.
__device__ __forceinline__ int corner_support(const float *v, V3 d, V3 &best)
{
    float maxd = -FLT_MAX;
    int idx = 8;
    best = mk3(0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const V3 c = mk3(v[3 * k], v[3 * k + 1], v[3 * k + 2]);
        const float dist = dot(c, d);
        const bool t = dist > maxd;
        maxd = t ? dist : maxd;
        idx = t ? k : idx;
        fsel(best, t, c);
    }
    return idx;
}

// The simplex of a queued hit as the lane's polytope; false if it has a NaN.
__device__ __forceinline__ bool epa_lane_start(EpaLane &e, const float *qa, const float *qb)
{
    V3 P[4];
    bool ok = true;
    e.cls = 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        P[v] = sub(mk3(qa[3 * v], qa[3 * v + 1], qa[3 * v + 2]), mk3(qb[3 * v], qb[3 * v + 1], qb[3 * v + 2]));
        ok = ok && !has_nan(P[v]);
        int c = v;
#pragma unroll
        for (int u = v - 1; u >= 0; --u) c = veq(P[u], P[v]) ? u : c;
        e.cls |= (unsigned)c << (4 * v);
        e.put(v, P[v]);
    }
    // ABC, ACD, ADB, BDC (code/nans.cpp:799-802)
    e.push(0, P[0], P[1], P[2], 0, 1, 2);
    e.push(1, P[0], P[2], P[3], 0, 2, 3);
    e.push(2, P[0], P[3], P[1], 0, 3, 1);
    e.push(3, P[1], P[3], P[2], 1, 3, 2);
    e.nf = e.nv = 4;
    e.ord = 0x3210;
    e.used = 0xF;
    e.iter = 0;
    e.sup = 0;
    return ok;
}

// One iteration of the loop (code/nans.cpp:804-902): EPA_NONE to go on, EPA_CONTACT
// once converged (e.best then is the closest face), another status if the loop ended,
// or EPA_SPILL.
__device__ __forceinline__ int epa_lane_trip(EpaLane &e, const NarrowParams &np)
{
    if (!(e.iter <= np.max_epa_iterations)) return EPA_ITER;
    e.iter += 1;
    if (e.nf == 0) return EPA_EMPTY;
    // closest face: the strict '<' scan from the first one
    int best = (int)e.ord & 15;
    float cur = e.dist(best);
    for (int i = 1; i < e.nf; i += 4) {
        const unsigned o = (unsigned)(e.ord >> (4 * i));
        float d[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) d[k] = e.dist((int)(o >> (4 * k)) & 15);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool t = i + k < e.nf && d[k] < cur;
            best = t ? (int)(o >> (4 * k)) & 15 : best;
            cur = t ? d[k] : cur;
        }
    }
    const V3 N = e.normal(best);
    V3 A, B;
    const int ia = corner_support(e.va, N, A);
    const int ib = corner_support(e.vb, mul(N, -1.0f), B);
    const V3 P = sub(A, B);
    if (dot(N, P) - cur < np.epa_tolerance) {
        e.best = best;
        return EPA_CONTACT;
    }
    if (e.nv >= EPL_V || has_nan(P)) return EPA_SPILL;
    // append the vertex
    const int vnew = e.nv;
    int nc = vnew;
#pragma unroll
    for (int v = EPL_V - 2; v >= 0; --v) nc = v < vnew && veq(e.p(v), P) ? v : nc;
    e.cls |= (unsigned)nc << (4 * vnew);
    e.sup |= (unsigned)(ia | (ib << 4)) << (8 * (vnew - 4));
    e.put(vnew, P);
    e.nv = vnew + 1;
    // visible faces, a bit per position
    unsigned vis = 0;
    for (int i = 0; i < e.nf; i += 2) {
        const unsigned o = (unsigned)(e.ord >> (4 * i));
        V3 n[2], a[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int f = (int)(o >> (4 * k)) & 15;
            n[k] = e.normal(f);
            a[k] = e.p(e.ids(f) & 7);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
            vis |= (i + k < e.nf && dot(n[k], sub(P, a[k])) > 0.0f) ? 1u << (i + k) : 0u;
    }
    // their directed edges as a set, bit 8 ca + cb; an edge pushed twice spills
    unsigned long long set = 0;
    bool dup = false;
    auto cls_of = [&](int v) { return (int)(e.cls >> (4 * v)) & 7; };
    for (unsigned m = vis; m; m &= m - 1) {
        const int id = e.ids((int)(e.ord >> (4 * __builtin_ctz(m))) & 15);
        const int ca = cls_of(id & 15), cb = cls_of((id >> 4) & 15), cc = cls_of(id >> 8);
        const unsigned long long b = (1ull << (8 * ca + cb)) | (1ull << (8 * cb + cc)) | (1ull << (8 * cc + ca));
        dup |= (set & b) != 0;
        set |= b;
    }
    // horizon (PushEdge, code/nans.cpp:232-266): in face order the edges whose reverse is
    // not in the set; vertices of edge k in byte k
    unsigned long long eids = 0;
    int ne = 0;
    for (unsigned m = vis; m; m &= m - 1) {
        const int id = e.ids((int)(e.ord >> (4 * __builtin_ctz(m))) & 15);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int a = (id >> (4 * k)) & 15, b = (id >> (4 * ((k + 1) % 3))) & 15;
            if (!((set >> (8 * cls_of(b) + cls_of(a))) & 1)) {
                eids |= (unsigned long long)(unsigned)(a | (b << 4)) << ((8 * ne) & 63);
                ne += 1;
            }
        }
    }
    if (dup || ne > 8 || e.nf - __popc(vis) + ne > EPL_F) return EPA_SPILL;
    // the visible faces leave the vector, the new ones follow in edge order
    int nf = e.nf;
    for (unsigned m = vis; m;) {
        const int i = 31 - __builtin_clz(m);
        m ^= 1u << i;
        e.used &= ~(1u << ((int)(e.ord >> (4 * i)) & 15));
        const unsigned long long low = (1ull << (4 * i)) - 1ull;
        e.ord = (e.ord & low) | ((e.ord >> 4) & ~low);
        nf -= 1;
    }
    e.ord &= (1ull << (4 * nf)) - 1ull;
    // two at a time, their chains side by side
    for (int k = 0; k < ne; k += 2) {
        const int ab = (int)(eids >> (8 * k)), a = ab & 7, b = (ab >> 4) & 7, a2 = (ab >> 8) & 7, b2 = (ab >> 12) & 7;
        const V3 A0 = e.p(a), B0 = e.p(b), A1 = e.p(a2), B1 = e.p(b2);
        float d0, d1;
        const V3 n0 = EpaLane::plane(P, A0, B0, d0), n1 = EpaLane::plane(P, A1, B1, d1);
        int f = __builtin_ctz(~e.used);
        e.store(f, n0, d0, vnew | (a << 4) | (b << 8));
        e.used |= 1u << f;
        e.ord |= (unsigned long long)f << (4 * (nf + k));
        if (k + 1 < ne) {
            f = __builtin_ctz(~e.used);
            e.store(f, n1, d1, vnew | (a2 << 4) | (b2 << 8));
            e.used |= 1u << f;
            e.ord |= (unsigned long long)f << (4 * (nf + k + 1));
        }
    }
    e.nf = nf + ne;
    return EPA_NONE;
}

// The contact of a converged lane (code/nans.cpp:826-866; ISL: the final face by
// binary64 plane distance, as epa_group's).  qa, qb: the queued simplex's supports.
template <bool ISL>
__device__ __forceinline__ EpaResult epa_lane_finish(const EpaLane &e, const float *qa, const float *qb)
{
    EpaResult r;
    r.pa = r.pb = r.n = mk3(0.0f, 0.0f, 0.0f);
    int best = e.best;
    r.depth = (double)e.dist(best);
    if constexpr (ISL) {
        double d0 = 0.0, bd = 0.0;
        for (int i = 0; i < e.nf; ++i) {
            const int f = (int)(e.ord >> (4 * i)) & 15, id = e.ids(f);
            const double d = face_plane64(e.p(id & 15), e.p((id >> 4) & 15), e.p((id >> 8) & 15));
            if (i == 0) d0 = bd = d;
            if (i == 0 || (d < d0 && d < bd)) {
                bd = d;
                best = f;
            }
        }
        r.depth = bd;
    }
    const V3 N = e.normal(best);
    const int id = e.ids(best), a = id & 15, b = (id >> 4) & 15, c = (id >> 8) & 15;
    const V3 PA = e.p(a), PB = e.p(b), PC = e.p(c);
    // Barycentric (code/nans.cpp:771-785) of N * d
    const V3 P = mul(N, e.dist(best));
    const V3 e0 = sub(PB, PA), e1 = sub(PC, PA), e2 = sub(P, PA);
    const float d00 = dot(e0, e0), d01 = dot(e0, e1), d11 = dot(e1, e1);
    const float d20 = dot(e2, e0), d21 = dot(e2, e1);
    const float denom = d00 * d11 - d01 * d01;
    const float V = (d11 * d20 - d01 * d21) / denom;
    const float W = (d00 * d21 - d01 * d20) / denom;
    const float U = 1.0f - V - W;
    if (fabsf(U) > 1.0f || fabsf(V) > 1.0f || fabsf(W) > 1.0f) {
        r.status = EPA_BARY;
    } else if (!isfinite(U) || !isfinite(V) || !isfinite(W)) {
        r.status = EPA_NONFINITE;
    } else {
        // a vertex's supports: the simplex's from its record, the others' from the boxes
        auto support = [&](const float *q, const float *box, int v, int shift) {
            const int k = (int)(e.sup >> (8 * (v & 3) + shift)) & 15;
            if (v >= 4 && k == 8) return mk3(0.0f, 0.0f, 0.0f);
            const float *x = v < 4 ? q + 3 * v : box + 3 * k;
            return mk3(x[0], x[1], x[2]);
        };
        r.pa = add(add(mul(support(qa, e.va, a, 0), U), mul(support(qa, e.va, b, 0), V)),
                   mul(support(qa, e.va, c, 0), W));
        r.n = mul(N, -1.0f);
        r.pb = add(add(mul(support(qb, e.vb, a, 4), U), mul(support(qb, e.vb, b, 4), V)),
                   mul(support(qb, e.vb, c, 4), W));
        r.status = EPA_CONTACT;
    }
    return r;
}

// ---------------------------------------------------------------------- block driver
// CheckCollision (code/nans.cpp:906-966) over the candidates [0, ncand) of one
// workgroup, in two phases:
//   GJK  every lane runs one candidate's EvolveSimplex loop; lanes whose loops
//        have ended take the next candidates together once GJK_REFILL_MIN of
//        them wait (work is handed out per wave by one LDS atomic), so a wave is
//        not held by its slowest lane;
//   EPA  the GJK hits are queued with their simplex; the waves take queued hits (LDS
//        atomic) and run ResolveCollision on them, a pair per lane or four per wave,
//        with the polytopes in the wave's LDS block.  A wave starts on the queue as
//        soon as its own GJK lanes are done, while other waves still run GJK: a
//        hit's queue slot is published with a release store of its candidate
//        index, and a lane that takes a slot not yet published waits for it, or
//        for every wave to leave GJK (then the slot will never be filled).
// Results go through the source object, per candidate, so their order is that
// of the candidates whatever the order of the work.
struct NarrowShared {
    int next;      // next candidate to hand out
    int nepa;      // GJK hits queued (in the end all of them)
    int epa_next;  // next queued hit to hand out
    int gjk_done;  // waves that have left the GJK phase
    int stalled;   // queue waits that hit their bound (counted as EPA overflow)
    int nwide[2];      // hits for the 16-lane groups: with a sphere, outgrown a lane
    int wide_next[2];  // next of them to hand out
};

// Bound of a wave's wait for a queue slot (each round sleeps ~128 cycles): far
// beyond any GJK phase, so reaching it means a fault, which is counted and the
// slot skipped rather than waited on for ever.
constexpr int EPA_WAIT_ROUNDS = 1 << 20;

// First EvolveSimplex call whose state enters the cycle check (any start finds
// a cycle; a later one spares the loops that end early).
constexpr int GJK_CYCLE_START = 8;

// Idle GJK lanes take new candidates once this many of them wait (or no lane
// is busy), so that the refill code runs once for a batch of lanes (config 3 on
// the MI355X: 1.429 ms per step at 16, 1.413 at 32-56, 1.484 at 64).
constexpr int GJK_REFILL_MIN = 48;

// Candidates per wave up to which a team's EPA runs in 16-lane groups: the few hits of
// so small a world leave most lanes idle, and a trip of the lanes' EPA lasts longer
// (1024 worlds of 16 bodies, 29 candidates a wave, rollout and gradient: 24.4 ms with
// lanes, 22.7 with groups; 48 worlds of 8-64, up to some 300 a wave: 4.9 against 6.7).
constexpr int EPL_MIN = 48;

// Lanes that wait for new pairs in the EPA phase before they are served, so that the
// code that starts and ends pairs runs for several.
constexpr int EPL_REFILL = 8;

// A queued GJK hit's simplex: the supports on A and B of its four vertices (the
// Minkowski point is recomputed as SupA - SupB, the expression that made it),
// and the pair's key (the source's key(c)), so that EPA looks nothing else up.
struct SimplexRec {
    float a[12], b[12];
    int key;
    int next;  // list of the slots whose pairs outgrew a lane (narrow_team)
};

__device__ __forceinline__ void simplex_rec_put(SimplexRec &q, const Vtx &v, int k)
{
    q.a[3 * k] = v.A.x; q.a[3 * k + 1] = v.A.y; q.a[3 * k + 2] = v.A.z;
    q.b[3 * k] = v.B.x; q.b[3 * k + 1] = v.B.y; q.b[3 * k + 2] = v.B.z;
}

__device__ __forceinline__ void simplex_rec_store(SimplexRec &q, const Simplex &S)
{
    simplex_rec_put(q, S.s0, 0);
    simplex_rec_put(q, S.s1, 1);
    simplex_rec_put(q, S.s2, 2);
    simplex_rec_put(q, S.s3, 3);
}

// One lane's GJK loop (CheckCollision's EvolveSimplex calls, code/nans.cpp:906-966)
// over the candidates it is handed.
//
// GJK cycles: EvolveSimplex's next call depends only on the simplex's Minkowski
// points (SupA/SupB ride along), so once the points repeat bit for bit the calls
// repeat for ever and the loop can only end at the cap.  Each lane keeps one
// earlier state (Brent's scheme, started at call GJK_CYCLE_START: saved after that
// call and then 1, 2, 4, ... calls later) in cyc[], its wave's [16][64] floats
// (P of s0..s3, n, then the pair's first direction).  Most loops end before the
// start, and pay nothing for the check.
struct GjkLane {
    Shape A, B;
    Simplex S;
    int c = -1, key = 0, calls = 0, power = 1, lam = 0;
    bool saved = false, retired = false;
};

// Candidate c for the lane (c >= ncand: none left, the lane retires).
template <class Src>
__device__ __forceinline__ void gjk_lane_take(GjkLane &G, const Src &src, int c, int ncand, float *cyc)
{
    if (c >= ncand) {
        G.retired = true;
        return;
    }
    const int tid = lane_id();
    G.c = c;
    G.key = src.key(c);
    src.shapes(G.key, G.A, G.B);
    const V3 d0 = gjk_first_dir(G.A, G.B);  // kept beside the cycle state
    cyc[13 * 64 + tid] = d0.x;
    cyc[14 * 64 + tid] = d0.y;
    cyc[15 * 64 + tid] = d0.z;
    G.S.n = 0;
    G.calls = 0;
    G.saved = false;
}

// One EvolveSimplex call of the lane's candidate, with the cycle check: the
// outcome once the loop has ended (GJK_NO, GJK_FOUND, or GJK_CAP at the 65-call
// cap), else GJK_STILL.
__device__ __forceinline__ int gjk_lane_call(GjkLane &G, float *cyc, const NarrowParams &np)
{
    const int tid = lane_id();
    Simplex &S = G.S;
    const V3 d0 = mk3(cyc[13 * 64 + tid], cyc[14 * 64 + tid], cyc[15 * 64 + tid]);
    int res = evolve_simplex(G.A, G.B, S, np.fp64_islands, d0);
    ++G.calls;
    if (res == GJK_STILL && G.calls <= np.max_gjk_iterations && G.calls >= GJK_CYCLE_START) {
        const float st[13] = {S.s0.P.x, S.s0.P.y, S.s0.P.z, S.s1.P.x, S.s1.P.y, S.s1.P.z,
                              S.s2.P.x, S.s2.P.y, S.s2.P.z, S.s3.P.x, S.s3.P.y, S.s3.P.z,
                              __int_as_float(S.n)};
        if (G.saved) {
            bool same = __float_as_int(cyc[12 * 64 + tid]) == S.n;
#pragma unroll
            for (int k = 0; k < 12; ++k)
                same = same && (k >= 3 * S.n || __float_as_int(cyc[k * 64 + tid]) == __float_as_int(st[k]));
            if (same) res = GJK_CAP;  // a repeated state: the cap is certain
        }
        ++G.lam;
        if (res == GJK_STILL && (!G.saved || G.lam == G.power)) {
#pragma unroll
            for (int k = 0; k < 13; ++k) cyc[k * 64 + tid] = st[k];
            G.power = G.saved ? 2 * G.power : 1;
            G.saved = true;
            G.lam = 0;
        }
    }
    if (res != GJK_STILL || G.calls > np.max_gjk_iterations) return res == GJK_STILL ? GJK_CAP : res;
    return GJK_STILL;
}

// EPA of one queued pair by the whole wave: supports of its four simplex vertices
// in q, every lane returns the result.
__device__ __forceinline__ EpaResult epa_whole(EpaLds &L, const EpaShapes &es, const SimplexRec &q, const NarrowParams &np,
                                              int lane = lane_id())
{
    V3 p0 = mk3(0.0f, 0.0f, 0.0f);
    if (lane < 4) {
        const V3 a = mk3(q.a[3 * lane], q.a[3 * lane + 1], q.a[3 * lane + 2]);
        const V3 b = mk3(q.b[3 * lane], q.b[3 * lane + 1], q.b[3 * lane + 2]);
        p0 = sub(a, b);
        st3(L.va, lane, a);
        st3(L.vb, lane, b);
        st3(L.vp, lane, p0);
    }
    wave_sync();
    const EpaResult r = epa_wave(L, es, p0, np, lane);
    wave_sync();
    return r;
}

// Four queue slots (job, uniform over each 16-lane group; groups without act idle along
// on a valid one) of candidates c in the 16-lane groups; one that outgrows its group by
// the whole wave.  Between its shapes' set-up and its loop it calls next().
template <bool ISL, class Src, class Next>
__device__ __forceinline__ void epa_four(const Src &src, EpaLds &L, const SimplexRec *qsim, int job, int c, bool act,
                                         const NarrowParams &np, int lane, Next &&next)
{
    const int j = lane & 15;
    const SimplexRec &q = qsim[job];
    const int key = q.key;
    Shape A, B;
    src.shapes_ref(key, A, B);
    const EpaShapes es = epa_shapes_group<true>(A, B, lane);
    V3 sa0 = mk3(0.0f, 0.0f, 0.0f), sb0 = sa0;
    if (j < 4) {
        sa0 = mk3(q.a[3 * j], q.a[3 * j + 1], q.a[3 * j + 2]);
        sb0 = mk3(q.b[3 * j], q.b[3 * j + 1], q.b[3 * j + 2]);
    }
    wave_sync();
    next();
    const EpaResult r = epa_group<16, ISL>(*reinterpret_cast<EpgLds<16> *>(&L), es, sa0, sb0, act, np, lane);
    if (act && j == 0 && r.status != EPA_SPILL) src.epa_result(c, key, r);
    wave_sync();
    for (uint64_t sp = ballot(act && j == 0 && r.status == EPA_SPILL); sp; sp &= sp - 1) {
        const int l = ffs64(sp);
        const int js = __builtin_amdgcn_readlane(job, l), cs = __builtin_amdgcn_readlane(c, l);
        const int ks = __builtin_amdgcn_readlane(key, l);
        Shape SA, SB;
        src.shapes_ref(ks, SA, SB);
        const EpaResult rw = epa_whole(L, epa_shapes_group<true>(SA, SB, lane), qsim[js], np, lane);
        if (lane == 0) src.epa_result(cs, ks, rw);
    }
}

// A lane number that the compiler does not know as threadIdx.x & 63: the wider tiers'
// lane constants are then worked out where they are used, not kept in registers through
// the step's other phases (168-register kernels: 45 spilled registers -> 10).
__device__ __forceinline__ int opaque_lane()
{
    int lane = lane_id();
    asm volatile("" : "+v"(lane));
    return lane;
}

// Source interface (duck-typed):
//   int key(int c) const                                 the pair of candidate c, as an int
//   void shapes(int key, Shape &A, Shape &B) const       both shapes of the pair
//   void shapes_ref(int key, Shape &A, Shape &B) const   the same with Shape::vm (box corners in
//                                                        memory) and no v[]
//   void gjk_result(int c, int gjk) const                 every candidate
//   void epa_result(int c, int key, const EpaResult &r) const   every GJK hit (lane 0 calls)
// ISL: the FP64-islands mode (the final face chosen in binary64).
// The team's wave k uses epa[k]; sh, qidx and qsim are the team's own.
template <bool ISL = false, class Src>
__device__ __forceinline__ void narrow_team(const Team &team, const Src &src, int ncand, const NarrowParams &np, EpaLds *epa,
                            NarrowShared &sh, int *qidx, SimplexRec *qsim)
{
    const int lane = lane_id();
    if (team.rank == 0) {
        sh.next = 0;
        sh.nepa = 0;
        sh.epa_next = 0;
        sh.gjk_done = 0;
        sh.stalled = 0;
        sh.nwide[0] = sh.nwide[1] = sh.wide_next[0] = sh.wide_next[1] = 0;
    }
    const int NW = team.waves();
    const bool lanes = ncand > EPL_MIN * NW;  // boxes a pair per lane
    for (int k = team.rank; k < ncand; k += team.size) qidx[k] = -1;  // queue slots: unpublished
    team.sync();
    {
        // GJK lanes (gjk_lane_call); the cycle state lives in the wave's EPA LDS,
        // idle until the wave's GJK ends
        float *cyc = reinterpret_cast<float *>(&epa[team.rank >> 6]);
        GjkLane G;
        for (;;) {
            const bool need = G.c < 0 && !G.retired;
            const uint64_t m = ballot(need);
            if (m && (__popcll(m) >= GJK_REFILL_MIN || !ballot(G.c >= 0))) {
                int base = 0;
                if (lane == 0) base = atomicAdd(&sh.next, __popcll(m));
                base = __builtin_amdgcn_readfirstlane(base);
                if (need) gjk_lane_take(G, src, base + __popcll(m & ((1ull << lane) - 1ull)), ncand, cyc);
            }
            if (!ballot(G.c >= 0)) break;
            if (G.c >= 0) {
                const int g = gjk_lane_call(G, cyc, np);
                if (g != GJK_STILL) {
                    src.gjk_result(G.c, g);
                    if (g == GJK_FOUND) {
                        // pairs that no lane takes from the back, marked below -1
                        const bool wide = lanes && (G.A.kind != SHAPE_BOX || G.B.kind != SHAPE_BOX);
                        const int q = wide ? ncand - 1 - atomicAdd(&sh.nwide[0], 1) : atomicAdd(&sh.nepa, 1);
                        simplex_rec_store(qsim[q], G.S);
                        qsim[q].key = G.key;
                        // publish the slot after its simplex
                        __hip_atomic_store(&qidx[q], wide ? -2 - G.c : G.c, __ATOMIC_RELEASE,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                    G.c = -1;
                }
            }
        }
        // this wave's queue slots are published before it counts itself out
        if (lane == 0) __hip_atomic_fetch_add(&sh.gjk_done, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    EpaLds &L = epa[team.rank >> 6];
    if (!lanes) {
        // few pairs, whose latency counts: four at a time in 16-lane groups, started while
        // other waves may still be in GJK.  The next pass's slots are claimed while this
        // one starts, their contents loaded (relaxed) under its work, and then confirmed
        // by an acquire fence, or waited for.
        const int ol = opaque_lane(), j = ol & 15;
        auto claim = [&]() __attribute__((always_inline)) {
            int b = 0;
            if (ol == 0) b = atomicAdd(&sh.epa_next, 4);
            return __builtin_amdgcn_readfirstlane(b);
        };
        auto peek = [&](int b) __attribute__((always_inline)) {
            const int job = b + (ol >> 4);
            return job < ncand ? __hip_atomic_load(&qidx[job], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : -1;
        };
        // the candidate of this group's slot, or -1 once it is certain the slot stays
        // empty (every wave has left GJK and it was never published)
        auto resolve = [&](int b, int seen) __attribute__((always_inline)) {
            const int job = b + (ol >> 4);
            int c = -1;
            if (job < ncand) {
                if (seen >= 0 && seen < ncand) {
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                    return seen;
                }
                for (int round = 0;; ++round) {
                    const bool last =
                        __hip_atomic_load(&sh.gjk_done, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) == NW;
                    c = __hip_atomic_load(&qidx[job], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
                    const bool bad = c >= ncand;  // not a candidate of this block: never published here
                    if (bad || (c < 0 && !last && round >= EPA_WAIT_ROUNDS)) {
                        if (j == 0) atomicAdd(&sh.stalled, 1);
                        c = -1;
                        break;
                    }
                    if (c >= 0 || last) break;
                    __builtin_amdgcn_s_sleep(2);
                }
            }
            return c;
        };
        int base = claim();
        int c = resolve(base, peek(base));
        for (;;) {
            // slots are filled in order, so an empty first slot ends the queue
            if (__builtin_amdgcn_readlane(c, 0) < 0) break;
            const bool act = c >= 0;
            const int c0 = __builtin_amdgcn_readlane(c, 0);
            int nbase = 0, seen = -1;
            epa_four<ISL>(src, L, qsim, act ? base + (ol >> 4) : base, act ? c : c0, act, np, ol, [&]() {
                nbase = claim();
                seen = peek(nbase);
            });
            base = nbase;
            c = resolve(base, seen);
        }
        team.sync();
        return;
    }
    // more: a pair of boxes per lane of EPL_LANES, started as above; a lane takes a queue
    // slot, waits for it to be published, and goes on to another when its pair is done.
    // Slots are taken and contacts worked out for EPL_REFILL lanes together.  Pairs with a
    // sphere, and after them what outgrew a lane, run after the queue's end (inside this
    // loop the wider tiers' lane constants would live through it), four at a time in
    // 16-lane groups and then, if they outgrow those, by the whole wave.
    // Waves share them: chained to the wave that met them, worlds of boxes and spheres
    // waited for the longest chain (500 worlds of 50 boxes and 50 spheres, 30 steps, 18.6
    // ms, now 13.3; one of 40 and 40 turned and overlapping, 10 steps, 11.9 ms, now 8.1,
    // 8.5 with groups only).
    const uint64_t lower = (1ull << lane) - 1ull;
    EpaLane e;
    e.w = reinterpret_cast<float *>(&L) + (lane < EPL_LANES ? lane : 0);
    int job = -1, c = -1;         // the lane's slot, and its candidate once it runs
    int st = EPA_NONE;            // of the pair: EPA_NONE while it runs
    bool out = lane >= EPL_LANES; // no more slots for this lane
    int rounds = 0;
    wave_sync();
    for (;;) {
        const uint64_t running = ballot(c >= 0 && st == EPA_NONE);
        if (!running || __popcll(running) <= EPL_LANES - EPL_REFILL) {
            // the pairs that are done
            if (c >= 0 && st != EPA_NONE) {
                if (st != EPA_SPILL) {
                    EpaResult r;
                    if (st == EPA_CONTACT) {
                        r = epa_lane_finish<ISL>(e, qsim[job].a, qsim[job].b);
                    } else {
                        r.pa = r.pb = r.n = mk3(0.0f, 0.0f, 0.0f);
                        r.depth = 0.0;
                        r.status = st;
                    }
                    src.epa_result(c, qsim[job].key, r);
                }
            }
            if (c >= 0 && st == EPA_SPILL) qsim[atomicAdd(&sh.nwide[1], 1)].next = job;
            if (c >= 0 && st != EPA_NONE) job = c = -1;
            // slots for the idle lanes
            const bool need = job < 0 && !out;
            const uint64_t m = ballot(need);
            if (m) {
                int b = 0;
                if (lane == 0) b = atomicAdd(&sh.epa_next, __popcll(m));
                b = __builtin_amdgcn_readfirstlane(b);
                if (need) job = b + __popcll(m & lower);
            }
            // start the pairs whose slots are published; a slot stays empty once every
            // wave has left GJK without filling it
            bool wait = job >= 0 && c < 0;
            if (wait) {
                const bool last = __hip_atomic_load(&sh.gjk_done, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) == NW;
                const int q = job < ncand ? __hip_atomic_load(&qidx[job], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP)
                                          : -1;
                if (q >= 0 && q < ncand) {
                    c = q;
                    Shape A, B;
                    src.shapes_ref(qsim[job].key, A, B);
                    e.va = A.vm;
                    e.vb = B.vm;
                    st = epa_lane_start(e, qsim[job].a, qsim[job].b) ? EPA_NONE : EPA_SPILL;
                    wait = false;
                } else if (q >= ncand || last || job >= ncand) {
                    if (q >= ncand) atomicAdd(&sh.stalled, 1);
                    job = -1;
                    out = true;
                    wait = false;
                }
            }
            if (!ballot(c >= 0)) {
                const uint64_t w = ballot(wait);
                if (!w) {
                    if (!ballot(!out)) break;
                    continue;
                }
                if (++rounds >= EPA_WAIT_ROUNDS) {
                    if (lane == 0) atomicAdd(&sh.stalled, __popcll(w));
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
                continue;
            }
        }
        if (c >= 0 && st == EPA_NONE) st = epa_lane_trip(e, np);
    }
    // the pairs with a sphere, all listed once every wave has left GJK, are shared out
    // before those that outgrew a lane, listed once every wave has come here
    for (rounds = 0; __hip_atomic_load(&sh.gjk_done, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) != NW;) {
        if (++rounds >= EPA_WAIT_ROUNDS) {
            if (lane == 0) atomicAdd(&sh.stalled, 1);
            break;
        }
        __builtin_amdgcn_s_sleep(2);
    }
    const int ol = opaque_lane();
    for (int list = 0; list < 2;) {
        int b = 0;
        if (ol == 0) b = atomicAdd(&sh.wide_next[list], 4);
        b = __builtin_amdgcn_readfirstlane(b);
        const int total = __builtin_amdgcn_readfirstlane(
            __hip_atomic_load(&sh.nwide[list], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
        if (b >= total) {
            team.sync();
            ++list;
            continue;
        }
        const int k = b + (ol >> 4);
        const bool act = k < total;
        const int i = act ? k : b;
        const int slot = list ? qsim[i].next : ncand - 1 - i;
        const int q = qidx[slot];
        epa_four<ISL>(src, L, qsim, slot, list ? q : -2 - q, act, np, ol, []() {});
    }
    if (team.rank == 0) sh.nepa += sh.nwide[0];  // all GJK hits
}

// The same driver for one wave on its own: CheckCollision over the candidates
// [0, ncand) of src, with no other wave to wait for.  A GJK hit's simplex goes to
// sim(c), and the wave lists its hits in list[0, ncand): pairs for the narrow tier
// from the front, pairs for the wide tier from the back.  The tiers then run over
// dense lists: four pairs at a time in 16-lane groups, their spills with the wide list
// two at a time in 32-lane groups, and what outgrows those by the whole wave.  A wave
// with one hit gives it to the whole wave at once, and two to the 32-lane tier, since
// the lanes are idle otherwise and the narrow tiers' attempts would only lengthen the
// chain.  The tiers see an opaque lane (25 spilled registers -> 2; 777 pairs 137 -> 124
// us, 200k 1.06 -> 1.04 ms).  Returns whether a pair hit.
template <bool ISL, class Src>
__device__ __forceinline__ bool narrow_wave(const Src &src, int ncand, const NarrowParams &np, EpaLds &L, int *list)
{
    const int lane = lane_id();
    const uint64_t lower = (1ull << lane) - 1ull;
    auto fence = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    };
    int nn = 0, nw = 0;  // hits of the narrow and of the wide list
    {
        float *cyc = reinterpret_cast<float *>(&L);
        GjkLane G;
        int next = 0;
        for (;;) {
            const bool need = G.c < 0 && !G.retired;
            const uint64_t m = ballot(need);
            if (m && (__popcll(m) >= GJK_REFILL_MIN || !ballot(G.c >= 0))) {
                if (need) gjk_lane_take(G, src, next + __popcll(m & lower), ncand, cyc);
                next += __popcll(m);
            }
            if (!ballot(G.c >= 0)) break;
            int g = GJK_STILL;
            if (G.c >= 0) g = gjk_lane_call(G, cyc, np);
            const bool hit = g == GJK_FOUND;
            if (g != GJK_STILL) {
                src.gjk_result(G.c, g);
                if (hit) {
                    SimplexRec &q = src.sim(G.c);
                    simplex_rec_store(q, G.S);
                    q.key = G.key;
                }
            }
            // a sphere's support gives a new vertex at every iteration, so its polytopes
            // outgrow a 16-lane group
            const bool wide = hit && (G.A.kind != SHAPE_BOX || G.B.kind != SHAPE_BOX);
            const uint64_t mn = ballot(hit && !wide), mw = ballot(wide);
            if (hit) list[wide ? ncand - 1 - nw - __popcll(mw & lower) : nn + __popcll(mn & lower)] = G.c;
            nn += __popcll(mn);
            nw += __popcll(mw);
            if (g != GJK_STILL) G.c = -1;
        }
    }
    fence();
    int nspill = 0;  // pairs that outgrew the narrow tier, at list[0, nspill)
    if (nn + nw <= 2) {
        nspill = nn;
    } else {
        EpgLds<16> &G = *reinterpret_cast<EpgLds<16> *>(&L);
        const int ol = opaque_lane(), j = ol & 15;
        for (int base = 0; base < nn; base += 4) {
            const int k = base + (ol >> 4);
            const bool act = k < nn;
            const int c = list[act ? k : base];
            const SimplexRec &q = src.sim(c);
            const int key = q.key;
            Shape A, B;
            src.shapes(key, A, B);
            const EpaShapes es = epa_shapes_group(A, B, ol);
            V3 sa0 = mk3(0.0f, 0.0f, 0.0f), sb0 = sa0;
            if (j < 4) {
                sa0 = mk3(q.a[3 * j], q.a[3 * j + 1], q.a[3 * j + 2]);
                sb0 = mk3(q.b[3 * j], q.b[3 * j + 1], q.b[3 * j + 2]);
            }
            wave_sync();
            const EpaResult r = epa_group<16, ISL>(G, es, sa0, sb0, act, np, ol);
            if (act && j == 0 && r.status != EPA_SPILL) src.epa_result(c, key, r);
            // the spilled pairs move to the front of the list, over entries already read
            const bool sp = act && j == 0 && r.status == EPA_SPILL;
            const uint64_t ms = ballot(sp);
            if (sp) list[nspill + __popcll(ms & ((1ull << ol) - 1ull))] = c;
            nspill += __popcll(ms);
        }
        fence();
    }
    // the wide tiers over the spills, then the wide list
    const int nwide = nspill + nw;
    auto item = [&](int k) { return list[k < nspill ? k : ncand - 1 - (k - nspill)]; };
    EpgLds<32> &G2 = *reinterpret_cast<EpgLds<32> *>(&L);
    const int wl = opaque_lane(), jw = wl & 31;
    for (int base = 0; base < nwide; base += 2) {
        const int k = base + (wl >> 5);
        const bool act = k < nwide;
        const int c = item(act ? k : base);
        uint64_t sp = 1;  // a pair on its own goes to the whole wave
        if (nwide > 1) {
            const SimplexRec &q = src.sim(c);
            const int key = q.key;
            Shape A, B;
            src.shapes(key, A, B);
            const EpaShapes es = epa_shapes_group(A, B, wl);
            V3 sa0 = mk3(0.0f, 0.0f, 0.0f), sb0 = sa0;
            if (jw < 4) {
                sa0 = mk3(q.a[3 * jw], q.a[3 * jw + 1], q.a[3 * jw + 2]);
                sb0 = mk3(q.b[3 * jw], q.b[3 * jw + 1], q.b[3 * jw + 2]);
            }
            wave_sync();
            const EpaResult r = epa_group<32, ISL>(G2, es, sa0, sb0, act, np, wl);
            if (act && jw == 0 && r.status != EPA_SPILL) src.epa_result(c, key, r);
            sp = ballot(act && jw == 0 && r.status == EPA_SPILL);
            wave_sync();
        }
        for (; sp; sp &= sp - 1) {
            const int cw = __builtin_amdgcn_readlane(c, ffs64(sp));
            const SimplexRec &q = src.sim(cw);
            const int key = q.key;
            Shape A, B;
            src.shapes(key, A, B);
            const EpaResult r = epa_whole(L, epa_shapes(A, B), q, np, wl);
            if (wl == 0) src.epa_result(cw, key, r);
        }
    }
    fence();
    return nn + nw != 0;
}

}  // namespace nans
