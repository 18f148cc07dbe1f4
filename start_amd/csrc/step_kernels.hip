// Step kernels of the particle path (gfx950).
//
// One launch = step_main    one thread per particle: skip rules, push, move,
//                           collision, certified relocation, charge, for the
//                           steps fused in the launch
//           -> step_resolve one thread per deferred particle: exact tet walk
//                           along the step segment, surface hit and settle,
//                           grid search for degenerate cases, charge.
// The rare exact work (segments through edges and vertices, end points on
// faces) is compacted into a work list so the streaming kernel stays short.
#include <type_traits>

#include "kernels.h"
#include "predicates.h"

namespace sg {

// ---------------------------------------------------------------------------
// exact geometry on the device
// ---------------------------------------------------------------------------
__device__ inline void load_node(const DevMesh& M, int32_t n, double* p)
{
    p[0] = M.nodes[3 * (int64_t)n];
    p[1] = M.nodes[3 * (int64_t)n + 1];
    p[2] = M.nodes[3 * (int64_t)n + 2];
}

__device__ inline int nth(const int4& v, int k) { return k == 0 ? v.x : (k == 1 ? v.y : (k == 2 ? v.z : v.w)); }

// closed containment: 0 outside, 1 on the boundary, 2 strictly inside, -1 error
__device__ int tet_contains(const DevMesh& M, int32_t t, const double* p)
{
    int4 nv = M.tnode[t];
    double P[4][3];
    for (int k = 0; k < 4; ++k) load_node(M, nth(nv, k), P[k]);
    int strict = 1;
    for (int f = 0; f < 4; ++f) {
        int s = orient3d(P[kFace[f][0]], P[kFace[f][1]], P[kFace[f][2]], p);
        if (s == 2) return -1;
        if (s < 0) return 0;
        if (s == 0) strict = 0;
    }
    return strict ? 2 : 1;
}

__device__ inline void bary64(const double* __restrict__ g, double x, double y, double z, double lam[4])
{
    double dx = x - g[0], dy = y - g[1], dz = z - g[2];
    lam[1] = (g[3] * dx + g[4] * dy) + g[5] * dz;
    lam[2] = (g[6] * dx + g[7] * dy) + g[8] * dz;
    lam[3] = (g[9] * dx + g[10] * dy) + g[11] * dz;
    lam[0] = 1.0 - ((lam[1] + lam[2]) + lam[3]);
}

// rounding bound of lambda at a point whose coordinates are l (tau: the bound
// where sum |l| <= 2; it is linear in |x - v0| <= diam * sum |l|)
__device__ inline double walk_tol(double tau, const double l[4])
{
    const double s = (fabs(l[0]) + fabs(l[1])) + (fabs(l[2]) + fabs(l[3]));
    return tau * fmax(1.0, 0.5 * s) * (1.0 + 1e-6);
}

// tau up to which the (1 + 1e-6) of walk_tol covers the rounding of sum |l|
constexpr double kMaxTau = 1e-7;

// The barycentric map of one tet in registers.
struct TetMap {
    double g[12];
    __device__ inline void load(const DevMesh& M, int32_t t)
    {
        const double2* p = reinterpret_cast<const double2*>(M.geo + 12 * (int64_t)t);
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const double2 d = p[q];
            g[2 * q] = d.x;
            g[2 * q + 1] = d.y;
        }
    }
};

// Sides of the tet's faces that p lies on, as orient3d gives them: bit f of
// pos: strictly inside face f, of neg: strictly outside.  A face whose
// coordinate is within its rounding bound is in neither; the exact predicates
// decide it.
struct Sides {
    int pos, neg;
};
__device__ inline Sides certified_sides(const DevMesh& M, const TetMap& m, const double* p)
{
    double l[4];
    bary64(m.g, p[0], p[1], p[2], l);
    const double tol = M.tau < kMaxTau ? walk_tol(M.tau, l) : INFINITY;
    Sides s{0, 0};
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        s.pos |= (int)(l[f] > tol) << f;
        s.neg |= (int)(l[f] < -tol) << f;
    }
    return s;
}

__device__ inline bool in_box(const TetBox& b, const double* p)
{
    bool in = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) in &= (p[k] >= (double)b.lo[k]) & (p[k] <= (double)b.hi[k]);
    return in;
}

// minimum-id tet whose closed volume holds p (CubicGrid.cpp:94-104, :149-159).
// The candidates of a cell (48 where the cells of the grid are those of a
// structured mesh, with the owner near the end) are dropped by their FP32
// bounding boxes, rounded outwards, eight loads at a time; one that is left is
// decided by its barycentric map and only within that map's rounding bound by
// the exact predicates, which need its four nodes.  In id order throughout, so
// that the answer is the exact scan's on any mesh.
__device__ int32_t locate_grid(const DevMesh& M, const double* p, int* strict, int* err)
{
    constexpr int kBatch = 8;
    int a = grid_coord(M.grid, 0, p[0]), b = grid_coord(M.grid, 1, p[1]), c = grid_coord(M.grid, 2, p[2]);
    int64_t cell = ((int64_t)a * M.grid.div[1] + b) * M.grid.div[2] + c;
    const int32_t end = M.tgrid_start[cell + 1];
    const bool finite = isfinite(p[0]) && isfinite(p[1]) && isfinite(p[2]);  // else the predicates' answer
    for (int32_t j = M.tgrid_start[cell]; j < end; j += kBatch) {
        int32_t id[kBatch];
        TetBox box[kBatch];
#pragma unroll
        for (int q = 0; q < kBatch; ++q) id[q] = M.tgrid_list[min(j + q, end - 1)];
#pragma unroll
        for (int q = 0; q < kBatch; ++q) box[q] = M.tbox[id[q]];
        int in = 0;
#pragma unroll
        for (int q = 0; q < kBatch; ++q) {
            in |= (int)((in_box(box[q], p) | !finite) & (j + q < end)) << q;
        }
        while (in) {
            const int q = __ffs(in) - 1;
            in &= in - 1;
            const int32_t t = M.tgrid_list[j + q];
            TetMap m;
            m.load(M, t);
            const Sides sd = certified_sides(M, m, p);
            if (sd.neg) continue;
            int r = 2;
            if (sd.pos != 15) {
                r = tet_contains(M, t, p);
                if (r < 0) {
                    *err = 1;
                    continue;
                }
            }
            if (r > 0) {
                *strict = (r == 2);
                return t;
            }
        }
    }
    *strict = 0;
    return -1;
}

// closed segment/triangle intersection (SegmentTriangleIntersection.cpp:7-40);
// *t = parameter of the intersection point the reference ranks by distance
__device__ int seg_tri(const double* p, const double* q, const double* a, const double* b, const double* c,
                       double* t, int* err)
{
    int sp = orient3d(a, b, c, p), sq = orient3d(a, b, c, q);
    if (sp == 2 || sq == 2) { *err = 1; return 0; }
    if ((sp > 0 && sq > 0) || (sp < 0 && sq < 0)) return 0;
    if (sp == 0 && sq == 0) {
        double ux = b[0] - a[0], uy = b[1] - a[1], uz = b[2] - a[2];
        double wx = c[0] - a[0], wy = c[1] - a[1], wz = c[2] - a[2];
        double nx = fabs(uy * wz - uz * wy), ny = fabs(uz * wx - ux * wz), nz = fabs(ux * wy - uy * wx);
        int i0, i1;
        if (nx >= ny && nx >= nz) { i0 = 1; i1 = 2; }
        else if (ny >= nz) { i0 = 0; i1 = 2; }
        else { i0 = 0; i1 = 1; }
        double P2[2] = {p[i0], p[i1]}, Q2[2] = {q[i0], q[i1]};
        double V[3][2] = {{a[i0], a[i1]}, {b[i0], b[i1]}, {c[i0], c[i1]}};
        auto in_tri = [&](const double* X) {
            int o1 = orient2d(V[0], V[1], X), o2 = orient2d(V[1], V[2], X), o3 = orient2d(V[2], V[0], X);
            if (o1 == 2 || o2 == 2 || o3 == 2) *err = 1;
            return (o1 >= 0 && o2 >= 0 && o3 >= 0) || (o1 <= 0 && o2 <= 0 && o3 <= 0);
        };
        auto on_seg = [](const double* s0, const double* s1, const double* r) {
            return fmin(s0[0], s1[0]) <= r[0] && r[0] <= fmax(s0[0], s1[0]) && fmin(s0[1], s1[1]) <= r[1] &&
                   r[1] <= fmax(s0[1], s1[1]);
        };
        auto seg_seg = [&](const double* p1, const double* p2, const double* q1, const double* q2) {
            int d1 = orient2d(q1, q2, p1), d2 = orient2d(q1, q2, p2);
            int d3 = orient2d(p1, p2, q1), d4 = orient2d(p1, p2, q2);
            if (((d1 > 0 && d2 < 0) || (d1 < 0 && d2 > 0)) && ((d3 > 0 && d4 < 0) || (d3 < 0 && d4 > 0))) return true;
            if (d1 == 0 && on_seg(q1, q2, p1)) return true;
            if (d2 == 0 && on_seg(q1, q2, p2)) return true;
            if (d3 == 0 && on_seg(p1, p2, q1)) return true;
            if (d4 == 0 && on_seg(p1, p2, q2)) return true;
            return false;
        };
        bool p_in = in_tri(P2);
        bool hit = p_in || in_tri(Q2) || seg_seg(P2, Q2, V[0], V[1]) || seg_seg(P2, Q2, V[1], V[2]) ||
                   seg_seg(P2, Q2, V[2], V[0]);
        if (!hit) return 0;
        if (p_in) {
            *t = 0.0;
        } else {
            double best = 1.0;
            for (int k = 0; k < 3; ++k) {
                const double* e0 = V[k];
                const double* e1 = V[(k + 1) % 3];
                double ex = e1[0] - e0[0], ey = e1[1] - e0[1];
                double dx = Q2[0] - P2[0], dy = Q2[1] - P2[1];
                double den = dx * ey - dy * ex;
                if (den == 0.0) continue;
                double tt = ((e0[0] - P2[0]) * ey - (e0[1] - P2[1]) * ex) / den;
                if (tt >= 0.0 && tt < best) best = tt;
            }
            *t = best;
        }
        return 1;
    }
    int o1 = orient3d(p, q, a, b), o2 = orient3d(p, q, b, c), o3 = orient3d(p, q, c, a);
    if (o1 == 2 || o2 == 2 || o3 == 2) { *err = 1; return 0; }
    bool hit = (o1 >= 0 && o2 >= 0 && o3 >= 0) || (o1 <= 0 && o2 <= 0 && o3 <= 0);
    if (!hit) return 0;
    if (sp == 0) *t = 0.0;
    else if (sq == 0) *t = 1.0;
    else {
        double pm;
        double fp = orient3d_fast(a, b, c, p, pm), fq = orient3d_fast(a, b, c, q, pm);
        *t = fp / (fp - fq);
    }
    return 1;
}

// closest surface triangle met by the closed segment p->q, ties to the
// smaller id (ParticleSurfaceCollisionHandler.cpp:104-123)
__device__ int32_t first_hit_grid(const DevMesh& M, const double* p, const double* q, int* err)
{
    int i0[3], i1[3];
    for (int k = 0; k < 3; ++k) {
        i0[k] = grid_coord(M.grid, k, fmin(p[k], q[k]));
        i1[k] = grid_coord(M.grid, k, fmax(p[k], q[k]));
    }
    int32_t best = -1;
    double best_t = INFINITY;
    for (int a = i0[0]; a <= i1[0]; ++a)
        for (int b = i0[1]; b <= i1[1]; ++b)
            for (int c = i0[2]; c <= i1[2]; ++c) {
                int64_t cell = ((int64_t)a * M.grid.div[1] + b) * M.grid.div[2] + c;
                for (int32_t j = M.sgrid_start[cell]; j < M.sgrid_start[cell + 1]; ++j) {
                    int32_t s = M.sgrid_list[j];
                    if (M.tri_degenerate[s]) continue;
                    double A[3], B[3], Cc[3];
                    load_node(M, M.tris[3 * (int64_t)s], A);
                    load_node(M, M.tris[3 * (int64_t)s + 1], B);
                    load_node(M, M.tris[3 * (int64_t)s + 2], Cc);
                    double t;
                    if (!seg_tri(p, q, A, B, Cc, &t, err)) continue;
                    if (t < best_t || (t == best_t && s < best)) {
                        best_t = t;
                        best = s;
                    }
                }
            }
    return best;
}

struct Resolved {
    int32_t hit;     // >= 0: settled on this triangle
    int32_t tet;     // owner of x1 (-1: outside the mesh)
    int32_t strict;  // x1 strictly inside tet
    int32_t exhaustive;
    int32_t err;
};

// The tet behind one of the faces in `neg`, in the order of step `it`, and only
// if there is no other the one it came from; -1: these are boundary faces.
__device__ inline int32_t next_tet(const int4& nb, int neg, int32_t prev, int it)
{
    int32_t next = -1, back = -1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int f = (q + it) & 3;
        const int32_t c = nth(nb, f);
        if (!(neg >> f & 1) || c < 0) continue;
        if (c != prev) {
            if (next < 0) next = c;
        } else {
            back = c;
        }
    }
    return next < 0 ? back : next;
}

// Owner of p starting from a nearby tet: visibility walk (move across a face
// whose plane separates p from the tet) until p is strictly inside a tet,
// which is then the unique (so minimum-id) closed-containing tet.  A point on
// a face/edge/vertex, a walk that reaches the boundary or runs long goes to
// the grid search, which applies the minimum-id rule directly.
__device__ int32_t locate_near_exact(const DevMesh& M, int32_t hint, const double* p, int* strict, int* err)
{
    int32_t t = hint, prev = -1;
    for (int it = 0; t >= 0 && it < 64; ++it) {
        int4 nv = M.tnode[t];
        double P[4][3];
#pragma unroll
        for (int k = 0; k < 4; ++k) load_node(M, nth(nv, k), P[k]);
        int s[4], nneg = 0, nzero = 0;
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            s[f] = orient3d(P[kFace[f][0]], P[kFace[f][1]], P[kFace[f][2]], p);
            if (s[f] == 2) {
                *err = 1;
                s[f] = 0;
            }
            nneg += s[f] < 0;
            nzero += s[f] == 0;
        }
        if (nneg == 0) {
            if (nzero == 0) {
                *strict = 1;
                return t;
            }
            break;  // on the boundary of t: ties need the grid's minimum-id rule
        }
        // cross a separating face, preferring one that does not lead back
        int neg = 0;
#pragma unroll
        for (int f = 0; f < 4; ++f) neg |= (int)(s[f] < 0) << f;
        const int32_t next = next_tet(M.tnbr[t], neg, prev, it);
        if (next < 0) break;  // separated by a boundary face: outside or non-convex
        prev = t;
        t = next;
    }
    return locate_grid(M, p, strict, err);
}

// The same walk as long as every sign is certain from the barycentric maps
// (which decide them without the nodes): true when it ends in the tet that
// holds p strictly inside, then t and its map m.
__device__ inline bool walk_near(const DevMesh& M, int32_t& t, TetMap& m, const double* p)
{
    int32_t cur = t, prev = -1;
#pragma unroll 1
    for (int it = 0; it < 64; ++it) {
        const Sides s = certified_sides(M, m, p);
        if (s.pos == 15) {
            t = cur;
            return true;
        }
        if ((s.pos | s.neg) != 15) return false;
        const int32_t next = next_tet(M.tnbr[cur], s.neg, prev, it);
        if (next < 0) return false;
        prev = cur;
        cur = next;
        m.load(M, cur);
    }
    return false;
}

__device__ int32_t locate_near(const DevMesh& M, int32_t hint, const double* p, int* strict, int* err)
{
    int32_t t = hint;
    TetMap m;
    m.load(M, t);
    if (walk_near(M, t, m, p)) {
        *strict = 1;
        return t;
    }
    return locate_near_exact(M, hint, p, strict, err);
}

__device__ Resolved resolve_exhaustive(const DevMesh& M, const double* x0, const double* x1, int32_t hint)
{
    Resolved r{-1, -1, 0, 1, 0};
    r.hit = first_hit_grid(M, x0, x1, &r.err);
    if (r.hit < 0) {
        int strict = 0;
        r.tet = hint >= 0 ? locate_near(M, hint, x1, &strict, &r.err) : locate_grid(M, x1, &strict, &r.err);
        r.strict = strict;
    }
    return r;
}

// Straight walk from t0 (x0 strictly inside) along x0->x1 through exit faces.
// Generic crossings are decided with exact signs; any zero sign (the segment
// meets an edge, a vertex or ends on a face) falls back to the grid search,
// which applies the reference rules directly.
__device__ __noinline__ Resolved resolve(const DevMesh& M, const double* x0, const double* x1, int32_t t0,
                                        bool strict0)
{
    if (t0 < 0 || !strict0) return resolve_exhaustive(M, x0, x1, t0);
    int32_t t = t0;
    int entry = -1;
    for (int iter = 0; iter < 256; ++iter) {
        int4 nv = M.tnode[t];
        double P[4][3];
        for (int k = 0; k < 4; ++k) load_node(M, nth(nv, k), P[k]);
        int s[4];
        int neg = 0, zero = 0;
        for (int f = 0; f < 4; ++f) {
            s[f] = orient3d(P[kFace[f][0]], P[kFace[f][1]], P[kFace[f][2]], x1);
            if (s[f] == 2) return resolve_exhaustive(M, x0, x1, t0);
            neg += s[f] < 0;
            zero += s[f] == 0;
        }
        if (neg == 0) {
            if (zero == 0) return Resolved{-1, t, 1, 0, 0};
            return resolve_exhaustive(M, x0, x1, t0);  // x1 on a face/edge/vertex of t
        }
        int exit_f = -1, nexit = 0;
        for (int f = 0; f < 4; ++f) {
            if (f == entry || s[f] >= 0) continue;
            const double* a = P[kFace[f][0]];
            const double* b = P[kFace[f][1]];
            const double* c = P[kFace[f][2]];
            int o1 = orient3d(x0, x1, a, b), o2 = orient3d(x0, x1, b, c), o3 = orient3d(x0, x1, c, a);
            if (o1 == 0 || o2 == 0 || o3 == 0 || o1 == 2 || o2 == 2 || o3 == 2)
                return resolve_exhaustive(M, x0, x1, t0);
            if (o1 == o2 && o2 == o3) {
                exit_f = f;
                ++nexit;
            }
        }
        if (nexit != 1) return resolve_exhaustive(M, x0, x1, t0);
        int4 nb = M.tnbr[t];
        int32_t code = nth(nb, exit_f);
        if (code <= -2) return Resolved{-2 - code, -1, 0, 0, 0};  // surface triangle crossed first
        if (code == -1) return Resolved{-1, -1, 0, 0, 0};         // left through an open face
        int4 back = M.tnbr[code];
        entry = -1;
        for (int g = 0; g < 4; ++g)
            if (nth(back, g) == t) entry = g;
        t = code;
    }
    return resolve_exhaustive(M, x0, x1, t0);
}

// ---------------------------------------------------------------------------
// barycentric map and charge
// ---------------------------------------------------------------------------
// FP64 atomic adds with the address space stated: a pointer that reaches the
// add through a struct is generic to the compiler, which then emits a FLAT
// atomic (slower, and for LDS it waits on both memory counters).
typedef __attribute__((address_space(3))) double lds_f64;
typedef __attribute__((address_space(1))) double global_f64;
__device__ inline void lds_add_f64(double* p, double v)
{
    __hip_atomic_fetch_add((lds_f64*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);  // ds_add_f64
}
__device__ inline void global_add_f64(double* p, double v)
{
    __hip_atomic_fetch_add((global_f64*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // global_atomic_add_f64
}

__device__ inline void scatter4(double* __restrict__ node_charge, const int4& nv, double q, const double lam[4])
{
    global_add_f64(&node_charge[nv.x], q * lam[0]);
    global_add_f64(&node_charge[nv.y], q * lam[1]);
    global_add_f64(&node_charge[nv.z], q * lam[2]);
    global_add_f64(&node_charge[nv.w], q * lam[3]);
}

// Block-local reduction of the charge scatter: contributions to the same node
// from the block's particles are summed in an LDS hash table (open addressing,
// linear probing) and flushed with one FP64 atomic per distinct node.  With
// particles sorted by tet a 256-particle block touches ~100-150 nodes instead
// of issuing 1,024 global atomics.
template <int Bits>
__device__ inline uint32_t hash_slot(int32_t node)
{
    return ((uint32_t)node * 2654435761u) >> (32 - Bits);
}

// The probes after the first, for a node whose first slot holds another one.
// A rolled loop: unrolled 32-fold at every insertion it was three quarters of
// the kernel's 17,000 instructions, and its nested branches spilled about
// 2,000 SGPRs.
template <int Bits>
__device__ inline void lds_charge_probe(int32_t* hk, double* hv, double* __restrict__ node_charge, int32_t node,
                                        uint32_t h, double val)
{
#pragma unroll 1
    for (int probe = 1; probe < 32; ++probe) {
        h = (h + 1) & ((1u << Bits) - 1u);
        const int32_t prev = atomicCAS(&hk[h], -1, node);
        if (prev == -1 || prev == node) {
            lds_add_f64(&hv[h], val);
            return;
        }
    }
    global_add_f64(&node_charge[node], val);  // crowded table: straight to memory
}

// The four contributions of one tet.  Node window (Win > 0): a block's
// tet-sorted particles touch nodes within a few thousand ids of the lowest one
// (the node numbering of a structured mesh puts a cell's nodes one layer,
// (nx+1)(ny+1) ids, apart), so nodes in [wbase, wbase + Win) are summed in a
// plain LDS array without the hash's compare-and-swap; the others go to the
// hash.  The four compare-and-swaps are issued together (their results are a
// full LDS latency away) and only a node that finds its first slot taken
// probes on.  base: offset of the run's node-charge array (0 for a single
// simulation).
template <int Bits, int Win>
__device__ inline void lds_scatter4(int32_t* hk, double* hv, double* wv, int32_t wbase,
                                    double* __restrict__ node_charge, const int4& nv, int32_t base,
                                    const double val[4])
{
    const int32_t node[4] = {base + nv.x, base + nv.y, base + nv.z, base + nv.w};
    bool todo[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        todo[q] = true;
        if (Win > 0) {
            const uint32_t off = (uint32_t)(node[q] - wbase);
            if (off < (uint32_t)Win) {
                lds_add_f64(&wv[off], val[q]);
                todo[q] = false;
            }
        }
    }
    if (Win > 0 && !(todo[0] || todo[1] || todo[2] || todo[3])) return;
    uint32_t h[4];
    int32_t prev[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        h[q] = hash_slot<Bits>(node[q]);
        prev[q] = node[q];
        if (Win == 0 || todo[q]) prev[q] = atomicCAS(&hk[h[q]], -1, node[q]);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const bool here = prev[q] == -1 || prev[q] == node[q];
        if (here && (Win == 0 || todo[q])) lds_add_f64(&hv[h[q]], val[q]);
        todo[q] = !here;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (todo[q]) lds_charge_probe<Bits>(hk, hv, node_charge, node[q], h[q], val[q]);
}

// ---------------------------------------------------------------------------
// per-thread tet cache and the two arithmetic layouts
//   FP64:  position absolute (double), map = v0 + A (double), E (double)
//   mixed: position relative to v0 of the owning tet (float), map A (float),
//          E (float); absolute coordinates are v0 (double) + local
// ---------------------------------------------------------------------------
// lazily loaded pieces of the owning tet's record (keeps registers free across
// the collision code)
__device__ inline void load_E(const DevMesh& M, int32_t t, double& ex, double& ey, double& ez)
{
    const double* E = M.E + 3 * (int64_t)t;
    ex = E[0];
    ey = E[1];
    ez = E[2];
}
__device__ inline void load_E(const DevMesh& M, int32_t t, float& ex, float& ey, float& ez)
{
    float4 e = reinterpret_cast<const float4*>(M.E32)[t];
    ex = e.x;
    ey = e.y;
    ez = e.z;
}
__device__ inline void load_E1(const DevMesh& M, int32_t t, double& ex, double& ey, double& ez)
{
    const double* E = M.E1 + 3 * (int64_t)t;
    ex = E[0];
    ey = E[1];
    ez = E[2];
}
__device__ inline void load_E1(const DevMesh& M, int32_t t, float& ex, float& ey, float& ez)
{
    float4 e = reinterpret_cast<const float4*>(M.E1_32)[t];
    ex = e.x;
    ey = e.y;
    ez = e.z;
}
// field of the particle's run in tet t: s0 * E_0 + s1 * E_1 (s0 = 1 and no
// second basis for a single simulation, where this is E_0 exactly)
template <typename R, bool kBatch>
__device__ inline void run_field(const DevMesh& M, const RunK* __restrict__ rk, int32_t t, R& ex, R& ey, R& ez)
{
    load_E(M, t, ex, ey, ez);
    if (!kBatch) return;
    const R s0 = (R)rk->s0;
    ex = s0 * ex;
    ey = s0 * ey;
    ez = s0 * ez;
    if (M.E1) {
        R fx, fy, fz;
        load_E1(M, t, fx, fy, fz);
        const R s1 = (R)rk->s1;
        ex = ex + s1 * fx;
        ey = ey + s1 * fy;
        ez = ez + s1 * fz;
    }
}
// push increment of tet t for the species in table `slot`
__device__ inline void load_push(const DevMesh& M, int slot, int32_t t, double& hx, double& hy, double& hz)
{
    const double* h = M.H + 3 * ((int64_t)slot * M.n_tets + t);
    hx = h[0];
    hy = h[1];
    hz = h[2];
}
__device__ inline void load_push(const DevMesh& M, int slot, int32_t t, float& hx, float& hy, float& hz)
{
    const float4 h = reinterpret_cast<const float4*>(M.H32)[(int64_t)slot * M.n_tets + t];
    hx = h.x;
    hy = h.y;
    hz = h.z;
}
__device__ inline void bary_at(const DevMesh& M, int32_t t, double x, double y, double z, double lam[4])
{
    bary64(M.geo + 12 * (int64_t)t, x, y, z, lam);
}
__device__ inline void bary_at(const DevMesh& M, int32_t t, float x, float y, float z, double lam[4])
{
    const float4* a = reinterpret_cast<const float4*>(M.geo32) + 3 * (int64_t)t;
    float4 a0 = a[0], a1 = a[1], a2 = a[2];
    float l1 = (a0.x * x + a0.y * y) + a0.z * z;
    float l2 = (a0.w * x + a1.x * y) + a1.y * z;
    float l3 = (a1.z * x + a1.w * y) + a2.x * z;
    float l0 = 1.0f - ((l1 + l2) + l3);
    lam[0] = l0;
    lam[1] = l1;
    lam[2] = l2;
    lam[3] = l3;
}
// bbox test of the frozen rule on the stored position
__device__ inline bool in_bbox_at(const DevMesh& M, const StepParams& S, int32_t t, double x, double y, double z)
{
    return (x >= S.lo[0]) & (x <= S.hi[0]) & (y >= S.lo[1]) & (y <= S.hi[1]) & (z >= S.lo[2]) & (z <= S.hi[2]);
}
__device__ inline bool in_bbox_at(const DevMesh& M, const StepParams& S, int32_t t, float x, float y, float z)
{
    float ax = x, ay = y, az = z;
    if (t >= 0) {
        float4 a2 = (reinterpret_cast<const float4*>(M.geo32) + 3 * (int64_t)t)[2];
        ax += a2.y;
        ay += a2.z;
        az += a2.w;
    }
    return (ax >= (float)S.lo[0]) & (ax <= (float)S.hi[0]) & (ay >= (float)S.lo[1]) & (ay <= (float)S.hi[1]) &
           (az >= (float)S.lo[2]) & (az <= (float)S.hi[2]);
}

template <typename R>
__device__ inline double tau_of(const DevMesh& M);
template <>
__device__ inline double tau_of<double>(const DevMesh& M) { return M.tau; }
template <>
__device__ inline double tau_of<float>(const DevMesh& M) { return (double)M.tau32; }

__device__ inline void v0_of(const DevMesh& M, int32_t t, double* v0)
{
    const double* g = M.geo + 12 * (int64_t)t;
    v0[0] = g[0];
    v0[1] = g[1];
    v0[2] = g[2];
}

// absolute position of a stored state
__device__ inline void abs_pos(const DevMesh& M, int32_t t, double x, double y, double z, double* p)
{
    p[0] = x;
    p[1] = y;
    p[2] = z;
}
__device__ inline void abs_pos(const DevMesh& M, int32_t t, float x, float y, float z, double* p)
{
    double v0[3] = {0.0, 0.0, 0.0};
    if (t >= 0) v0_of(M, t, v0);
    p[0] = v0[0] + (double)x;
    p[1] = v0[1] + (double)y;
    p[2] = v0[2] + (double)z;
}

// store an absolute position in the frame of tet t
__device__ inline void to_frame(const DevMesh& M, int32_t t, const double* p, double& x, double& y, double& z)
{
    x = p[0];
    y = p[1];
    z = p[2];
}
__device__ inline void to_frame(const DevMesh& M, int32_t t, const double* p, float& x, float& y, float& z)
{
    double v0[3] = {0.0, 0.0, 0.0};
    if (t >= 0) v0_of(M, t, v0);
    x = (float)(p[0] - v0[0]);
    y = (float)(p[1] - v0[1]);
    z = (float)(p[2] - v0[2]);
}

// ---------------------------------------------------------------------------
// charge sinks: LDS hash (streaming kernel) or direct atomics (rare paths)
// ---------------------------------------------------------------------------
template <int Bits, int Win>
struct LdsSink {
    int32_t* hk;
    double* hv;
    double* wv;
    int32_t wbase;
    double* nc;
    __device__ void add4(const int4& nv, int32_t base, const double val[4])
    {
        lds_scatter4<Bits, Win>(hk, hv, wv, wbase, nc, nv, base, val);
    }
};
struct GlobalSink {
    double* nc;
    __device__ void add4(const int4& nv, int32_t base, const double val[4])
    {
        scatter4(nc + base, nv, 1.0, val);
    }
};
// Per-particle accumulation across the steps of a launch: while the particle
// stays in one tet the charge weights lambda are summed in four registers; the
// sums, times the particle's charge q, go to the inner sink only when it
// changes tet or the launch ends.  base is the offset of the particle's run in
// the node-charge buffer; t < 0 or q = 0: nothing is scattered.
template <typename Inner>
struct RegSink {
    Inner inner;
    double a0, a1, a2, a3;
    __device__ void add(double w, const double lam[4])
    {
        a0 = __builtin_fma(w, lam[0], a0);
        a1 = __builtin_fma(w, lam[1], a1);
        a2 = __builtin_fma(w, lam[2], a2);
        a3 = __builtin_fma(w, lam[3], a3);
    }
    __device__ void flush(const DevMesh& M, int32_t t, int32_t base, double q)
    {
        if (t >= 0 && q != 0.0) flush_nodes(M.tnode[t], base, q);
        a0 = a1 = a2 = a3 = 0.0;
    }
    __device__ void flush_nodes(const int4& nv, int32_t base, double q)
    {
        const double v[4] = {q * a0, q * a1, q * a2, q * a3};
        inner.add4(nv, base, v);
        a0 = a1 = a2 = a3 = 0.0;
    }
    // The flush at the end of a tile, where every lane of the wavefront is
    // active: lanes of one run of equal (tet, run offset) -- neighbours in the
    // tet-sorted order -- sum their four weights into the run's first lane
    // (segmented Hillis-Steele over the wavefront), which alone goes to the
    // inner sink.  One LDS insertion per run instead of one per particle; per
    // 2^kRounds particles of a run with fewer rounds, which single steps of a
    // batch take (its runs are short: 109 -> 107 us with 4 of them).
    template <int kRounds = 6>
    __device__ void flush_wave(const DevMesh& M, int32_t cur, int32_t base, double q)
    {
        if (q == 0.0) cur = -1;
        a0 *= q;
        a1 *= q;
        a2 *= q;
        a3 *= q;
        const int lane = threadIdx.x & 63;
        const int32_t up_t = __shfl_up(cur, 1), up_b = __shfl_up(base, 1);
        const bool head = lane == 0 || up_t != cur || up_b != base;
        const unsigned long long hm = __ballot(head);
        const int seg = __popcll(hm & (~0ull >> (63 - lane)));  // runs starting at or below this lane
#pragma unroll
        for (int d = 1; d < 1 << kRounds; d <<= 1) {
            const int sd = __shfl_down(seg, d);
            const double b0 = __shfl_down(a0, d), b1 = __shfl_down(a1, d), b2 = __shfl_down(a2, d),
                         b3 = __shfl_down(a3, d);
            if (lane + d < 64 && sd == seg) {
                a0 += b0;
                a1 += b1;
                a2 += b2;
                a3 += b3;
            }
        }
        const int start = 63 - __builtin_clzll(hm & (~0ull >> (63 - lane)));
        if (((lane - start) & ((1 << kRounds) - 1)) != 0) cur = -1;
        flush(M, cur, base, 1.0);
    }
    // flush_wave with the node window of an LDS sink, when no charge has gone
    // to LDS yet in this tile (single-step launches): the window starts at the
    // lowest node the tile's runs touch (a block minimum, s_wbase preset to
    // INT32_MAX); called by every thread of the workgroup.  The segmented sum
    // runs two rounds (shifts 1 and 2): lane i then holds the sum of lanes
    // i..i+3 of its run, and the lanes 0, 4, 8, ... after the start of their
    // run insert, so every lane is counted once.  With about one particle per
    // tet, runs longer than four are rare; the full six rounds cost more
    // cross-lane moves than the inserts they save (measured: 63.5 against
    // 65.8 us per single-step FP64 launch on the large box).
    __device__ void flush_wave_window(const DevMesh& M, int32_t cur, int32_t base, double q, int32_t* s_wbase)
    {
        if (q == 0.0) cur = -1;
        a0 *= q;
        a1 *= q;
        a2 *= q;
        a3 *= q;
        const int lane = threadIdx.x & 63;
        const int32_t up_t = __shfl_up(cur, 1), up_b = __shfl_up(base, 1);
        const bool head = lane == 0 || up_t != cur || up_b != base;
        const unsigned long long hm = __ballot(head);
        const int seg = __popcll(hm & (~0ull >> (63 - lane)));
        const unsigned long long below = hm & (~0ull >> (63 - lane));
        const int start = 63 - __builtin_clzll(below);
#pragma unroll
        for (int d = 1; d < 4; d <<= 1) {
            const int sd = __shfl_down(seg, d);
            const double b0 = __shfl_down(a0, d), b1 = __shfl_down(a1, d), b2 = __shfl_down(a2, d),
                         b3 = __shfl_down(a3, d);
            if (lane + d < 64 && sd == seg) {
                a0 += b0;
                a1 += b1;
                a2 += b2;
                a3 += b3;
            }
        }
        if (((lane - start) & 3) != 0) cur = -1;
        int4 nv = make_int4(0, 0, 0, 0);
        int32_t lo = INT32_MAX;
        if (cur >= 0) {
            nv = M.tnode[cur];
            lo = base + min(min(nv.x, nv.y), min(nv.z, nv.w));
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) lo = min(lo, __shfl_xor(lo, off));
        if (lane == 0) atomicMin(s_wbase, lo);
        __syncthreads();
        inner.wbase = __builtin_amdgcn_readfirstlane(*s_wbase);
        if (cur >= 0) {
            const double v[4] = {a0, a1, a2, a3};
            inner.add4(nv, base, v);
        }
    }
};

// Collision decision u1 < P (HSModel.cpp:15-19, VHSModel.cpp:60-70).  For
// VHS/VSS the FP64 probability needs pow() every step; an FP32 estimate with a
// relative error far below 1e-4 decides all draws outside a +-1e-4 band
// around it, and only draws inside the band evaluate the FP64 expression, so
// the FP64 decision is reproduced exactly at FP32 cost.
__device__ __noinline__ bool collides_exact64(int model, double sigma_hs, double vhs_c, double two_kt, double m_r,
                                              double vhs_exp, double conc, double dt, double vm, double u1)
{
    CollideK<double> ck{sigma_hs, vhs_c, two_kt, m_r, vhs_exp, 0.0, 0.0, 0.0};
    return u1 < collision_probability<double>(model, ck, conc, dt, vm);
}

template <typename R>
__device__ inline bool collides(int model, double dt, const SpeciesK& k, double conc, R vx, R vy, R vz, double u1)
{
    R vm = m_sqrt<R>(vx * vx + vy * vy + vz * vz);
    if (model == 1) {  // HS: no transcendental, evaluate directly
        CollideK<R> ck{(R)k.sigma_hs, (R)0, (R)0, (R)0, (R)0, (R)0, (R)0, (R)0};
        return (R)u1 < collision_probability<R>(1, ck, (R)conc, (R)dt, vm);
    }
    float vmf = (float)vm;
    CollideK<float> cf{(float)k.sigma_hs, (float)k.vhs_c, (float)k.two_kt, (float)k.m_r, (float)k.vhs_exp,
                       0.0f, 0.0f, 0.0f};
    float p32 = collision_probability<float>(model, cf, (float)conc, (float)dt, vmf);
    if (!std::is_same<R, double>::value) return (float)u1 < p32;
    double p = (double)p32;
    if (!(p > 1e-30 && p < 1e30))  // outside the range the FP32 bound covers
        return collides_exact64(model, k.sigma_hs, k.vhs_c, k.two_kt, k.m_r, k.vhs_exp, conc, dt, (double)vm, u1);
    if (u1 < p * (1.0 - 1e-4)) return true;
    if (u1 >= p * (1.0 + 1e-4)) return false;
    return collides_exact64(model, k.sigma_hs, k.vhs_c, k.two_kt, k.m_r, k.vhs_exp, conc, dt, (double)vm, u1);
}

// The collision of one step for the few draws may_collide() lets through
// (about once per 1e3-1e4 particle-steps): the decision, then the
// post-collision velocity; unchanged if there is none.  Out of line to keep
// the streaming kernel lean; the variates are drawn here so that few of the
// caller's registers are live at the call; arguments and result by value so
// nothing of the caller escapes to memory.  The scattering is FP64 in both
// precisions: evaluated in FP32, sin(chi) = sqrt((1 - cos)(1 + cos)) of a
// forward scatter (cos near 1 from an FP64 variate rounded to FP32) loses most
// of its digits.
struct V3 {
    double x, y, z;
};
template <typename R>
__device__ __noinline__ V3 collide_step(int model, double dt, const SpeciesK* k, double conc, uint64_t seed,
                                        uint32_t key, uint32_t vid, uint32_t step, double vx, double vy, double vz)
{
    double u1, u2, u3;
    variates(seed, key, vid, step, 0u, u1, u2);
    if (collides<R>(model, dt, *k, conc, (R)vx, (R)vy, (R)vz, u1)) {
        variates(seed, key, vid, step, 1u, u2, u3);
        scatter_velocity(model, k->mass_cp, k->mass_ct, k->inv_alpha, u2, u3, vx, vy, vz);
    }
    return V3{vx, vy, vz};
}

// Whether the collision test u1 < P of a step can pass, from the first variate
// word w0 alone (u1 >= w0 2^-32) and an FP32 estimate of P in the log domain:
// log2(P 2^32) = ca + cb log2(|v|^2), ca from the host's FP64 constants
// (species, gas, time step; +inf where one of them is outside the range the
// FP32 bound covers) plus 32 and log2(1.001).  The exponents stay below 200 in
// magnitude, so ca, the product and the sum err by less than 5e-5 and v_log /
// v_exp by an ulp: 1e-4 relative in P, a tenth of the margin.  "false" is
// certain; "true" (P itself, and one draw in a thousand beyond it) goes to
// collide_step, which decides as the reference does.  This replaces an FP32
// pow, two square roots and the second variate word in every step.
template <typename R>
__device__ inline bool may_collide(uint32_t w0, float ca, float cb, R v2)
{
    const float v2f = (float)v2;
    const float p = __builtin_amdgcn_exp2f(ca + cb * __builtin_amdgcn_logf(v2f));
    // (below 1e-6 the FP32 probability of the mixed path leaves its range)
    return !((float)w0 > p && (std::is_same<R, double>::value || v2f > 1e-6f));
}

// Barycentric classification with a certified threshold: strictly inside,
// strictly outside exactly one face (strictly inside the other three), or
// uncertain.  tau bounds the rounding of lambda at points within 2 diam of v0
// (diam: largest vertex coordinate difference).  Since x - v0 = sum_j
// lambda_j (v_j - v0), |x - v0|_inf <= diam * sum |lambda_j|, so the
// classification is only trusted when sum |lambda| <= 2: a long step that
// ends far outside the tet is left to the exact walk.
enum { kInside = 0, kOneFace = 1, kUncertain = 2 };
__device__ inline int classify(const double lam[4], double tau, int& fneg)
{
    int npos = 0, nneg = 0;
    fneg = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        npos += lam[q] > tau;
        if (lam[q] < -tau) {
            ++nneg;
            fneg = q;
        }
    }
    if (fabs(lam[0]) + fabs(lam[1]) + fabs(lam[2]) + fabs(lam[3]) > 2.0) return kUncertain;
    if (npos == 4) return kInside;
    if (npos == 3 && nneg == 1) return kOneFace;
    return kUncertain;
}

// Certified walk of the segment p0 -> p1 (absolute FP64, p0 strictly inside
// t) through as many tets as it crosses, with the FP64 barycentric maps, for
// steps longer than a tet.  In each tet the exit face is the face f with
// lambda_f(p1) < 0 whose plane the segment meets first: s_f = l0_f / (l0_f -
// l1_f) is smallest, i.e. D_fg = l0_f l1_g - l0_g l1_f > 0 for every other
// such g.  Signs and orderings are trusted only beyond their rounding bound:
// lambda at a point with sum|lambda| = S errs by at most tau * max(1, S/2)
// (tau covers S <= 2 and the bound is linear in |x - v0| <= diam * S).  The
// entry point lies inside a face (all other lambdas > 0), so the exit point
// found this way lies inside the exit face.  Anything closer than the bounds
// (edges, vertices, end points near a face) is left to the exact walk.
enum { kWalkInside = 0, kWalkSurface = 1, kWalkOpen = 2, kWalkUnsure = 3 };
constexpr int kWalkHops = 16;

// The face of a tet through which the segment p0 -> p1 leaves it: l1 the
// coordinates of p1 with their bound t1, l0() those of p0 (only needed when p1
// lies beyond several faces).  kInHere: p1 is inside; kNoFace: not certain.
enum { kInHere = -1, kNoFace = -2 };
template <typename L0>
__device__ inline int exit_face(double tau, const double l1[4], L0 l0_of)
{
    constexpr double kE = 1.1102230246251565e-16;  // 2^-53
    const double t1 = walk_tol(tau, l1);
    int nneg = 0, npos = 0, f1 = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        npos += l1[q] > t1;
        if (l1[q] < -t1) {
            ++nneg;
            f1 = q;
        }
    }
    if (npos + nneg < 4) return kNoFace;  // p1 too close to a face plane
    if (nneg == 0) return kInHere;
    if (nneg == 1) return f1;
    double l0[4];
    l0_of(l0);
    const double t0 = walk_tol(tau, l0);
    int exit_f = kNoFace;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        bool first = l1[f] < -t1;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (g == f) continue;
            const double a = l0[f] * l1[g], b = l0[g] * l1[f];
            const double err = t0 * (fabs(l1[f]) + fabs(l1[g]) + 2.0 * t1) +
                               t1 * (fabs(l0[f]) + fabs(l0[g]) + 2.0 * t0) + 4.0 * kE * (fabs(a) + fabs(b));
            first = first && (!(l1[g] < -t1) || a - b > err);
        }
        if (first && exit_f == kNoFace) exit_f = f;
    }
    return exit_f;
}

__device__ inline int walk64(const DevMesh& M, int32_t t, const double* p0, const double* p1, int32_t& out)
{
    int32_t cur = t;
#pragma unroll 1
    for (int hop = 0; hop < kWalkHops; ++hop) {
        double l1[4];
        bary_at(M, cur, p1[0], p1[1], p1[2], l1);
        const int f = exit_face(M.tau, l1, [&](double* l0) { bary_at(M, cur, p0[0], p0[1], p0[2], l0); });
        if (f == kNoFace) return kWalkUnsure;
        if (f == kInHere) {
            out = cur;
            return kWalkInside;
        }
        const int32_t code = nth(M.tnbr[cur], f);
        if (code <= -2) {
            out = -2 - code;
            return kWalkSurface;
        }
        if (code == -1) return kWalkOpen;
        cur = code;
    }
    return kWalkUnsure;
}

constexpr int32_t kDeferredLane = -1;  // a lane's flags once its particle has deferred
enum StepOutcome { kDone = 0, kSettledNow = 1, kDeferNow = 2, kFrozenNow = 3 };

// settle record for the adjoint
__device__ inline void record_settle(SettleRec* rec, uint32_t pidx, uint32_t step, double x0, double y0,
                                           double z0)
{
    SettleRec r;
    r.x0 = x0;
    r.y0 = y0;
    r.z0 = z0;
    r.step = (int32_t)step;
    r.pad = 0;
    rec[pidx] = r;
}

// Where the segment xa -> xa + D meets the plane of triangle `tri`:
// xa + s D with s = n.(A - xa) / n.D, n = (B - A) x (C - A).
__device__ inline void hit_plane(const DevMesh& M, int32_t tri, const double* xa, const double* D, double* n,
                                 double& s)
{
    double A[3], B[3], C[3];
    load_node(M, M.tris[3 * (int64_t)tri], A);
    load_node(M, M.tris[3 * (int64_t)tri + 1], B);
    load_node(M, M.tris[3 * (int64_t)tri + 2], C);
    double u[3] = {B[0] - A[0], B[1] - A[1], B[2] - A[2]};
    double w[3] = {C[0] - A[0], C[1] - A[1], C[2] - A[2]};
    n[0] = u[1] * w[2] - u[2] * w[1];
    n[1] = u[2] * w[0] - u[0] * w[2];
    n[2] = u[0] * w[1] - u[1] * w[0];
    double nD = (n[0] * D[0] + n[1] * D[1]) + n[2] * D[2];
    double nA = (n[0] * (A[0] - xa[0]) + n[1] * (A[1] - xa[1])) + n[2] * (A[2] - xa[2]);
    s = nA / nD;
}

// Movement records of the tracked particles (ParticleMovementTracker.cpp:4-16):
// one absolute point appended to the slot of load index li, if it has one.
// Points beyond the slot's capacity are counted, not stored.  One thread owns
// a slot at a time (the particle's lane in the step kernels), so no atomics.
// The callers test S.trk_slot (kernel-uniform) and look the slot up here, so
// that with recording off no register is held across the step loop.
__device__ __noinline__ void track_point(const int32_t* slot_of, int32_t* cnt, double* xyz, int32_t max_pts,
                                         uint32_t li, double x, double y, double z)
{
    const int32_t slot = slot_of[li];
    if (slot < 0) return;
    const int32_t c = cnt[slot];
    if (c < max_pts) {
        double* q = xyz + 3 * ((int64_t)slot * max_pts + c);
        q[0] = x;
        q[1] = y;
        q[2] = z;
    }
    cnt[slot] = c + 1;
}

// the position at the start of a step (recorded after the push, before the
// move: ParticleDynamicsProcessor.cpp:182-184)
template <typename R>
__device__ __forceinline__ void track_start(const DevMesh& M, const StepParams& S, uint32_t li, int32_t t, R x, R y,
                                            R z)
{
    double a[3];
    abs_pos(M, t, x, y, z, a);
    track_point(S.trk_slot, S.trk_count, S.trk_xyz, S.trk_max, li, a[0], a[1], a[2]);
}

// the point where the settling segment xa -> (x1 in the frame of t) meets its
// triangle (ParticleSurfaceCollisionHandler.cpp:91-99, :134-138)
template <typename R>
__device__ __forceinline__ void track_hit(const DevMesh& M, const StepParams& S, uint32_t li, const double* xa,
                                          int32_t t, R x1, R y1, R z1, int32_t tri)
{
    double b[3], D[3], n[3], s;
    abs_pos(M, t, x1, y1, z1, b);
    for (int k = 0; k < 3; ++k) D[k] = b[k] - xa[k];
    hit_plane(M, tri, xa, D, n, s);
    track_point(S.trk_slot, S.trk_count, S.trk_xyz, S.trk_max, li, xa[0] + s * D[0], xa[1] + s * D[1],
                xa[2] + s * D[2]);
}

// position in R (FP32 in the owner's frame in mixed mode), velocity FP64:
// accumulated in FP32, a per-tet increment much smaller than |v| rounds the
// same way step after step, and the velocity drifts linearly (about 6e-8 of
// |v| per step).  v2 = |v|^2 in R, kept with the velocity.
template <typename R>
struct PState {
    R x, y, z;
    double vx, vy, vz;
    R v2;
    int32_t t, f;
    __device__ void set_v2()
    {
        const R a = (R)vx, b = (R)vy, c = (R)vz;
        v2 = a * a + b * b + c * c;
    }
};

// sqrt(v2) < 10 without the root: the root is correctly rounded, so it is
// below 10 exactly for v2 below the smallest number whose root rounds to 10.
__device__ inline bool too_slow(double v2) { return v2 < 0x1.8ffffffffffffp+6; }
__device__ inline bool too_slow(float v2) { return v2 < 0x1.8ffffep+6f; }

// What stays the same over a particle's steps of a launch.
struct PConst {
    const SpeciesK* k;
    const RunK* rk;
    uint32_t vid;   // variate counter
    uint32_t key;   // the run's part of the variate key
    float ca, cb;   // may_collide
};
__device__ inline PConst particle_const(const StepParams& S, const SpeciesK* k, const RunK* rk, uint32_t vid)
{
    return PConst{k, rk, vid, rk->key, k->coll_a + rk->log2_conc + S.log2_dt, k->coll_b};
}

// face codes and nodes of a particle's tet; of a lane whose particle deferred,
// the deferred step
struct Deferral {
    double x0[3];
    int32_t t0, k;
};
union TetRows {
    struct {
        int4 nbr, node;
    };
    Deferral deferral;
};

// The record of one tet as a particle's step uses it: the barycentric map
// (FP64: v0 and A; mixed: A) and the push increment h of the particle in it.
template <typename R>
struct TetRec {
    static constexpr int kLen = std::is_same<R, double>::value ? 12 : 9;
    int32_t t;  // -1: nothing loaded
    R g[kLen];
    R hx, hy, hz;

    // The record of tet (-1: none).  rows: null, or where the tet's face codes
    // and nodes go (LDS; a lane that leaves the tet then needs no load before
    // that of the next tet's record).
    template <bool kBatch>
    __device__ inline void load(const DevMesh& M, const StepParams& S, const SpeciesK& k,
                                const RunK* __restrict__ rk, int32_t tet, TetRows* rows = nullptr)
    {
        if (tet >= 0) {
            load_in<kBatch>(M, S, k, rk, tet, rows);
        } else {  // outside the mesh: no push, and no point is certified inside
            t = tet;
#pragma unroll
            for (int q = 0; q < kLen; ++q) g[q] = R(0);
            hx = hy = hz = R(-0.0);
        }
    }
    template <bool kBatch>
    __device__ inline void load_in(const DevMesh& M, const StepParams& S, const SpeciesK& k,
                                   const RunK* __restrict__ rk, int32_t tet, TetRows* rows = nullptr)
    {
        t = tet;
        if constexpr (std::is_same<R, double>::value) {
            const double* p = M.geo + 12 * (int64_t)tet;
#pragma unroll
            for (int q = 0; q < 12; ++q) g[q] = p[q];
        } else {
            const float4* a = reinterpret_cast<const float4*>(M.geo32) + 3 * (int64_t)tet;
            const float4 a0 = a[0], a1 = a[1];
            g[0] = a0.x;
            g[1] = a0.y;
            g[2] = a0.z;
            g[3] = a0.w;
            g[4] = a1.x;
            g[5] = a1.y;
            g[6] = a1.z;
            g[7] = a1.w;
            g[8] = a[2].x;
        }
        if (rows) {
            rows->nbr = M.tnbr[tet];
            rows->node = M.tnode[tet];
        }
        load_h<kBatch>(M, S, k, rk, tet);
    }
    // h = (((E*q)/m)*dt)/2 (Particle.cpp:199-207); -0 where the push is skipped,
    // which leaves (v + h) + h = v bit for bit.  From the table of the species,
    // or evaluated here with the same operations: per lane once per tet it
    // enters, not once per step (three FP64 divisions).
    template <bool kBatch>
    __device__ inline void load_h(const DevMesh& M, const StepParams& S, const SpeciesK& k,
                                  const RunK* __restrict__ rk, int32_t tet)
    {
        if (!kBatch && S.em_push && k.push_slot >= 0) {
            load_push(M, k.push_slot, tet, hx, hy, hz);
            return;
        }
        const R dt = (R)S.dt, qc = (R)k.charge, m = (R)k.mass;
        R ex, ey, ez;
        run_field<R, kBatch>(M, rk, tet, ex, ey, ez);
        const bool push = S.em_push && dt != R(0) && !(ex == R(0) && ey == R(0) && ez == R(0));
        ex = ex * qc;
        ey = ey * qc;
        ez = ez * qc;
        if (kBatch || k.push_slot != -2) {  // (charge 0 in a single simulation: the signed zero E*q)
            ex = ((ex / m) * dt) / R(2);
            ey = ((ey / m) * dt) / R(2);
            ez = ((ez / m) * dt) / R(2);
        }
        hx = push ? ex : R(-0.0);
        hy = push ? ey : R(-0.0);
        hz = push ? ez : R(-0.0);
    }
    __device__ inline void bary(R x, R y, R z, double lam[4]) const
    {
        if constexpr (std::is_same<R, double>::value) {
            bary64(g, x, y, z, lam);
        } else {
            const float l1 = (g[0] * x + g[1] * y) + g[2] * z;
            const float l2 = (g[3] * x + g[4] * y) + g[5] * z;
            const float l3 = (g[6] * x + g[7] * y) + g[8] * z;
            const float l0 = 1.0f - ((l1 + l2) + l3);
            lam[0] = l0;
            lam[1] = l1;
            lam[2] = l2;
            lam[3] = l3;
        }
    }
};

// Where a step's end point went (relocate): the position in its owner's frame,
// the owner, the outcome, the triangle hit, and its coordinates in the owner.
struct Lam {
    double l[4];
};
template <typename R>
struct Relocated {
    R x, y, z;
    int32_t t;
    int32_t outcome;
    int32_t hit_tri;
    Lam lam;
};
// Relocation of a step whose end point x1 is not certified inside the owner t
// by its coordinates `l` there: faces, neighbours, the multi-tet walk.  x0
// strictly inside t.  Certified cases: x1 strictly inside the owner (by the
// FP64 map), or strictly outside exactly one face f and strictly inside the
// other three (the segment leaves through the open face f), or the walk's;
// the rest (kDeferNow, x1 in the frame of t) needs the exact walk.
// vneg: sign bits of the velocity (mixed only).
template <typename R, bool kWalk>
__device__ inline Relocated<R> relocate(const DevMesh& M, int32_t t, int32_t vneg, R x0, R y0, R z0, R x1, R y1,
                                              R z1, Lam l)
{
    const double tau = tau_of<R>(M);
    int fneg = 0;
    int cls = classify(l.l, tau, fneg);
    if (!std::is_same<R, double>::value && cls == kUncertain) {
        // FP32 too close to a face: certify with the FP64 map at the FP64
        // absolute position of the stored FP32 state
        double p1[3];
        abs_pos(M, t, x1, y1, z1, p1);
        bary_at(M, t, p1[0], p1[1], p1[2], l.l);
        cls = classify(l.l, M.tau, fneg);
    }
    if (cls == kInside) return Relocated<R>{x1, y1, z1, t, kDone, -1, l};
    if (cls == kOneFace) {
        const int32_t code = nth(M.tnbr[t], fneg);
        if (code <= -2) return Relocated<R>{x1, y1, z1, t, kSettledNow, -2 - code};  // crosses this triangle first
        // to the neighbour (or out through a face with no triangle)
        double p1[3];
        abs_pos(M, t, x1, y1, z1, p1);
        R nx, ny, nz;
        to_frame(M, code, p1, nx, ny, nz);
        if (code == -1) return Relocated<R>{nx, ny, nz, -1, kDone, -1};
        bary_at(M, code, nx, ny, nz, l.l);
        int f2;
        int c2 = classify(l.l, tau, f2);
        if (!std::is_same<R, double>::value && c2 == kUncertain) {
            double q[3];
            abs_pos(M, code, nx, ny, nz, q);
            bary_at(M, code, q[0], q[1], q[2], l.l);
            c2 = classify(l.l, M.tau, f2);
        }
        if (c2 == kInside) return Relocated<R>{nx, ny, nz, code, kDone, -1, l};
    }
    if (kWalk) {
        // a segment through several tets: the certified FP64 walk
        double p0[3], p1[3];
        abs_pos(M, t, x0, y0, z0, p0);
        abs_pos(M, t, x1, y1, z1, p1);
        int32_t where = -1;
        int w = walk64(M, t, p0, p1, where);
        if (!std::is_same<R, double>::value && w == kWalkUnsure) {
            // FP32 end points lie on a lattice (~1e-9 m apart in a 1 cm tet),
            // and about 1e-7 of them land exactly on a face plane (one through
            // v0, e.g. local x == y).  Such a point is moved by 1, 2 and 3 FP32
            // ulps along the step in x, y and z (unequal, so that it leaves
            // planes like x == y, which an equal move would keep it on) -- within
            // the FP32 state's own rounding -- and certified again; a point that
            // stays uncertain goes to the exact walk as before.
            const R ux = (vneg & 1) ? R(-INFINITY) : R(INFINITY);
            const R uy = (vneg & 2) ? R(-INFINITY) : R(INFINITY);
            const R uz = (vneg & 4) ? R(-INFINITY) : R(INFINITY);
            x1 = m_nextafter(x1, ux);
            y1 = m_nextafter(m_nextafter(y1, uy), uy);
            z1 = m_nextafter(m_nextafter(m_nextafter(z1, uz), uz), uz);
            abs_pos(M, t, x1, y1, z1, p1);
            w = walk64(M, t, p0, p1, where);
        }
        if (w == kWalkSurface) {
            return Relocated<R>{x1, y1, z1, t, kSettledNow, where};  // crosses this surface triangle first
        }
        if (w != kWalkUnsure) {
            R nx, ny, nz;
            to_frame(M, w == kWalkOpen ? -1 : where, p1, nx, ny, nz);
            if (w == kWalkOpen) return Relocated<R>{nx, ny, nz, -1, kDone, -1};
            // the position as stored (FP32 in its owner's frame in mixed mode)
            // must itself be strictly inside the owner the walk found
            bary_at(M, where, nx, ny, nz, l.l);
            int f2;
            int c2 = classify(l.l, tau, f2);
            if (!std::is_same<R, double>::value && c2 == kUncertain) {
                double q[3];
                abs_pos(M, where, nx, ny, nz, q);
                bary_at(M, where, q[0], q[1], q[2], l.l);
                c2 = classify(l.l, M.tau, f2);
            }
            if (!std::is_same<R, double>::value) {
                // Rounding the end point to FP32 in the new frame can put the
                // stored point (not the segment's end) just beyond a face of
                // `where`; it is then owned by the neighbour across that face,
                // where it is stored rounded in that neighbour's frame.
                for (int tries = 0; tries < 2 && c2 == kOneFace; ++tries) {
                    const int32_t code = nth(M.tnbr[where], f2);
                    if (code < 0) break;  // a surface or open face: the exact walk decides
                    double q[3];
                    abs_pos(M, where, nx, ny, nz, q);
                    where = code;
                    to_frame(M, where, q, nx, ny, nz);
                    bary_at(M, where, nx, ny, nz, l.l);
                    c2 = classify(l.l, tau, f2);
                    if (c2 == kUncertain) {
                        abs_pos(M, where, nx, ny, nz, q);
                        bary_at(M, where, q[0], q[1], q[2], l.l);
                        c2 = classify(l.l, M.tau, f2);
                    }
                }
            }
            if (c2 == kInside) return Relocated<R>{nx, ny, nz, where, kDone, -1, l};
        }
    }
    return Relocated<R>{x1, y1, z1, t, kDeferNow, -1};
}

// Frozen this step and every later one of the launch (nothing changes its
// state; it still carries charge): 2. |v| < 10 m/s or 3. outside the expanded
// bbox (ParticleDynamicsProcessor.cpp:166-176).  Where the expanded bbox holds
// every node, a finite point in a tet is inside it.
template <typename R>
__device__ inline bool frozen_finite(const DevMesh& M, const StepParams& S, const PState<R>& s)
{
    return too_slow(s.v2) || ((s.t < 0 || !S.bbox_covers) && !in_bbox_at(M, S, s.t, s.x, s.y, s.z));
}
// A NaN or infinite point, which the exact predicates can give an owner, is
// outside the bbox.  The common step does without this test: such a point ends
// its step nowhere certain, and comes here with the rare ones.
template <typename R>
__device__ inline bool not_finite(const PState<R>& s)
{
    return !((s.x - s.x) + (s.y - s.y) + (s.z - s.z) == R(0));
}
template <typename R>
__device__ inline bool is_frozen(const DevMesh& M, const StepParams& S, const PState<R>& s)
{
    return frozen_finite(M, S, s) || not_finite(s);
}

// 4. push with the owning tet's field (ParticleDynamicsProcessor.cpp:179-180);
// rec: the owner's record.
template <typename R>
__device__ inline void push_in(PState<R>& s, const TetRec<R>& rec)
{
    s.vx = (s.vx + (double)rec.hx) + (double)rec.hx;
    s.vy = (s.vy + (double)rec.hy) + (double)rec.hy;
    s.vz = (s.vz + (double)rec.hz) + (double)rec.hz;
    s.set_v2();
}

// 6. move (Particle.cpp:157-165): the end point in the owner's frame.  Mixed:
// rounded to FP32 stochastically, with 30 hashed bits of (particle, step, seed).
template <typename R>
__device__ inline void end_point(const StepParams& S, uint32_t vid, uint32_t key, uint32_t step, const PState<R>& s,
                                 R& x1, R& y1, R& z1)
{
    if constexpr (std::is_same<R, double>::value) {
        x1 = s.x + s.vx * S.dt;
        y1 = s.y + s.vy * S.dt;
        z1 = s.z + s.vz * S.dt;
    } else {
        const uint32_t h = hash3(vid, step, (uint32_t)S.seed ^ key);
        x1 = round_stochastic((double)s.x + s.vx * S.dt, h & 0x3ffu);
        y1 = round_stochastic((double)s.y + s.vy * S.dt, (h >> 10) & 0x3ffu);
        z1 = round_stochastic((double)s.z + s.vz * S.dt, h >> 22);
    }
}

// 7. gas collision (ParticlePhysicsUpdater.cpp:20-24) of a draw that may collide
template <typename R>
__device__ inline void collide(const StepParams& S, const PConst& c, uint32_t step, PState<R>& s)
{
    const V3 nv = collide_step<R>(S.model, S.dt, c.k, c.rk->conc, S.seed, c.key, c.vid, step, s.vx, s.vy, s.vz);
    s.vx = nv.x;
    s.vy = nv.y;
    s.vz = nv.z;
    s.set_v2();
}

// Outside the mesh: a segment wholly beyond one face of the nodes' bounding box
// meets no tet and no surface triangle (exact compares).
template <typename R>
__device__ inline bool stays_outside(const DevMesh& M, const PState<R>& s, R x1, R y1, R z1)
{
    const double p0[3] = {(double)s.x, (double)s.y, (double)s.z}, p1[3] = {(double)x1, (double)y1, (double)z1};
    bool away = false;
#pragma unroll
    for (int q = 0; q < 3; ++q)
        away = away || (p0[q] < M.node_lo[q] && p1[q] < M.node_lo[q]) ||
               (p0[q] > M.node_hi[q] && p1[q] > M.node_hi[q]);
    return away;
}

// 8. relocation and surface hit on the segment from the state's position to x1.
// Leaves the state at the end point (kDeferNow: in the frame of the unchanged
// owner; the caller resolves it exactly) and, for kDone with an owner, the end
// point's coordinates in lam.
template <typename R, bool kWalk>
__device__ inline int move_to(const DevMesh& M, PState<R>& s, bool strict, R x1, R y1, R z1, Lam& lam,
                              int32_t& hit_tri)
{
    if (s.t >= 0 && strict) {
        const int32_t vneg = (s.vx < 0.0 ? 1 : 0) | (s.vy < 0.0 ? 2 : 0) | (s.vz < 0.0 ? 4 : 0);
        const Relocated<R> r = relocate<R, kWalk>(M, s.t, vneg, s.x, s.y, s.z, x1, y1, z1, lam);
        s.x = r.x;
        s.y = r.y;
        s.z = r.z;
        s.t = r.t;
        lam = r.lam;
        hit_tri = r.hit_tri;
        return r.outcome;
    }
    const int outcome = s.t < 0 && stays_outside(M, s, x1, y1, z1) ? kDone : kDeferNow;
    s.x = x1;
    s.y = y1;
    s.z = z1;
    return outcome;
}

// The common step of a particle strictly inside its tet (rec: the tet's
// record), as step_tile takes it: pushed, moved and still inside, with no
// collision to look at.  False, and nothing done, in any other case.  For the
// straggler kernel, where a particle's steps are one serial chain: 390 -> 263
// us for the rest of 200 steps.
template <typename R, typename Sink>
__device__ inline bool plain_step(const DevMesh& M, const StepParams& S, const PConst& c, uint32_t step, PState<R>& s,
                                  const TetRec<R>& rec, Sink& sink)
{
    if (frozen_finite(M, S, s)) return false;
    PState<R> n = s;
    push_in(n, rec);
    R x1, y1, z1;
    end_point(S, c.vid, c.key, step, n, x1, y1, z1);
    if (S.model != 0 && may_collide<R>(variate_word(S.seed, c.key, c.vid, step), c.ca, c.cb, n.v2)) return false;
    Lam lam;
    rec.bary(x1, y1, z1, lam.l);
    const double tau = tau_of<R>(M);
    if (!(lam.l[0] > tau && lam.l[1] > tau && lam.l[2] > tau && lam.l[3] > tau)) return false;
    s = n;
    s.x = x1;
    s.y = y1;
    s.z = z1;
    sink.add(1.0, lam.l);
    return true;
}

// One step of one particle (ParticleDynamicsProcessor.cpp:166-199 stage order,
// then the relocation and charge of the next gather), as the straggler kernel
// takes it; step_tile runs the same stages with the common case first.
template <typename R, bool kBatch, bool kWalk, typename Sink>
__device__ inline int step_one(const DevMesh& M, const StepParams& S, const PConst& c, uint32_t step, int remaining,
                               PState<R>& s, TetRec<R>& rec, Sink& sink, int32_t& hit_tri)
{
    Lam lam;
    if (is_frozen(M, S, s)) {
        if (s.t >= 0) {
            bary_at(M, s.t, s.x, s.y, s.z, lam.l);
            sink.add((double)remaining, lam.l);
        }
        return kFrozenNow;
    }
    if (s.t >= 0) {
        if (s.t != rec.t) rec.template load<kBatch>(M, S, *c.k, c.rk, s.t);
        push_in(s, rec);
    }
    R x1, y1, z1;
    end_point(S, c.vid, c.key, step, s, x1, y1, z1);
    const bool still = x1 == s.x && y1 == s.y && z1 == s.z;  // degenerate segment (:188-190)
    if (!still && S.model != 0 && may_collide<R>(variate_word(S.seed, c.key, c.vid, step), c.ca, c.cb, s.v2))
        collide(S, c, step, s);
    int outcome = kDone;
    if (s.t >= 0) rec.bary(x1, y1, z1, lam.l);
    const int32_t t_before = s.t;
    if (!still) {
        outcome = move_to<R, kWalk>(M, s, (s.f & kStrict) != 0, x1, y1, z1, lam, hit_tri);
        if (s.t < 0) s.f &= ~kStrict;
    }
    if (s.t != t_before) sink.flush(M, S.charge ? t_before : -1, (int32_t)c.rk->node_base, c.k->charge);
    if (outcome == kDone && s.t >= 0) sink.add(1.0, lam.l);
    return outcome;
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
__global__ void prologue_kernel(double* __restrict__ a, double* __restrict__ b, int64_t n_nodes)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t j = i; j < n_nodes; j += stride) {
        a[j] = 0.0;
        if (b) b[j] = 0.0;
    }
}

// Arguments of the streaming kernels.
template <typename R>
struct StepArgs {
    DevMesh M;
    DevParticles<R> P;
    StepParams S;
    const SpeciesK* sp;
    double* node_charge;
    WorkItem* wl;
    unsigned long long* cnt;
    unsigned long long* tri_count;
};
// To the work list: one atomic for the lanes that come together.
template <typename R>
__device__ inline void append_work(const StepArgs<R>& A, uint32_t row, const Deferral& d)
{
    const unsigned long long dm = __ballot(true);
    const int lane = __lane_id();
    const int leader = __ffsll((long long)dm) - 1;
    unsigned int slot = 0u;
    if (lane == leader)
        slot = (unsigned int)atomicAdd(&A.cnt[kCntWork + 2 * A.S.work_slot], (unsigned long long)__popcll(dm));
    slot = __shfl(slot, leader);
    WorkItem it;
    it.x0 = d.x0[0];
    it.y0 = d.x0[1];
    it.z0 = d.x0[2];
    it.i = (int32_t)row;
    it.t0 = d.t0;
    it.k = d.k;
    it.pad = 0;
    A.wl[slot + (unsigned)__popcll(dm & ((1ull << lane) - 1ull))] = it;
}

// A particle that settled (flags, hit, counters, records) or deferred (to
// `stage`, for the work list at the end of the tile, or to the list itself) in a
// step from px, py, pz in tet t_before; s: its state after it, which the caller
// has stored.
template <typename R, bool kTrack>
__device__ inline void finish_rare(const StepArgs<R>& A, int outcome, uint32_t row, uint32_t li, const RunK* rk,
                                   const PState<R>& s, int32_t t_before, R px, R py, R pz, uint32_t step, int32_t ks,
                                   int32_t hit_tri, TetRows* stage)
{
    const StepParams& S = A.S;
    if (outcome == kSettledNow) {
        A.P.flags[row] = (s.f | kSettled) & ~kStrict;
        A.P.hit[row] = hit_tri;
        atomicAdd(&A.tri_count[rk->tri_base + hit_tri], 1ull);
        S.settle_log[atomicAdd(&A.cnt[kCntSettled], 1ull)] = li;
        if (S.settle || kTrack) {
            double a[3];
            abs_pos(A.M, t_before, px, py, pz, a);
            if (S.settle) record_settle(S.settle, li, step, a[0], a[1], a[2]);
            if (kTrack) track_hit<R>(A.M, S, li, a, s.t, s.x, s.y, s.z, hit_tri);
        }
        return;
    }
    Deferral d;
    abs_pos(A.M, t_before, px, py, pz, d.x0);
    d.t0 = t_before;
    d.k = ks;
    if (stage) stage->deferral = d;
    else append_work(A, row, d);
}

// What a rare step left: the owner, the outcome, and the charge weights lam,
// to be counted `weight` times in t.
struct RareStep {
    Lam lam;
    int32_t t;
    int32_t outcome;
    int32_t weight;
};

// Step ks of the launch for the lanes with `go` whose step is not the streaming
// loop's common case: frozen particles, collisions, segments the loop does not
// certify, surface hits.  The particle's state is in memory, before the step,
// and is left there after it: nothing of the caller's is live here but the
// charge sums, so that the walk's and the scattering's temporaries have the
// registers.  (With the state kept in registers across it, parts of the loop's
// own values went to scratch memory, which is 100 MB over the chip and misses
// the L2: up to 11 ms for 200 steps of 1M particles.  Called out of line
// it was slower too, for the calling convention's saves.)
template <typename R, bool kBatch, bool kWalk, bool kTrack, bool kPlain>
__device__ __forceinline__ RareStep rare_step(const StepArgs<R>& A, uint32_t row, uint32_t step, int32_t ks, int32_t remaining,
                                           bool go, TetRows* stage)
{
    RareStep r{{{0.0, 0.0, 0.0, 0.0}}, -1, kDone, 0};
    if (!go) return r;
    const DevMesh& M = A.M;
    const StepParams& S = A.S;
    const DevParticles<R>& P = A.P;
    PState<R> s;
    s.f = P.flags[row];
    s.t = P.tet[row];
    s.x = P.x[row];
    s.y = P.y[row];
    s.z = P.z[row];
    s.vx = P.vx[row];
    s.vy = P.vy[row];
    s.vz = P.vz[row];
    s.set_v2();
    const SpeciesK& k = A.sp[(s.f >> kSpeciesShift) & 0xff];
    const RunK* rk = kBatch ? S.runs + ((uint32_t)s.f >> kRunShift) : S.runs;
    const uint32_t li = P.pidx[row];
    r.t = s.t;
    if (is_frozen(M, S, s)) {
        if (s.t >= 0) {
            bary_at(M, s.t, s.x, s.y, s.z, r.lam.l);
            r.weight = remaining;
        }
        r.outcome = kFrozenNow;
        return r;
    }
    const PConst c = particle_const(S, &k, rk, li - rk->first);
    const R px = s.x, py = s.y, pz = s.z;
    const int32_t t_before = s.t;
    int32_t hit_tri = -1;
    R x1, y1, z1;
    {
        TetRec<R> rec;
        rec.template load<kBatch>(M, S, k, rk, s.t);
        push_in(s, rec);
        end_point(S, c.vid, c.key, step, s, x1, y1, z1);
        rec.bary(x1, y1, z1, r.lam.l);
    }
    if (kTrack) track_start<R>(M, S, li, t_before, px, py, pz);
    if (!(x1 == px && y1 == py && z1 == pz)) {  // (a degenerate segment ends here, :188-190)
        if (!kPlain && S.model != 0 && may_collide<R>(variate_word(S.seed, c.key, c.vid, step), c.ca, c.cb, s.v2))
            collide(S, c, step, s);
        r.outcome = move_to<R, kWalk>(M, s, (s.f & kStrict) != 0, x1, y1, z1, r.lam, hit_tri);
    }
    r.t = s.t;
    r.weight = r.outcome == kDone && s.t >= 0 ? 1 : 0;
    P.x[row] = s.x;
    P.y[row] = s.y;
    P.z[row] = s.z;
    P.vx[row] = s.vx;
    P.vy[row] = s.vy;
    P.vz[row] = s.vz;
    if (s.t != t_before) P.tet[row] = s.t;
    if (s.t < 0 && t_before >= 0) P.flags[row] = s.f & ~kStrict;
    if (r.outcome != kDone)
        finish_rare<R, kTrack>(A, r.outcome, row, li, rk, s, t_before, px, py, pz, step, ks, hit_tri, stage);
    return r;
}

// Mixed layout: a stored point that FP32 cannot place inside tet t, by the FP64
// map (lam: its coordinates then).
__device__ inline bool inside64(const DevMesh& M, int32_t t, float x, float y, float z, double* lam)
{
    double q[3], l[4];
    abs_pos(M, t, x, y, z, q);
    bary_at(M, t, q[0], q[1], q[2], l);
    const bool in = l[0] > M.tau && l[1] > M.tau && l[2] > M.tau && l[3] > M.tau;
    if (in)
        for (int k = 0; k < 4; ++k) lam[k] = l[k];
    return in;
}
__device__ inline bool inside64(const DevMesh&, int32_t, double, double, double, double*) { return false; }

// One tile of the streaming kernel: BS consecutive particles, one per thread,
// S.nsteps steps with the state and the owning tet's record in registers.  A
// particle whose relocation cannot be certified stops and goes to the work
// list with the step it stopped at.  Called with a block-uniform tile.
// kTrack: movement records on (S.trk_slot set), a kernel variant of its own so
// that the streaming kernels without them carry none of their code.
// What bounds a fused launch is the issue and latency of its instructions: a
// step is about 140 vector instructions (mixed 210), against 525 when every
// step read the record again, took an FP32 pow and two square roots for the
// collision test and ran through the code of the rare cases.  200 steps of 1M
// particles on 750k tets with their read-back, FP64: 3.31 -> 1.00 ms; of 16
// runs of 1e4 to 4e5 particles on 162k tets, mixed: 6.37 -> 2.42 ms.  Where one lane of nearly every wave
// changes tet in every step the latency of the next record bounds it and the
// gain is smaller: 200 steps of 16M particles on 3M tets, FP64 2.0e10 -> 2.6e10
// particle-steps/s, mixed 1.71e10 -> 1.77e10.
// 3 waves per SIMD (168 registers): 4 waves put values of the loop into
// scratch memory (1.47 ms), 2 waves hide too little of it (1.36 ms).
// kPlain: neither charge nor gas, without the charge sums, the hash and the
// collision test in the loop's registers.  Ions between plates, where lanes
// change tet all the time, 1,000 steps in launches of 50: 131,072 particles
// 2,750 -> 2,210 us, 262,144 (4,096 waves, a quarter of which waits for a
// second round) 4,150 -> 3,590 us; at 4 waves per SIMD 3,780 us.
template <typename R, int BS, int HashBits, bool kBatch, bool kWalk, bool kTrack, bool kPlain>
__device__ __forceinline__ void step_tile(const StepArgs<R>& A, int64_t tile, int64_t n_active, uint32_t step0,
                                          unsigned int* blk_processed, int32_t* hk, double* hv, TetRows* s_rows)
{
    constexpr int kSlots = 1 << HashBits;
    const DevMesh& M = A.M;
    const StepParams& S = A.S;
    const bool has_charge = !kPlain && S.charge;
    const DevParticles<R>& P = A.P;
    if (threadIdx.x == 0) *blk_processed = 0u;
    if (has_charge) {
        for (int h = threadIdx.x; h < kSlots; h += BS) {
            hk[h] = -1;
            hv[h] = 0.0;
        }
    }
    __syncthreads();
    // the tile's part of every array from a block-uniform base and the lane's
    // 32-bit offset: no per-lane 64-bit address outlives its load or store
    const int64_t i0 = tile * BS;
    const int tid = threadIdx.x;
    RegSink<LdsSink<HashBits, 0>> sink{LdsSink<HashBits, 0>{hk, hv, nullptr, 0, A.node_charge}, 0.0, 0.0, 0.0, 0.0};
    // A lane is alive while its particle has steps to take.  A lane without a
    // particle, or whose particle is done (frozen, settled, deferred: its state
    // is in memory), goes through the arithmetic of the others; nothing of it
    // is used.
    PState<R> s;
    s.f = kSettled;
    s.t = -1;
    s.x = s.y = s.z = R(0);
    s.vx = s.vy = s.vz = 0.0;
    auto read_state = [&]() {
        s.t = (P.tet + i0)[tid];
        s.x = (P.x + i0)[tid];
        s.y = (P.y + i0)[tid];
        s.z = (P.z + i0)[tid];
        s.vx = (P.vx + i0)[tid];
        s.vy = (P.vy + i0)[tid];
        s.vz = (P.vz + i0)[tid];
    };
    int32_t t_mem = -1;  // the owner in memory (the loop only moves a particle from tet to tet)
    auto write_state = [&]() {
        (P.x + i0)[tid] = s.x;
        (P.y + i0)[tid] = s.y;
        (P.z + i0)[tid] = s.z;
        (P.vx + i0)[tid] = s.vx;
        (P.vy + i0)[tid] = s.vy;
        (P.vz + i0)[tid] = s.vz;
        if (s.t != t_mem) (P.tet + i0)[tid] = s.t;
    };
    uint32_t vid = 0;
    if (i0 + tid < n_active) {
        s.f = (P.flags + i0)[tid];
        vid = (P.pidx + i0)[tid];
        read_state();
    }
    bool alive = !(s.f & kSettled);
    if (!alive) s.t = -1;
    const SpeciesK& k = A.sp[alive ? (s.f >> kSpeciesShift) & 0xff : 0];
    // one simulation: run 0 for every lane (scalar loads); a batch: the lane's run
    const RunK* rk = kBatch ? S.runs + (alive ? (uint32_t)s.f >> kRunShift : 0u) : S.runs;
    vid -= rk->first;
    const bool strict = (s.f & kStrict) != 0;  // (a particle that leaves the mesh is told by its tet)
    t_mem = s.t;
    s.set_v2();
    TetRec<R> rec;
    TetRows* const rows = s_rows + tid;
    rec.template load<kBatch>(M, S, k, rk, s.t, rows);
    const PConst pc = particle_const(S, &k, rk, vid);
    const int32_t base = kBatch ? (int32_t)rk->node_base : 0;
    const double charge = k.charge;
    const double tau = tau_of<R>(M);
    const int nsteps = S.nsteps;
    int ks = 0;
    while (ks < nsteps && __ballot(alive) != 0) {
        // The common case, alone in its loop: steps in which every live
        // particle of the wavefront stays strictly inside its tet (all four
        // coordinates of the end point above tau; their sum of magnitudes is
        // then 1) with no collision to look at.  The loop is uniform and the
        // common case touches no memory, so the state and the tet's record
        // stay in registers.  A lane that collides, crosses into a tet where it
        // is certified, meets a surface or flies on outside the mesh is handled
        // in place; a step with any other case in any lane leaves the loop.
        // Collisions in place matter in longer steps: at dt 5e-8 and 0.3 Pa a
        // third of the waves has one in every step, and sent through memory
        // they took 16M particles on 3M tets to 1.54e10 particle-steps/s
        // mixed, 2.29e10 FP64, against 1.75e10 and 2.64e10 here (1.71e10 and
        // 2.00e10 with four waves per SIMD and every case in the loop).
        bool rare;
        for (;;) {
            const uint32_t step = step0 + (uint32_t)ks;
            const int32_t t0 = s.t;
            rare = too_slow(s.v2);
            if (!S.bbox_covers) rare = rare || !in_bbox_at(M, S, s.t, s.x, s.y, s.z);
            PState<R> n = s;
            R x1, y1, z1;
            push_in(n, rec);
            end_point(S, pc.vid, pc.key, step, n, x1, y1, z1);
            bool draw = !kPlain && S.model != 0;
            if (draw) draw = may_collide<R>(variate_word(S.seed, pc.key, pc.vid, step), pc.ca, pc.cb, n.v2);
            Lam lam;
            rec.bary(x1, y1, z1, lam.l);
            bool inside = strict && lam.l[0] > tau && lam.l[1] > tau && lam.l[2] > tau && lam.l[3] > tau;
            bool settles = false, defers = false;
            if (__ballot(alive && (rare || draw || !inside)) != 0) {
                if (__ballot(alive && draw && !rare) != 0) {
                    // (a degenerate segment ends before the collision, :188-190)
                    if (alive && draw && !rare && !(x1 == s.x && y1 == s.y && z1 == s.z)) collide(S, pc, step, n);
                }
                if (alive && !rare && !inside) {
                    if (s.t < 0) {
                        inside = in_bbox_at(M, S, s.t, s.x, s.y, s.z) && stays_outside(M, s, x1, y1, z1);
                    } else if (strict) {
                        // From tet to tet along the segment.  (Mixed: one hop in
                        // FP32, further ones through the FP64 maps.)
                        constexpr bool kFar = kWalk && std::is_same<R, double>::value;
                        int fneg = 0;
                        int f = kFar ? exit_face(tau, lam.l, [&](double* l0) { rec.bary(s.x, s.y, s.z, l0); })
                                     : (classify(lam.l, tau, fneg) == kOneFace ? fneg : (int)kNoFace);
                        const bool one_face = f >= 0;
                        if (f < 0) inside = inside64(M, s.t, x1, y1, z1, lam.l);
                        if (f >= 0) {
                            int32_t code = (&rows->nbr.x)[f];
                            if (has_charge && charge != 0.0) sink.flush_nodes(rows->node, base, charge);
                            R nx = x1, ny = y1, nz = z1;
                            if constexpr (!std::is_same<R, double>::value) {
                                double p1[3];
                                abs_pos(M, s.t, x1, y1, z1, p1);
                                to_frame(M, code, p1, nx, ny, nz);
                            }
#pragma unroll 1
                            for (int hop = 0; code >= 0 && hop < (kFar ? 6 : 1); ++hop) {
                                rec.template load_in<kBatch>(M, S, k, rk, code, rows);
                                rec.bary(nx, ny, nz, lam.l);
                                if ((lam.l[0] > tau && lam.l[1] > tau && lam.l[2] > tau && lam.l[3] > tau) ||
                                    inside64(M, code, nx, ny, nz, lam.l)) {
                                    inside = true;
                                    break;
                                }
                                f = kNoFace;
                                if constexpr (kFar)
                                    f = exit_face(tau, lam.l, [&](double* l0) { rec.bary(s.x, s.y, s.z, l0); });
                                if (f < 0) break;
                                code = (&rows->nbr.x)[f];
                            }
                            if (inside) {
                                s.t = code;
                                x1 = nx;
                                y1 = ny;
                                z1 = nz;
                            } else if (f >= 0 && code <= -2) {
                                settles = true;  // on triangle -2 - code
                                s.f = code;
                            }
                        }
                        if constexpr (!kWalk) {
                            // Deferred, as relocate() has it: what is neither
                            // certified nor an exit through an open face (f is
                            // then still that face).  Without the walk most
                            // long segments are (10 steps of 1M particles, dt
                            // 1e-6 in 1 cm tets: 942 -> 499 us against
                            // rare_step).
                            const bool known = std::is_same<R, double>::value || one_face;
                            if (!inside && !settles && f < 0 && known && !(x1 == s.x && y1 == s.y && z1 == s.z)) {
                                defers = true;
                                if (!one_face && has_charge && charge != 0.0) sink.flush_nodes(rows->node, base, charge);
                            }
                        }
                        if constexpr (kWalk && !std::is_same<R, double>::value) {
                            // Where steps are a tenth of a tet, half the waves
                            // have a lane beyond two faces, and on a curved mesh
                            // many points FP32 cannot place.  Both left to
                            // rare_step, 16M particles on 3M tets ran at 1.15e10
                            // particle-steps/s, so at 1.54e10 (collisions still
                            // in rare_step in both).
                            if (!inside && !settles) {
                                if (f < 0 && has_charge && charge != 0.0) sink.flush_nodes(rows->node, base, charge);
                                double p0[3], p1[3];
                                abs_pos(M, s.t, s.x, s.y, s.z, p0);
                                abs_pos(M, s.t, x1, y1, z1, p1);
                                int32_t where = -1;
                                const int w = walk64(M, s.t, p0, p1, where);
                                if (w == kWalkSurface) {
                                    settles = true;
                                    s.f = -2 - where;
                                } else if (w == kWalkInside) {
                                    R nx, ny, nz;
                                    to_frame(M, where, p1, nx, ny, nz);
                                    rec.template load_in<kBatch>(M, S, k, rk, where, rows);
                                    rec.bary(nx, ny, nz, lam.l);
                                    if ((lam.l[0] > tau && lam.l[1] > tau && lam.l[2] > tau && lam.l[3] > tau) ||
                                        inside64(M, where, nx, ny, nz, lam.l)) {
                                        inside = true;
                                        s.t = where;
                                        x1 = nx;
                                        y1 = ny;
                                        z1 = nz;
                                    }
                                }
                            }
                        }
                    }
                }
                rare = rare || !inside;
            }
            if (kTrack && alive && (!rare || settles || defers)) track_start<R>(M, S, vid + rk->first, t0, s.x, s.y, s.z);
            if (__builtin_expect(__ballot(settles || defers) != 0, 0)) {
                if (settles || defers) {
                    const R px = s.x, py = s.y, pz = s.z;
                    const int32_t tri = settles ? -2 - s.f : -1;
                    s.f = (P.flags + i0)[tid];
                    s.x = x1;  // in the frame of the owner it leaves
                    s.y = y1;
                    s.z = z1;
                    s.vx = n.vx;
                    s.vy = n.vy;
                    s.vz = n.vz;
                    write_state();
                    finish_rare<R, kTrack>(A, settles ? kSettledNow : kDeferNow, (uint32_t)(i0 + tid), vid + rk->first,
                                           rk, s, t0, px, py, pz, step, ks, tri, rows);
                    atomicAdd(blk_processed, (unsigned int)ks + 1u);
                    alive = false;
                    if (defers) s.f = kDeferredLane;
                    s.t = -1;
                    rec.template load<kBatch>(M, S, k, rk, -1, rows);
                }
                if constexpr (!kWalk) {
                    if (__ballot(alive) == 0) {  // a wave can defer as a whole
                        ks = nsteps;
                        break;
                    }
                }
            }
            if (!rare) {
                s.x = x1;
                s.y = y1;
                s.z = z1;
                s.vx = n.vx;
                s.vy = n.vy;
                s.vz = n.vz;
                s.v2 = n.v2;
                if (!kPlain) {
                    sink.a0 += lam.l[0];
                    sink.a1 += lam.l[1];
                    sink.a2 += lam.l[2];
                    sink.a3 += lam.l[3];
                }
            }
            rare = rare && alive;
            if (__ballot(rare) != 0) break;
            if (++ks == nsteps) break;
        }
        if (ks == nsteps) break;
        // A step that is rare in some lanes (the others have taken it): every
        // lane's state goes through memory.
        if (alive) write_state();
        const int32_t t_before = s.t;
        const RareStep r = rare_step<R, kBatch, kWalk, kTrack, kPlain>(
            A, (uint32_t)(i0 + tid), step0 + (uint32_t)ks, ks,
            nsteps - ks, rare, rows);
        asm volatile("" ::: "memory");
        if (rare) {
            const bool done = r.outcome != kDone;
            if (has_charge && t_before >= 0 && (done || r.t != t_before)) {
                if (r.outcome == kFrozenNow) sink.add((double)r.weight, r.lam.l);
                sink.flush(M, t_before, base, charge);
            }
            if (!kPlain && !done) sink.add((double)r.weight, r.lam.l);
            if (done) {
                const unsigned int taken = (unsigned int)ks + (r.outcome == kFrozenNow ? 0u : 1u);
                if (taken) atomicAdd(blk_processed, taken);
                alive = false;
                if (r.outcome == kDeferNow) s.f = kDeferredLane;
            }
            s.t = done ? -1 : r.t;
        }
        t_mem = s.t;
        if (alive) read_state();
        s.set_v2();
        rec.template load<kBatch>(M, S, k, rk, s.t, rows);
        ++ks;
    }
    if (alive) write_state();
    // The particles that deferred, of all steps together: where most of them do
    // (10 steps of 1M particles, no walk), the wave's atomics in every step, all
    // to one address, took 1.0 of 1.95 ms.
    if (s.f == kDeferredLane) append_work(A, (uint32_t)(i0 + tid), rows->deferral);
    if (!alive) sink.a0 = sink.a1 = sink.a2 = sink.a3 = 0.0;  // flushed when it stopped
    if (has_charge) sink.flush_wave(M, s.t, base, charge);  // every lane is active here
    // processed particle-steps: LDS per block, one atomic per tile spread over slots
    const unsigned long long am = __ballot(alive);
    if ((threadIdx.x & 63) == 0 && am) atomicAdd(blk_processed, (unsigned int)__popcll(am) * (unsigned int)nsteps);
    __syncthreads();
    if (threadIdx.x == 0 && *blk_processed)
        atomicAdd(&A.cnt[kCntProcSlot0 + (tile & (kProcSlots - 1))], (unsigned long long)*blk_processed);
    if (has_charge) {
        for (int h = threadIdx.x; h < kSlots; h += BS) {
            int32_t node = hk[h];
            if (node >= 0) global_add_f64(&A.node_charge[node], hv[h]);
        }
    }
    __syncthreads();  // the LDS table and counter are reused by the next tile
}

// One tile of a single-step launch: each particle's step in registers from load
// to store.  All charge goes to LDS in the flush at the end of the tile: that of
// one simulation into a window of consecutive nodes (flush_wave_window), a
// batch's, whose runs are interleaved, into the hash.
// HBM and the charge atomics bound it: 219 B per particle-step, mixed 158.  1M particles
// on 750k tets: FP64 53.4 -> 52.6 us, mixed 57.8 -> 45.0 us; 4M particles FP64
// 211 -> 183 us.  4 workgroups per CU, no scratch memory; a fifth (half the
// hash, 96 registers) was slower, 55.5 and 193 us.
template <typename R, int BS, int HashBits, int Win, bool kBatch, bool kWalk, bool kTrack>
__device__ __forceinline__ void single_tile(const StepArgs<R>& A, int64_t tile, int64_t n_active, uint32_t step,
                                            unsigned int* blk_processed, int32_t* hk, double* hv, double* wv,
                                            int32_t* s_wbase)
{
    constexpr int kSlots = 1 << HashBits;
    const DevMesh& M = A.M;
    const StepParams& S = A.S;
    const DevParticles<R>& P = A.P;
    if (threadIdx.x == 0) {
        *blk_processed = 0u;
        *s_wbase = INT32_MAX;
    }
    if (S.charge) {
        for (int h = threadIdx.x; h < kSlots; h += BS) {
            hk[h] = -1;
            hv[h] = 0.0;
        }
        for (int h = threadIdx.x; h < Win; h += BS) wv[h] = 0.0;
    }
    __syncthreads();
    const int64_t i0 = tile * BS;
    const int tid = threadIdx.x;
    RegSink<LdsSink<HashBits, Win>> sink{LdsSink<HashBits, Win>{hk, hv, wv, INT32_MAX, A.node_charge}, 0.0, 0.0, 0.0,
                                         0.0};
    int32_t cur = -1;  // the tet the charge goes to
    double charge = 0.0;
    bool taken = false, rare = false, draw = false;
    PState<R> s;
    R x1 = R(0), y1 = R(0), z1 = R(0);
    Lam lam;
    lam.l[0] = lam.l[1] = lam.l[2] = lam.l[3] = 0.0;
    const SpeciesK* kp = A.sp;
    const RunK* rk = S.runs;
    uint32_t vid = 0;
    if (i0 + tid < n_active) {
        s.f = (P.flags + i0)[tid];
        s.t = (P.tet + i0)[tid];
        s.x = (P.x + i0)[tid];
        s.y = (P.y + i0)[tid];
        s.z = (P.z + i0)[tid];
        s.vx = (P.vx + i0)[tid];
        s.vy = (P.vy + i0)[tid];
        s.vz = (P.vz + i0)[tid];
        if (kBatch) rk = S.runs + ((uint32_t)s.f >> kRunShift);
        vid = (P.pidx + i0)[tid] - rk->first;
        if (!(s.f & kSettled)) {
            kp = A.sp + ((s.f >> kSpeciesShift) & 0xff);
            charge = kp->charge;
            s.set_v2();
            TetRec<R> rec;
            rec.template load<kBatch>(M, S, *kp, rk, s.t);
            if (frozen_finite(M, S, s)) {
                rec.bary(s.x, s.y, s.z, lam.l);
                cur = s.t;
            } else {
                taken = true;
                const PConst pc = particle_const(S, kp, rk, vid);
                const double tau = tau_of<R>(M);
                push_in(s, rec);
                end_point(S, vid, pc.key, step, s, x1, y1, z1);
                rec.bary(x1, y1, z1, lam.l);
                if (S.model != 0) draw = may_collide<R>(variate_word(S.seed, pc.key, vid, step), pc.ca, pc.cb, s.v2);
                rare = draw || !((s.f & kStrict) && lam.l[0] > tau && lam.l[1] > tau && lam.l[2] > tau &&
                                 lam.l[3] > tau);
                if (!rare) {
                    if (kTrack) track_start<R>(M, S, vid + rk->first, s.t, s.x, s.y, s.z);
                    (P.x + i0)[tid] = x1;
                    (P.y + i0)[tid] = y1;
                    (P.z + i0)[tid] = z1;
                    (P.vx + i0)[tid] = s.vx;
                    (P.vy + i0)[tid] = s.vy;
                    (P.vz + i0)[tid] = s.vz;
                    cur = s.t;
                }
            }
        }
    }
    // collisions and segments that leave the tet
    if (__ballot(rare) != 0) {
        if (rare && not_finite(s)) {  // frozen
            bary_at(M, s.t, s.x, s.y, s.z, lam.l);
            cur = s.t;
            taken = false;
        } else if (rare) {
            const int32_t t_in = s.t;
            const R px = s.x, py = s.y, pz = s.z;
            int outcome = kDone;
            int32_t hit_tri = -1;
            if (kTrack) track_start<R>(M, S, vid + rk->first, t_in, px, py, pz);
            if (!(x1 == px && y1 == py && z1 == pz)) {  // (a degenerate segment ends here, :188-190)
                if (draw) collide(S, PConst{kp, rk, vid, rk->key, 0.0f, 0.0f}, step, s);
                outcome = move_to<R, kWalk>(M, s, (s.f & kStrict) != 0, x1, y1, z1, lam, hit_tri);
            }
            const uint32_t row = (uint32_t)(i0 + tid);
            P.x[row] = s.x;
            P.y[row] = s.y;
            P.z[row] = s.z;
            P.vx[row] = s.vx;
            P.vy[row] = s.vy;
            P.vz[row] = s.vz;
            if (s.t != t_in) {
                P.tet[row] = s.t;
                if (s.t < 0) P.flags[row] = s.f & ~kStrict;
            }
            if (outcome == kDone) cur = s.t;
            else
                finish_rare<R, kTrack>(A, outcome, row, vid + rk->first, rk, s, t_in, px, py, pz, step, 0, hit_tri,
                                       nullptr);
        }
    }
    sink.a0 = lam.l[0];
    sink.a1 = lam.l[1];
    sink.a2 = lam.l[2];
    sink.a3 = lam.l[3];
    if (S.charge) {  // every lane is active here
        const int32_t base = kBatch ? (int32_t)rk->node_base : 0;
        if constexpr (Win > 0) sink.flush_wave_window(M, cur, base, charge, s_wbase);
        else sink.template flush_wave<2>(M, cur, base, charge);
    }
    const unsigned long long am = __ballot(taken);
    if ((threadIdx.x & 63) == 0 && am) atomicAdd(blk_processed, (unsigned int)__popcll(am));
    __syncthreads();
    if (threadIdx.x == 0 && *blk_processed)
        atomicAdd(&A.cnt[kCntProcSlot0 + (tile & (kProcSlots - 1))], (unsigned long long)*blk_processed);
    if (S.charge) {
        for (int h = threadIdx.x; h < kSlots; h += BS) {
            const int32_t node = hk[h];
            if (node >= 0) global_add_f64(&A.node_charge[node], hv[h]);
        }
        // window slots that received charge (untouched ones hold 0.0)
        const int32_t wbase = sink.inner.wbase;
        for (int h = threadIdx.x; h < Win; h += BS) {
            const double v = wv[h];
            if (v != 0.0) global_add_f64(&A.node_charge[wbase + h], v);
        }
    }
}

// Streaming kernel.  With persistent == 0 workgroup b takes tile b; otherwise
// a grid sized to the chip pulls tiles from a queue counter until the live
// prefix is covered (one launch for every run of a batch, whatever their
// sizes).  The charge of a tile is summed in LDS (node window and hash) and
// flushed with one FP64 atomic per distinct node.
template <typename R, int BS, bool kBatch, bool kPersistent, bool kWalk, bool kTrack = false, bool kSingle = false,
          bool kPlain = false>
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(kSingle ? 4 : 3))) step_main(StepArgs<R> A)
{
    const StepParams& S = A.S;
    unsigned long long* const cnt = A.cnt;
    // Single-step launches (256 threads) of one simulation: a 3,072-node window
    // (24 KB) and a 1,024-slot hash (12 KB), 36 KB in all, so that four
    // workgroups (the 16 waves the 128-VGPR budget allows) share a CU's 160 KB.
    // Otherwise the hash alone, 8 slots per thread: fused launches add to LDS
    // while they step, and batches interleave their runs in the tet order.  (The
    // window run fused was 5% slower on the 3M-tet chamber, whose node layers lie
    // 6,600 ids apart.)
    static_assert(!kSingle || (BS == 256 && !kPersistent), "single steps: 256 threads, a workgroup per tile");
    constexpr int kWin = kSingle && !kBatch ? 3072 : 0;
    constexpr int kBits = kWin > 0 ? 10 : (BS == 256 ? 11 : 10);
    __shared__ unsigned int blk_processed;
    __shared__ int64_t s_tile;
    __shared__ int32_t s_wbase;
    __shared__ int32_t hk[1 << kBits];
    __shared__ double hv[1 << kBits];
    __shared__ double wv[kWin > 0 ? kWin : 1];
    __shared__ TetRows s_rows[kSingle ? 1 : BS];
    const uint32_t step0 = (uint32_t)cnt[kCntStep + S.work_slot];
    {
        // clear the next launch's charge buffers and counters, and give it its first step
        int64_t g = blockIdx.x * (int64_t)BS + threadIdx.x;
        int64_t gs = (int64_t)gridDim.x * BS;
        if (S.zero_charge)
            for (int64_t j = g; j < S.charge_len; j += gs) S.zero_charge[j] = 0.0;
        if (g == 0) {
            cnt[kCntWork + 2 * (1 - S.work_slot)] = 0ull;
            cnt[kCntStep + (1 - S.work_slot)] = (unsigned long long)step0 + (unsigned long long)S.nsteps;
            cnt[kCntTile + (1 - S.work_slot)] = 0ull;
        }
    }
    // (an append that failed half-way can leave the count ahead of the rows)
    const int64_t n_active = min(*S.n_active, A.P.n);
    if (!kPersistent) {
        if ((int64_t)blockIdx.x * BS < n_active)  // else the whole block is past the live particles
        {
            if constexpr (kSingle)
                single_tile<R, BS, kBits, kWin, kBatch, kWalk, kTrack>(A, blockIdx.x, n_active, step0, &blk_processed,
                                                                       hk, hv, wv, &s_wbase);
            else
                step_tile<R, BS, kBits, kBatch, kWalk, kTrack, kPlain>(A, blockIdx.x, n_active, step0, &blk_processed,
                                                                       hk, hv, s_rows);
        }
        return;
    }
    for (;;) {
        if (threadIdx.x == 0) s_tile = (int64_t)atomicAdd(&cnt[kCntTile + S.work_slot], 1ull);
        __syncthreads();
        const int64_t tile = s_tile;
        if (tile * BS >= n_active) break;  // queue drained: every workgroup exits here
        step_tile<R, BS, kBits, kBatch, kWalk, kTrack, kPlain>(A, tile, n_active, step0, &blk_processed, hk, hv,
                                                               s_rows);
    }
}

// Exact relocation of a deferred step: the state holds x1 in the frame of the
// owner at the step start; x0abs is the absolute start.  Returns true when the
// particle settled.
template <typename R>
__device__ inline bool finish_exact(const DevMesh& M, const double* x0abs, PState<R>& s, int32_t& hit_tri, int& exh,
                                    int& err)
{
    double x1[3];
    abs_pos(M, s.t, s.x, s.y, s.z, x1);
    Resolved r = resolve(M, x0abs, x1, s.t, (s.f & kStrict) != 0);
    exh += r.exhaustive;
    err |= r.err;
    if (r.hit >= 0) {
        hit_tri = r.hit;
        return true;
    }
    to_frame(M, r.tet, x1, s.x, s.y, s.z);
    int strict = r.strict;
    if (!std::is_same<R, double>::value && r.tet >= 0) {
        // the stored (rounded) position decides the fast path next step
        double q[3];
        abs_pos(M, r.tet, s.x, s.y, s.z, q);
        strict = tet_contains(M, r.tet, q) == 2;
    }
    s.t = r.tet;
    s.f = strict ? (s.f | kStrict) : (s.f & ~kStrict);
    return false;
}
template <typename R, typename Sink>
__device__ inline void add_here(const DevMesh& M, const PState<R>& s, Sink& sink)
{
    if (s.t < 0) return;
    double lam[4];
    bary_at(M, s.t, s.x, s.y, s.z, lam);
    sink.add(1.0, lam);
}

// Straggler kernel: finishes each deferred relocation exactly, then runs the
// particle's remaining steps of the launch with the certified fast path,
// resolving exactly again whenever a step defers.  (Holding it to 128 VGPRs
// for 4 waves per SIMD spills ~300 registers and was slower than 1 wave.)
template <typename R, bool kWalk>
__global__ void __launch_bounds__(64) step_resolve(DevMesh M, DevParticles<R> P, StepParams S,
                                                   const SpeciesK* __restrict__ sp, double* __restrict__ node_charge,
                                                   const WorkItem* __restrict__ wl,
                                                   unsigned long long* __restrict__ cnt,
                                                   unsigned long long* __restrict__ tri_count)
{
    const uint64_t nw = cnt[kCntWork + 2 * S.work_slot];
    const uint32_t step0 = (uint32_t)cnt[kCntStep + S.work_slot];
    // Items go to the waves in turn: lanes of one wave wait for each other's
    // exact work (10 us and more an item), waves do not.  16 runs of 1e4 to 4e5
    // particles, mixed, 200 steps, 123 items: 640-860 -> 390 us.  A list that
    // fills the lanes is taken in order (2.3M items over 6 launches: 8.9 -> 8.2
    // ms; the rows of neighbouring items are neighbours).
    const uint64_t lanes = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t first = nw < lanes ? blockIdx.x + (uint64_t)gridDim.x * threadIdx.x
                                      : blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    for (uint64_t w = first; w < nw; w += lanes) {
        RegSink<GlobalSink> sink{GlobalSink{node_charge}, 0.0, 0.0, 0.0, 0.0};
        WorkItem it = wl[w];
        int64_t i = it.i;
        PState<R> s;
        s.f = P.flags[i];
        s.t = it.t0;
        s.x = P.x[i];
        s.y = P.y[i];
        s.z = P.z[i];
        s.vx = P.vx[i];
        s.vy = P.vy[i];
        s.vz = P.vz[i];
        const SpeciesK& k = sp[(s.f >> kSpeciesShift) & 0xff];
        const RunK* rk = S.runs + ((uint32_t)s.f >> kRunShift);
        const int32_t base = (int32_t)rk->node_base;
        int exh = 0, err = 0, nexact = 0;
        int32_t hit_tri = -1;
        double x0[3] = {it.x0, it.y0, it.z0};
        // (the step's start was recorded by the streaming kernel)
        bool settled = finish_exact(M, x0, s, hit_tri, exh, err);
        if (!settled) add_here(M, s, sink);
        if (settled && S.trk_slot) track_hit<R>(M, S, P.pidx[i], x0, s.t, s.x, s.y, s.z, hit_tri);
        uint32_t settle_step = step0 + (uint32_t)it.k;  // step and start of the settling segment
        double sx = x0[0], sy = x0[1], sz = x0[2];
        if (!settled) {
            const PConst pc = particle_const(S, &k, rk, P.pidx[i] - rk->first);
            TetRec<R> rec;
            rec.t = -1;
            s.set_v2();
            unsigned long long extra = 0;
            for (int ks = it.k + 1; ks < S.nsteps; ++ks) {
                if (s.t >= 0 && (s.f & kStrict) && !S.trk_slot) {
                    if (s.t != rec.t) rec.template load<true>(M, S, k, rk, s.t);
                    while (ks < S.nsteps && plain_step(M, S, pc, step0 + (uint32_t)ks, s, rec, sink)) {
                        ++ks;
                        ++extra;
                    }
                    if (ks == S.nsteps) break;
                }
                const R px = s.x, py = s.y, pz = s.z;
                const int32_t t_before = s.t;
                int32_t tri = -1;
                const int outcome =
                    step_one<R, true, kWalk>(M, S, pc, step0 + (uint32_t)ks, S.nsteps - ks, s, rec, sink, tri);
                if (outcome == kFrozenNow) break;
                ++extra;
                if (S.trk_slot) track_start<R>(M, S, P.pidx[i], t_before, px, py, pz);
                if (outcome == kDeferNow || outcome == kSettledNow) {
                    double x0s[3];
                    abs_pos(M, t_before, px, py, pz, x0s);
                    if (outcome == kDeferNow) {
                        ++nexact;
                        // (the sums belong to the tet the step started in)
                        sink.flush(M, S.charge ? t_before : -1, base, k.charge);
                        settled = finish_exact(M, x0s, s, hit_tri, exh, err);
                        if (!settled) add_here(M, s, sink);
                    } else {
                        hit_tri = tri;
                        settled = true;
                    }
                    if (settled && S.trk_slot) track_hit<R>(M, S, P.pidx[i], x0s, s.t, s.x, s.y, s.z, hit_tri);
                    settle_step = step0 + (uint32_t)ks;
                    sx = x0s[0];
                    sy = x0s[1];
                    sz = x0s[2];
                }
                if (settled) break;
            }
            if (extra) atomicAdd(&cnt[kCntProcSlot0 + (w & (kProcSlots - 1))], extra);
        }
        if (settled) {
            s.f = (s.f | kSettled) & ~kStrict;
            P.hit[i] = hit_tri;
            atomicAdd(&tri_count[rk->tri_base + hit_tri], 1ull);
            S.settle_log[atomicAdd(&cnt[kCntSettled], 1ull)] = P.pidx[i];
            if (S.settle) record_settle(S.settle, P.pidx[i], settle_step, sx, sy, sz);
        }
        // (a settling step left the owner as it was, with the sums of the steps before)
        sink.flush(M, S.charge ? s.t : -1, base, k.charge);
        P.x[i] = s.x;
        P.y[i] = s.y;
        P.z[i] = s.z;
        P.vx[i] = s.vx;
        P.vy[i] = s.vy;
        P.vz[i] = s.vz;
        P.tet[i] = s.t;
        P.flags[i] = s.f;
        if (err) atomicOr(&cnt[kCntError], 1ull);
        if (exh) atomicAdd(&cnt[kCntExhaustive], (unsigned long long)exh);
        if (nexact) atomicAdd(&cnt[kCntDeferred], (unsigned long long)nexact);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&cnt[kCntDeferred], (unsigned long long)nw);
}

// locate_grid by the G lanes of a group for one point p (the same in each of
// them): a lane per candidate, the first that holds p is the answer.
template <int G>
__device__ inline int32_t locate_grid_group(const DevMesh& M, const double* p, int* strict, int* err)
{
    const int lane = threadIdx.x & (G - 1), base = threadIdx.x & 63 & ~(G - 1);
    constexpr unsigned long long kAll = G == 64 ? ~0ull : (1ull << (G & 63)) - 1;
    const unsigned long long below = (1ull << lane) - 1;
    const int a = grid_coord(M.grid, 0, p[0]), b = grid_coord(M.grid, 1, p[1]), c = grid_coord(M.grid, 2, p[2]);
    const int64_t cell = ((int64_t)a * M.grid.div[1] + b) * M.grid.div[2] + c;
    const int32_t begin = M.tgrid_start[cell], end = M.tgrid_start[cell + 1];
    const bool finite = isfinite(p[0]) && isfinite(p[1]) && isfinite(p[2]);
    for (int32_t j = begin; j < end; j += G) {
        int32_t t = -1;
        int r = 0;  // as tet_contains
        bool unsure = false;
        if (j + lane < end) {
            t = M.tgrid_list[j + lane];
            if (!finite || in_box(M.tbox[t], p)) {
                TetMap m;
                m.load(M, t);
                const Sides sd = certified_sides(M, m, p);
                if (sd.pos == 15) r = 2;
                else unsure = !sd.neg;
            }
        }
        const unsigned long long sure = __ballot(r > 0) >> base & kAll;
        // (candidates behind the first certain one cannot be the answer)
        if (unsure && (sure & below) == 0) r = tet_contains(M, t, p);
        const unsigned long long in = __ballot(r > 0) >> base & kAll, bad = __ballot(r < 0) >> base & kAll;
        const int first = in ? __ffsll((long long)in) - 1 : G;
        if (in ? bad & ((1ull << first) - 1) : bad) *err = 1;
        if (in) {
            *strict = __shfl(r, first, G) == 2;
            return __shfl(t, first, G);
        }
    }
    *strict = 0;
    return -1;
}

// Owners of absolute positions (min-id closed containment); with `lx` the
// positions are also written in the frame of their owner (mixed layout).
// G lanes per point: the candidates of a cell come in runs of consecutive
// ids, so that a group reads their boxes and maps together, and with G = 64 a
// point takes a chain of four loads.  Latency bounds it, so G is as large as
// leaves every group resident at once.  On 374k tets, random points, with
// G = 1, 4, 16, 64 (us): 500 points 43, 17, 7.3, 4.8; 16,000 63, 26, 14, 20;
// 131,072 90, 63, 73, 124; 1M 527, 426, 516, 799.  (The exact scan by one
// lane per point took 107 us for any number up to some thousands, 300 us for
// 131,072 and 1.6 ms for 1M.)
template <int G>
__global__ void __launch_bounds__(256) locate_kernel(DevMesh M, const double* __restrict__ x,
                                                     const double* __restrict__ y, const double* __restrict__ z,
                                                     int64_t n, int32_t* __restrict__ tet,
                                                     int32_t* __restrict__ flags, float* __restrict__ lx,
                                                     float* __restrict__ ly, float* __restrict__ lz,
                                                     unsigned long long* __restrict__ cnt)
{
    constexpr int kPoints = 256 / G;  // of a workgroup at a time
    const bool writer = (threadIdx.x & (G - 1)) == 0;
    int err = 0;
    for (int64_t i = blockIdx.x * (int64_t)kPoints + threadIdx.x / G; i < n; i += gridDim.x * (int64_t)kPoints) {
        const double p[3] = {x[i], y[i], z[i]};
        int strict = 0;
        const int32_t t = locate_grid_group<G>(M, p, &strict, &err);
        if (lx) {
            float a, b, c;
            to_frame(M, t, p, a, b, c);
            if (writer) {
                lx[i] = a;
                ly[i] = b;
                lz[i] = c;
            }
            if (t >= 0) {
                double q[3];
                abs_pos(M, t, a, b, c, q);
                TetMap m;
                m.load(M, t);
                strict = certified_sides(M, m, q).pos == 15;
                if (!strict) {
                    int r = tet_contains(M, t, q);
                    if (r < 0) err = 1;
                    strict = r == 2;
                }
            }
        }
        if (writer) {
            tet[i] = t;
            if (flags) flags[i] = strict ? (flags[i] | kStrict) : (flags[i] & ~kStrict);
        }
    }
    if (err && cnt && writer) atomicOr(&cnt[kCntError], 1ull);
}

template <typename R>
__global__ void gather_kernel(DevMesh M, DevParticles<R> P, const SpeciesK* __restrict__ sp,
                              const RunK* __restrict__ runs, double* __restrict__ node_charge)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= P.n) return;
    int32_t f = P.flags[i];
    int32_t t = P.tet[i];
    if ((f & kSettled) || t < 0) return;
    double q = sp[(f >> kSpeciesShift) & 0xff].charge;
    if (q == 0.0) return;
    double lam[4];
    bary_at(M, t, P.x[i], P.y[i], P.z[i], lam);
    scatter4(node_charge + runs[(uint32_t)f >> kRunShift].node_base, M.tnode[t], q, lam);
}

// Occupancy and summed charge of each tet (one owner per unsettled particle).
template <typename R>
__global__ void tet_occupancy_kernel(DevParticles<R> P, const SpeciesK* __restrict__ sp, double* __restrict__ tet_q,
                                     int32_t* __restrict__ tet_n)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= P.n) return;
    int32_t f = P.flags[i], t = P.tet[i];
    if ((f & kSettled) || t < 0) return;
    atomicAdd(&tet_n[t], 1);
    double q = sp[(f >> kSpeciesShift) & 0xff].charge;
    if (q != 0.0) global_add_f64(&tet_q[t], q);
}

// rho_n = sum(rho_t V_t) / sum V_t over the occupied tets around n, ascending tet id
// (NodeChargeDensityProcessor.cpp:69-93).
__global__ void node_density_kernel(const int32_t* __restrict__ adj_start, const int32_t* __restrict__ adj_list,
                                    const double* __restrict__ tet_vol, const double* __restrict__ tet_q,
                                    const int32_t* __restrict__ tet_n, int64_t n_nodes, double* __restrict__ rho,
                                    int32_t* __restrict__ written)
{
    int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (n >= n_nodes) return;
    double tc = 0.0, tv = 0.0;
    for (int32_t j = adj_start[n]; j < adj_start[n + 1]; ++j) {
        int32_t t = adj_list[j];
        if (tet_n[t] == 0) continue;
        double v = tet_vol[t];
        double rt = tet_q[t] / v;
        tc += rt * v;
        tv += v;
    }
    rho[n] = tv > 0.0 ? tc / tv : 0.0;
    if (written) written[n] = tv > 0.0;
}

__global__ void node_density_bary_kernel(const double* __restrict__ q, const double* __restrict__ node_vol,
                                         int64_t n_nodes, double* __restrict__ rho, int32_t* __restrict__ written)
{
    int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (n >= n_nodes) return;
    rho[n] = q[n] / node_vol[n];
    if (written) written[n] = 1;
}

// Push increments h = (((E*q)/m)*dt)/2 of a single run's field for each charged
// species slot (TetRec::load_h's arithmetic, FP64 from E and FP32 from the FP32
// field), -0 where the push is skipped (dt == 0 or E == 0 exactly,
// Particle.cpp:199-207).
struct PushSlots {
    double q[kMaxPushSlots], m[kMaxPushSlots];
    int32_t n;
};
template <typename R>
__device__ inline R push_increment(R e, R q, R m, R dt)
{
    return (((e * q) / m) * dt) / R(2);
}
__device__ inline void push_rows(const double* e, const float* e32, int64_t t, int64_t nt, const PushSlots& ps,
                                 double dt, double* __restrict__ H, float* __restrict__ H32)
{
    for (int k = 0; k < ps.n; ++k) {
        if (H) {
            const bool skip = dt == 0.0 || (e[0] == 0.0 && e[1] == 0.0 && e[2] == 0.0);
            double* h = H + 3 * ((int64_t)k * nt + t);
            for (int c = 0; c < 3; ++c) h[c] = skip ? -0.0 : push_increment<double>(e[c], ps.q[k], ps.m[k], dt);
        }
        if (H32) {
            const float q = (float)ps.q[k], m = (float)ps.m[k], d = (float)dt;
            const bool skip = d == 0.0f || (e32[0] == 0.0f && e32[1] == 0.0f && e32[2] == 0.0f);
            float4 h;
            h.x = skip ? -0.0f : push_increment<float>(e32[0], q, m, d);
            h.y = skip ? -0.0f : push_increment<float>(e32[1], q, m, d);
            h.z = skip ? -0.0f : push_increment<float>(e32[2], q, m, d);
            h.w = 0.0f;
            reinterpret_cast<float4*>(H32)[(int64_t)k * nt + t] = h;
        }
    }
}

// E = -grad(phi) = -sum_j (phi_j - phi_0) A_j  (A_j: gradient of lambda_j), and
// the push increments with it (ps.n slots, 0: none) while the field is in
// registers: FP64 bound by memory, 160 B per tet in one launch instead of 184 in
// two.  750k tets: 17.5 + 8.0 -> 20.9 us.
__global__ void field_kernel(DevMesh M, const double* __restrict__ phi, double* __restrict__ E, float* __restrict__ E32,
                             PushSlots ps, double dt, double* __restrict__ H, float* __restrict__ H32)
{
    int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= M.n_tets) return;
    int4 nv = M.tnode[t];
    TetMap m;
    m.load(M, (int32_t)t);
    const double* g = m.g;
    double p0 = phi[nv.x], d1 = phi[nv.y] - p0, d2 = phi[nv.z] - p0, d3 = phi[nv.w] - p0;
    double e[3];
    float e32[3];
    for (int c = 0; c < 3; ++c) {
        e[c] = -((d1 * g[3 + c] + d2 * g[6 + c]) + d3 * g[9 + c]);
        e32[c] = (float)e[c];
        E[3 * t + c] = e[c];
    }
    if (E32) reinterpret_cast<float4*>(E32)[t] = make_float4(e32[0], e32[1], e32[2], 0.0f);
    push_rows(e, e32, t, M.n_tets, ps, dt, H, H32);
}

// The increments of run 0's field, with run_field's operations where it is not
// basis 0 as given.
__global__ void push_table_kernel(DevMesh M, const RunK* __restrict__ run, int32_t scaled, PushSlots ps, double dt,
                                  double* __restrict__ H, float* __restrict__ H32)
{
    int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= M.n_tets) return;
    double e[3];
    float e32[3] = {0.0f, 0.0f, 0.0f};
    if (scaled) run_field<double, true>(M, run, (int32_t)t, e[0], e[1], e[2]);
    else run_field<double, false>(M, run, (int32_t)t, e[0], e[1], e[2]);
    if (H32) {
        if (scaled) run_field<float, true>(M, run, (int32_t)t, e32[0], e32[1], e32[2]);
        else run_field<float, false>(M, run, (int32_t)t, e32[0], e32[1], e32[2]);
    }
    push_rows(e, e32, t, M.n_tets, ps, dt, H, H32);
}

static PushSlots push_slots(const double* q, const double* m, int32_t n_slots)
{
    PushSlots ps{};
    ps.n = n_slots;
    for (int k = 0; k < n_slots && k < kMaxPushSlots; ++k) {
        ps.q[k] = q[k];
        ps.m[k] = m[k];
    }
    return ps;
}

void launch_push_table(hipStream_t s, const DevMesh& M, const RunK* run, bool scaled, const double* q,
                       const double* m, int32_t n_slots, double dt, double* H, float* H32)
{
    if (M.n_tets > 0 && n_slots > 0)
        push_table_kernel<<<(unsigned)((M.n_tets + 255) / 256), 256, 0, s>>>(M, run, scaled ? 1 : 0,
                                                                             push_slots(q, m, n_slots), dt, H, H32);
}

__device__ inline float round_down(double x)
{
    const float f = (float)x;
    return (double)f > x ? nextafterf(f, -INFINITY) : f;
}
__global__ void tet_box_kernel(DevMesh M, TetBox* __restrict__ box)
{
    int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= M.n_tets) return;
    const int4 nv = M.tnode[t];
    double P[4][3];
    for (int k = 0; k < 4; ++k) load_node(M, nth(nv, k), P[k]);
    TetBox b;
    for (int c = 0; c < 3; ++c) {
        b.lo[c] = round_down(fmin(fmin(P[0][c], P[1][c]), fmin(P[2][c], P[3][c])));
        b.hi[c] = -round_down(-fmax(fmax(P[0][c], P[1][c]), fmax(P[2][c], P[3][c])));
    }
    box[t] = b;
}

void launch_tet_boxes(hipStream_t s, const DevMesh& M, TetBox* box)
{
    tet_box_kernel<<<(unsigned)((M.n_tets + 255) / 256), 256, 0, s>>>(M, box);
}

__global__ void e32_kernel(const double* __restrict__ E, float* __restrict__ E32, int64_t nt)
{
    int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= nt) return;
    E32[4 * t] = (float)E[3 * t];
    E32[4 * t + 1] = (float)E[3 * t + 1];
    E32[4 * t + 2] = (float)E[3 * t + 2];
    E32[4 * t + 3] = 0.0f;
}

__global__ void orient_batch_kernel(const double* __restrict__ pts, int64_t n, int32_t* __restrict__ out)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double* p = pts + 12 * i;
    out[i] = orient3d(p, p + 3, p + 6, p + 9);
}

// the shared elementary functions (dm_*) over n arguments, for checks:
// which = 0 pow(x, y), 1 sin x and cos x, 2 acos x, 3 atan2(y, x), 4 log x, 5 exp x
__global__ void math_batch_kernel(int which, const double* __restrict__ x, const double* __restrict__ y, int64_t n,
                                  double* __restrict__ out, double* __restrict__ out2)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    double r = 0.0, r2 = 0.0;
    if (which == 0) r = dm_pow(x[i], y[i]);
    else if (which == 1) dm_sincos(x[i], &r, &r2);
    else if (which == 2) r = dm_acos(x[i]);
    else if (which == 3) r = dm_atan2(y[i], x[i]);
    else if (which == 4) r = dm_log(x[i]);
    else r = dm_exp(x[i]);
    out[i] = r;
    out2[i] = r2;
}

// The rows of a new population besides its state: load indices, hit triangle
// -1, and the flags of its species and run (species null: the flags are there);
// with them the live row count and the next launch's step, and the state from
// the staging buffer (one launch instead of six copies of 3 us each).
__global__ void init_rows_kernel(int64_t first, int64_t m, RowColumns cols, const int32_t* __restrict__ species,
                                 const RunK* __restrict__ runs, int32_t n_runs, int32_t* __restrict__ flags,
                                 int32_t* __restrict__ hit, uint32_t* __restrict__ pidx, int64_t* __restrict__ n_active,
                                 int64_t active, unsigned long long* __restrict__ step_cnt, unsigned long long step)
{
    const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (j == 0) {
        *n_active = active;
        *step_cnt = step;
    }
    if (j >= m) return;
    for (int k = 0; k < 6; ++k)
        if (cols.src[k]) cols.dst[k][j] = cols.src[k][j];
    const int64_t i = first + j;
    hit[i] = -1;
    pidx[i] = (uint32_t)i;
    if (species) {
        int32_t lo = 0, hi = n_runs - 1;  // the last run whose first row is not after i
        while (lo < hi) {
            const int32_t mid = (lo + hi + 1) / 2;
            if ((int64_t)runs[mid].first <= i) lo = mid;
            else hi = mid - 1;
        }
        flags[i] = (species[j] << kSpeciesShift) | (lo << kRunShift);
    }
}

void launch_init_rows(hipStream_t s, int64_t first, int64_t m, const RowColumns& cols, const int32_t* species, const RunK* runs,
                      int32_t n_runs, int32_t* flags, int32_t* hit, uint32_t* pidx, int64_t* n_active, int64_t active,
                      unsigned long long* step_cnt, unsigned long long step)
{
    init_rows_kernel<<<(unsigned)std::max<int64_t>(1, (m + 255) / 256), 256, 0, s>>>(
        first, m, cols, species, runs, n_runs, flags, hit, pidx, n_active, active, step_cnt, step);
}

// The state by load index, positions absolute in FP64: the rows written
// where they belong, so that the host only copies.  Null outputs are skipped.
template <typename R>
__global__ void load_order_kernel(DevMesh M, DevParticles<R> P, ReadBack out)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= P.n) return;
    const uint32_t j = P.pidx[i];
    if (out.f[0] || out.f[1] || out.f[2]) {
        double p[3];
        abs_pos(M, P.tet[i], P.x[i], P.y[i], P.z[i], p);
        for (int k = 0; k < 3; ++k)
            if (out.f[k]) out.f[k][j] = p[k];
    }
    if (out.f[3]) out.f[3][j] = P.vx[i];
    if (out.f[4]) out.f[4][j] = P.vy[i];
    if (out.f[5]) out.f[5][j] = P.vz[i];
    if (out.tet) out.tet[j] = P.tet[i];
    if (out.settled) out.settled[j] = (P.flags[i] & kSettled) ? 1 : 0;
    if (out.hit) out.hit[j] = P.hit[i];
}

template <typename R>
void launch_load_order(hipStream_t s, const DevMesh& M, const DevParticles<R>& P, const ReadBack& out)
{
    if (P.n > 0) load_order_kernel<R><<<(unsigned)((P.n + 255) / 256), 256, 0, s>>>(M, P, out);
}
template void launch_load_order<double>(hipStream_t, const DevMesh&, const DevParticles<double>&, const ReadBack&);
template void launch_load_order<float>(hipStream_t, const DevMesh&, const DevParticles<float>&, const ReadBack&);

// ---------------------------------------------------------------------------
// Adjoint of the collisionless push and the surface-hit map.
//
// Forward, step k with owner t_k of x_k:
//   v_{k+1} = v_k + a(t_k) dt,  a = (q/m) (s0 E_0 + s1 E_1),  x_{k+1} = x_k + v_{k+1} dt.
// The particle settles in step k* on triangle T (plane n.x = n.A); its hit
// point is x_h = x_a + s D with x_a = x_{k*}, D = x_{k*+1} - x_a and
// s = n.(A - x_a) / n.D.  Linearised: dx_h = P (dx_a + s dt dv_{k*+1}) with
// P = I - D n^T / (n.D).  For a loss L with lambda = dL/dx_h the reverse sweep is
//   lx = P^T lambda                    adjoint of every x_k (E is constant per tet)
//   mu_k* = s dt P^T lambda            adjoint of v_{k*+1}
//   mu_{k-1} = mu_k + dt lx
//   dL/ds_j += mu_k . (q/m) E_j(t_k) dt,   k = k*, ..., k0.
// The owners t_k are recomputed backwards -- x_{k-1} = x_k - v_k dt with v_k
// the push of t_k undone -- instead of storing the trajectory.
// ---------------------------------------------------------------------------

// Which particles the next step records a movement for, by load index: not
// settled, |v| >= 10 m/s and inside the expanded bounding box (the filters of
// ParticleDynamicsProcessor.cpp:166-176, as step_one applies them).
template <typename R>
__global__ void track_eligible_kernel(DevMesh M, DevParticles<R> P, StepParams S, uint8_t* __restrict__ out)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= P.n) return;
    const int32_t f = P.flags[i];
    const R vx = (R)P.vx[i], vy = (R)P.vy[i], vz = (R)P.vz[i];
    const R vmod = m_sqrt<R>(vx * vx + vy * vy + vz * vz);
    const bool live = !(f & kSettled) && !(vmod < R(10)) && in_bbox_at(M, S, P.tet[i], P.x[i], P.y[i], P.z[i]);
    out[P.pidx[i]] = live ? 1 : 0;
}

// hit points, triangles and settle steps of the settled particles, in load order
template <typename R>
__global__ void hit_points_kernel(DevMesh M, DevParticles<R> P, const SettleRec* __restrict__ rec,
                                  double* __restrict__ xh, int32_t* __restrict__ tri, int32_t* __restrict__ step)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= P.n) return;
    uint32_t p = P.pidx[i];
    SettleRec r = rec[p];
    if (!(P.flags[i] & kSettled) || r.step < 0) {
        xh[3 * (int64_t)p] = xh[3 * (int64_t)p + 1] = xh[3 * (int64_t)p + 2] = 0.0;
        tri[p] = -1;
        step[p] = -1;
        return;
    }
    double xb[3], xa[3] = {r.x0, r.y0, r.z0}, D[3], n[3], s;
    abs_pos(M, P.tet[i], P.x[i], P.y[i], P.z[i], xb);
    for (int k = 0; k < 3; ++k) D[k] = xb[k] - xa[k];
    hit_plane(M, P.hit[i], xa, D, n, s);
    for (int k = 0; k < 3; ++k) xh[3 * (int64_t)p + k] = xa[k] + s * D[k];
    tri[p] = P.hit[i];
    step[p] = r.step;
}

// Out of line, so that the exact predicates' registers are not the kernel's.
struct Located {
    int32_t tet, err;
};
__device__ __noinline__ Located locate_slow(const DevMesh& M, int32_t hint, double x, double y, double z)
{
    const double p[3] = {x, y, z};
    int strict = 0, err = 0;
    const int32_t t = hint >= 0 ? locate_near_exact(M, hint, p, &strict, &err) : locate_grid(M, p, &strict, &err);
    return Located{t, err};
}

// A lane per particle; latency of the few waves there are bounds it (4 waves
// per SIMD for 262,144 particles), so a step reads memory only where the owner
// changes, and the owner is found from barycentric maps, the exact predicates
// out of line.  262,144 particles, 1,000 steps, 203k tets: 5.6 -> 1.9 ms
// (the predicates in every step, three divisions, fields read in every step).
template <typename R>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) adjoint_push_kernel(DevMesh M, DevParticles<R> P,
                                                           const SpeciesK* __restrict__ sp,
                                                           const RunK* __restrict__ runs, double dt, int32_t k0,
                                                           const SettleRec* __restrict__ rec,
                                                           const double* __restrict__ lambda,
                                                           double* __restrict__ grad,
                                                           unsigned long long* __restrict__ cnt)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    double g0 = 0.0, g1 = 0.0;
    int err = 0;
    if (i < P.n) {
        const int32_t f = P.flags[i];
        const uint32_t p = P.pidx[i];
        const double lam[3] = {lambda[3 * (int64_t)p], lambda[3 * (int64_t)p + 1], lambda[3 * (int64_t)p + 2]};
        const SettleRec r = rec[p];
        if ((f & kSettled) && r.step >= k0 && (lam[0] != 0.0 || lam[1] != 0.0 || lam[2] != 0.0)) {
            const SpeciesK& k = sp[(f >> kSpeciesShift) & 0xff];
            const RunK& rk = runs[(uint32_t)f >> kRunShift];
            const double qm = k.charge / k.mass;
            int32_t t = P.tet[i];
            double xb[3], x[3] = {r.x0, r.y0, r.z0}, D[3], n[3], s;
            abs_pos(M, t, P.x[i], P.y[i], P.z[i], xb);
            for (int c = 0; c < 3; ++c) D[c] = xb[c] - x[c];
            hit_plane(M, P.hit[i], x, D, n, s);
            const double nD = (n[0] * D[0] + n[1] * D[1]) + n[2] * D[2];
            const double Dl = (D[0] * lam[0] + D[1] * lam[1]) + D[2] * lam[2];
            double pl[3], mu[3];
            for (int c = 0; c < 3; ++c) {
                pl[c] = lam[c] - n[c] * (Dl / nD);
                mu[c] = (s * dt) * pl[c];
            }
            double v[3] = {(double)P.vx[i], (double)P.vy[i], (double)P.vz[i]};
            // of the owner t, read when it changes: the basis fields, the
            // push increment and the barycentric map
            double e0[3], e1[3], h[3];
            TetMap m;
            auto enter = [&] {
                bool zero = true;
                for (int c = 0; c < 3; ++c) {
                    e0[c] = t >= 0 ? M.E[3 * (int64_t)t + c] : 0.0;
                    e1[c] = t >= 0 && M.E1 ? M.E1[3 * (int64_t)t + c] : 0.0;
                    const double E = rk.s0 * e0[c] + rk.s1 * e1[c];
                    zero = zero && E == 0.0;
                    h[c] = (((E * k.charge) / k.mass) * dt) / 2.0;
                }
                if (t < 0 || zero)
                    for (int c = 0; c < 3; ++c) h[c] = 0.0;  // (v - 0) - 0 = v
            };
            enter();
            if (t >= 0) m.load(M, t);
            for (int32_t kk = r.step;; --kk) {
                g0 += (((mu[0] * e0[0] + mu[1] * e0[1]) + mu[2] * e0[2]) * qm) * dt;
                g1 += (((mu[0] * e1[0] + mu[1] * e1[1]) + mu[2] * e1[2]) * qm) * dt;
                if (kk <= k0) break;
                for (int c = 0; c < 3; ++c) v[c] = (v[c] - h[c]) - h[c];  // the push of step kk undone: forward (v + h) + h
                for (int c = 0; c < 3; ++c) x[c] = x[c] - v[c] * dt;
                const int32_t from = t;
                if (t < 0 || !walk_near(M, t, m, x)) {
                    const Located at = locate_slow(M, from, x[0], x[1], x[2]);
                    t = at.tet;
                    err |= at.err;
                    if (t >= 0) m.load(M, t);
                }
                if (t != from) enter();
                for (int c = 0; c < 3; ++c) mu[c] = mu[c] + dt * pl[c];
            }
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        g0 += __shfl_xor(g0, off);
        g1 += __shfl_xor(g1, off);
    }
    if ((threadIdx.x & 63) == 0 && (g0 != 0.0 || g1 != 0.0)) {
        global_add_f64(&grad[0], g0);
        global_add_f64(&grad[1], g1);
    }
    if (err) atomicOr(&cnt[kCntError], 1ull);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline unsigned blocks_for(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

void launch_zero_charge(hipStream_t s, double* a, double* b, int64_t n_nodes)
{
    unsigned nb = std::max(1u, std::min(blocks_for(n_nodes, 256), 2048u));
    prologue_kernel<<<nb, 256, 0, s>>>(a, b, n_nodes);
}

template <typename R>
void launch_step(hipStream_t s, const DevMesh& M, const DevParticles<R>& P, const StepParams& S,
                 const SpeciesK* sp, double* node_charge, WorkItem* wl, unsigned long long* cnt,
                 unsigned long long* tri_count, const StepLaunch& L, hipEvent_t ev_mid)
{
    const StepArgs<R> A{M, P, S, sp, node_charge, wl, cnt, tri_count};
    if (P.n > 0 && S.nsteps == 1) {
        // single steps: 256 threads and a workgroup per tile, whatever shape the
        // fused launches have.  1M particles on 750k tets, in us, FP64 and mixed,
        // against step_tile in the shape asked for: a batch of 4 runs 107 and
        // 102 (122, 117); with movement records 70 and 70 (95, 109); block 128
        // without the walk 51 and 46 (75, 69); persistent 52 and 46 (117, 117)
        const unsigned grid = blocks_for(P.n, 256);
        switch ((S.trk_slot ? 4 : 0) + (L.batch ? 2 : 0) + (L.walk ? 1 : 0)) {
#define SG_STEP_SINGLE(T_, B_, W_) \
    step_main<R, 256, B_, false, W_, T_, true><<<grid, 256, 0, s>>>(A)
        case 0: SG_STEP_SINGLE(false, false, false); break;
        case 1: SG_STEP_SINGLE(false, false, true); break;
        case 2: SG_STEP_SINGLE(false, true, false); break;
        case 3: SG_STEP_SINGLE(false, true, true); break;
        case 4: SG_STEP_SINGLE(true, false, false); break;
        case 5: SG_STEP_SINGLE(true, false, true); break;
        case 6: SG_STEP_SINGLE(true, true, false); break;
        default: SG_STEP_SINGLE(true, true, true); break;
#undef SG_STEP_SINGLE
        }
    } else if (P.n > 0 && S.trk_slot) {
        // movement records: the tracking variants (256-thread workgroups, one per tile)
        const unsigned grid = blocks_for(P.n, 256);
        switch ((L.batch ? 2 : 0) + (L.walk ? 1 : 0)) {
#define SG_STEP_TRACK(B_, W_) \
    step_main<R, 256, B_, false, W_, true><<<grid, 256, 0, s>>>(A)
        case 0: SG_STEP_TRACK(false, false); break;
        case 1: SG_STEP_TRACK(false, true); break;
        case 2: SG_STEP_TRACK(true, false); break;
        default: SG_STEP_TRACK(true, true); break;
#undef SG_STEP_TRACK
        }
    } else if (P.n > 0 && !S.charge && S.model == 0 && L.walk && !L.persistent) {
        // neither charge nor gas (electrode optimisation and its adjoint, in
        // its own launch shape): see step_tile
        const unsigned grid = blocks_for(P.n, 256);
        if (L.batch)
            step_main<R, 256, true, false, true, false, false, true><<<grid, 256, 0, s>>>(A);
        else
            step_main<R, 256, false, false, true, false, false, true><<<grid, 256, 0, s>>>(A);
    } else if (P.n > 0) {
        const unsigned grid = L.persistent ? (unsigned)L.grid : blocks_for(P.n, L.block == 128 ? 128 : 256);
        // the multi-tet walk is instantiated for 256-thread workgroups only
        // (the host sets block = 256 with it)
        const int v = L.walk ? 8 + (L.batch ? 2 : 0) + (L.persistent ? 1 : 0)
                             : (L.block == 128 ? 4 : 0) + (L.batch ? 2 : 0) + (L.persistent ? 1 : 0);
        switch (v) {
#define SG_STEP_MAIN(BS_, B_, P_, W_) \
    step_main<R, BS_, B_, P_, W_><<<grid, BS_, 0, s>>>(A)
        case 0: SG_STEP_MAIN(256, false, false, false); break;
        case 1: SG_STEP_MAIN(256, false, true, false); break;
        case 2: SG_STEP_MAIN(256, true, false, false); break;
        case 3: SG_STEP_MAIN(256, true, true, false); break;
        case 4: SG_STEP_MAIN(128, false, false, false); break;
        case 5: SG_STEP_MAIN(128, false, true, false); break;
        case 6: SG_STEP_MAIN(128, true, false, false); break;
        case 7: SG_STEP_MAIN(128, true, true, false); break;
        case 8: SG_STEP_MAIN(256, false, false, true); break;
        case 9: SG_STEP_MAIN(256, false, true, true); break;
        case 10: SG_STEP_MAIN(256, true, false, true); break;
        default: SG_STEP_MAIN(256, true, true, true); break;
#undef SG_STEP_MAIN
        }
    }
    if (ev_mid) (void)hipEventRecord(ev_mid, s);
    // the work list is only known on the device: a grid of up to 1,024
    // single-wave workgroups -- one per SIMD, all that can be resident at the
    // kernel's 300+ VGPRs -- and the rest of the list by grid stride; 64 for
    // a single step, whose list is short (one exact relocation per deferred
    // particle) and mostly empty.  (4,096 cost 10 us per launch with an empty
    // list, 13% of a single step; 64 saves 0.3 us per step against 256.)
    const unsigned cap = S.nsteps == 1 ? 64u : 1024u;
    unsigned nb = std::max(1u, std::min(blocks_for(P.n, 64), cap));
    if (L.walk)
        step_resolve<R, true><<<nb, 64, 0, s>>>(M, P, S, sp, node_charge, wl, cnt, tri_count);
    else
        step_resolve<R, false><<<nb, 64, 0, s>>>(M, P, S, sp, node_charge, wl, cnt, tri_count);
}

void launch_locate(hipStream_t s, const DevMesh& M, const double* x, const double* y, const double* z, int64_t n,
                   int32_t* tet, int32_t* flags, float* lx, float* ly, float* lz, unsigned long long* cnt)
{
    if (n <= 0) return;
    // as many lanes per point as the chip holds at once (16 waves on each of
    // 256 CUs): see locate_kernel
    constexpr int64_t kLanes = 256 * 16 * 64;
    auto go = [&](auto group) {
        constexpr int G = decltype(group)::value;
        locate_kernel<G><<<std::min(blocks_for(n, 256 / G), 65536u), 256, 0, s>>>(M, x, y, z, n, tet, flags, lx, ly,
                                                                                lz, cnt);
    };
    if (64 * n <= kLanes) go(std::integral_constant<int, 64>{});
    else if (16 * n <= kLanes) go(std::integral_constant<int, 16>{});
    else go(std::integral_constant<int, 4>{});
}

template <typename R>
void launch_gather(hipStream_t s, const DevMesh& M, const DevParticles<R>& P, const SpeciesK* sp, const RunK* runs,
                   double* node_charge)
{
    if (P.n > 0) gather_kernel<R><<<blocks_for(P.n, 256), 256, 0, s>>>(M, P, sp, runs, node_charge);
}

template <typename R>
void launch_hit_points(hipStream_t s, const DevMesh& M, const DevParticles<R>& P, const SettleRec* rec, double* xh,
                       int32_t* tri, int32_t* step)
{
    if (P.n > 0) hit_points_kernel<R><<<blocks_for(P.n, 256), 256, 0, s>>>(M, P, rec, xh, tri, step);
}

template <typename R>
void launch_track_eligible(hipStream_t s, const DevMesh& M, const DevParticles<R>& P, const StepParams& S,
                           uint8_t* out)
{
    if (P.n > 0) track_eligible_kernel<R><<<blocks_for(P.n, 256), 256, 0, s>>>(M, P, S, out);
}
template void launch_track_eligible<double>(hipStream_t, const DevMesh&, const DevParticles<double>&,
                                            const StepParams&, uint8_t*);
template void launch_track_eligible<float>(hipStream_t, const DevMesh&, const DevParticles<float>&,
                                           const StepParams&, uint8_t*);

template <typename R>
void launch_adjoint_push(hipStream_t s, const DevMesh& M, const DevParticles<R>& P, const SpeciesK* sp,
                         const RunK* runs, double dt, int32_t k0, const SettleRec* rec, const double* lambda,
                         double* grad, unsigned long long* cnt)
{
    if (P.n > 0)
        adjoint_push_kernel<R><<<blocks_for(P.n, 256), 256, 0, s>>>(M, P, sp, runs, dt, k0, rec, lambda, grad, cnt);
}
template void launch_hit_points<double>(hipStream_t, const DevMesh&, const DevParticles<double>&, const SettleRec*,
                                        double*, int32_t*, int32_t*);
template void launch_hit_points<float>(hipStream_t, const DevMesh&, const DevParticles<float>&, const SettleRec*,
                                       double*, int32_t*, int32_t*);
template void launch_adjoint_push<double>(hipStream_t, const DevMesh&, const DevParticles<double>&, const SpeciesK*,
                                          const RunK*, double, int32_t, const SettleRec*, const double*, double*,
                                          unsigned long long*);
template void launch_adjoint_push<float>(hipStream_t, const DevMesh&, const DevParticles<float>&, const SpeciesK*,
                                         const RunK*, double, int32_t, const SettleRec*, const double*, double*,
                                         unsigned long long*);

template <typename R>
void launch_node_density(hipStream_t s, const DevParticles<R>& P, const SpeciesK* sp, int32_t mode,
                         const double* node_q, const double* node_vol, const int32_t* adj_start,
                         const int32_t* adj_list, const double* tet_vol, double* tet_q, int32_t* tet_n,
                         int64_t n_nodes, double* rho, int32_t* written)
{
    if (mode == 0) {
        node_density_bary_kernel<<<blocks_for(n_nodes, 256), 256, 0, s>>>(node_q, node_vol, n_nodes, rho, written);
        return;
    }
    if (P.n > 0) tet_occupancy_kernel<R><<<blocks_for(P.n, 256), 256, 0, s>>>(P, sp, tet_q, tet_n);
    node_density_kernel<<<blocks_for(n_nodes, 256), 256, 0, s>>>(adj_start, adj_list, tet_vol, tet_q, tet_n, n_nodes,
                                                                  rho, written);
}
template void launch_node_density<double>(hipStream_t, const DevParticles<double>&, const SpeciesK*, int32_t,
                                          const double*, const double*, const int32_t*, const int32_t*,
                                          const double*, double*, int32_t*, int64_t, double*, int32_t*);
template void launch_node_density<float>(hipStream_t, const DevParticles<float>&, const SpeciesK*, int32_t,
                                         const double*, const double*, const int32_t*, const int32_t*,
                                         const double*, double*, int32_t*, int64_t, double*, int32_t*);

void launch_field(hipStream_t s, const DevMesh& M, const double* phi, double* E, float* E32, const double* q,
                  const double* m, int32_t n_slots, double dt, double* H, float* H32)
{
    field_kernel<<<blocks_for(M.n_tets, 256), 256, 0, s>>>(M, phi, E, E32, push_slots(q, m, n_slots), dt, H, H32);
}

void launch_e32(hipStream_t s, const double* E, float* E32, int64_t nt)
{
    e32_kernel<<<blocks_for(nt, 256), 256, 0, s>>>(E, E32, nt);
}

void launch_orient_batch(hipStream_t s, const double* pts, int64_t n, int32_t* out)
{
    if (n > 0) orient_batch_kernel<<<blocks_for(n, 64), 64, 0, s>>>(pts, n, out);
}

void launch_math_batch(hipStream_t s, int which, const double* x, const double* y, int64_t n, double* out,
                       double* out2)
{
    if (n > 0) math_batch_kernel<<<blocks_for(n, 256), 256, 0, s>>>(which, x, y, n, out, out2);
}

template void launch_step<double>(hipStream_t, const DevMesh&, const DevParticles<double>&, const StepParams&,
                                  const SpeciesK*, double*, WorkItem*, unsigned long long*, unsigned long long*,
                                  const StepLaunch&, hipEvent_t);
template void launch_step<float>(hipStream_t, const DevMesh&, const DevParticles<float>&, const StepParams&,
                                 const SpeciesK*, double*, WorkItem*, unsigned long long*, unsigned long long*,
                                 const StepLaunch&, hipEvent_t);
template void launch_gather<double>(hipStream_t, const DevMesh&, const DevParticles<double>&, const SpeciesK*,
                                    const RunK*, double*);
template void launch_gather<float>(hipStream_t, const DevMesh&, const DevParticles<float>&, const SpeciesK*,
                                   const RunK*, double*);

}  // namespace sg
