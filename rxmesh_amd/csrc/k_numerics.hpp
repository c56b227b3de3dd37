// Numerics on top of the query engine: cotangent CSR assembly over the
// oriented VV ring, SpMV-3 with the fused explicit mean-curvature-flow update,
// and the symmetric Dirichlet energy with its hand-written adjoint.
#pragma once
#include <cfloat>
#include <type_traits>

#include "k_geometry.hpp"

namespace rxm {

struct f3
{
    float x, y, z;
};
__device__ __forceinline__ f3 sub(f3 a, f3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ float dot(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ f3 cross(f3 a, f3 b)
{
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// reference: include/rxmesh/geometry_util.cuh:50-58 (tri_area)
__device__ __forceinline__ float tri_area(f3 p0, f3 p1, f3 p2)
{
    const f3 c = cross(sub(p1, p0), sub(p2, p0));
    return 0.5f * sqrtf(dot(c, c));
}
// reference: geometry_util.cuh:107-114 (clamp_cot, +-19.1)
__device__ __forceinline__ float clamp_cot(float v) { return (v < -19.1f) ? -19.1f : ((v > 19.1f) ? 19.1f : v); }

// reference: geometry_util.cuh:120-172 (partial_voronoi_area of p in CCW p->q->r)
__device__ __forceinline__ float partial_voronoi_area(f3 p, f3 q, f3 r)
{
    const f3    pq = sub(q, p), qr = sub(r, q), pr = sub(r, p);
    const float area = tri_area(p, q, r);
    if (area <= FLT_MIN) return -1.f;
    const float dotp = dot(pq, pr), dotq = -dot(qr, pq), dotr = dot(qr, pr);
    if (dotp < 0.f) return 0.25f * area;
    if (dotq < 0.f || dotr < 0.f) return 0.125f * area;
    const float cotq = clamp_cot(dotq / area), cotr = clamp_cot(dotr / area);
    return 0.125f * (dot(pr, pr) * cotq + dot(pq, pq) * cotr);
}

// reference: geometry_util.cuh:178-206 (edge_cotan_weight of edge p-r with
// opposite vertices q and s; "cot" = dot / area)
__device__ __forceinline__ float edge_cotan_weight(f3 p, f3 r, f3 q, f3 s)
{
    auto part = [&](f3 v) {
        const f3    d0 = sub(p, v), d1 = sub(r, v);
        const float area = tri_area(p, r, v);
        return (area > FLT_MIN) ? clamp_cot(dot(d0, d1) / area) : 0.f;
    };
    return part(q) + part(s);
}

// ---- cotangent CSR assembly ------------------------------------------------
// One wedge (p, a, b) of a vertex's ring: the clamped cotangents of the
// angles at a and at b (reference "cot" = dot / tri_area) and the wedge's
// partial Voronoi area at p (geometry_util.cuh:120-172, clamped at 0). Each
// wedge enters two edge weights and one area, so a ring of K edges costs K
// wedges (one reciprocal square root each) instead of 3K triangle areas.
// |cross|^2 <= FLT_MIN counts as degenerate (area 0): cotangents 0 and no
// Voronoi share, as the reference's area <= FLT_MIN tests give.
struct Wedge
{
    float ca, cb, vor;
};
__device__ __forceinline__ Wedge wedge(f3 p, f3 a, f3 b)
{
    const f3    pa = sub(a, p), pb = sub(b, p), ab = sub(b, a);
    const f3    c  = cross(pa, pb);
    const float cc = dot(c, c);
    Wedge       w{0.f, 0.f, 0.f};
    if (!(cc > FLT_MIN)) return w;
    const float rs   = __builtin_amdgcn_rsqf(cc);
    const float area = 0.5f * cc * rs;  // tri_area
    const float inv  = 2.0f * rs;       // 1 / tri_area
    const float dp = dot(pa, pb), da = -dot(pa, ab), db = dot(pb, ab);
    w.ca = clamp_cot(da * inv);
    w.cb = clamp_cot(db * inv);
    if (dp < 0.f) w.vor = 0.25f * area;
    else if (da < 0.f || db < 0.f) w.vor = 0.125f * area;
    else w.vor = fmaxf(0.125f * (dot(pb, pb) * w.ca + dot(pa, pa) * w.cb), 0.f);
    return w;
}

// Per-face terms of the reference weights (geometry_util.cuh:107-206) for
// face (a0, a1, a2): cot[j] = the clamped cotangent of the angle at a_j
// ("cot" = dot / tri_area), which enters the weight of the opposite edge
// (face slot j + 1, a_{j+1} -> a_{j+2}); vor[j] = the partial Voronoi area of
// a_j in the face (partial_voronoi_area(a_j, a_{j+1}, a_{j+2}) clamped at 0).
// |cross|^2 <= FLT_MIN counts as degenerate: all terms 0, as the
// reference's area <= FLT_MIN tests give.
struct FaceCot
{
    float cot[3], vor[3];
};
__device__ __forceinline__ FaceCot face_cot(f3 P0, f3 P1, f3 P2)
{
    const f3    E0 = sub(P1, P0), E1 = sub(P2, P1), E2 = sub(P0, P2);
    const f3    c  = cross(E0, E2);
    const float cc = dot(c, c);
    FaceCot     r{{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
    if (!(cc > FLT_MIN)) return r;
    const float rs = __builtin_amdgcn_rsqf(cc);
    const float area = 0.5f * cc * rs, inv = 2.0f * rs;
    const float D[3] = {-dot(E0, E2), -dot(E1, E0), -dot(E2, E1)};  // corner dots
    const float L[3] = {dot(E0, E0), dot(E1, E1), dot(E2, E2)};     // |a_{j+1} - a_j|^2
#pragma unroll
    for (int j = 0; j < 3; ++j) r.cot[j] = clamp_cot(D[j] * inv);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int j1 = (j + 1) % 3, j2 = (j + 2) % 3;
        if (D[j] < 0.f) r.vor[j] = 0.25f * area;
        else if (D[j1] < 0.f || D[j2] < 0.f) r.vor[j] = 0.125f * area;
        else r.vor[j] = fmaxf(0.125f * (L[j2] * r.cot[j1] + L[j] * r.cot[j2]), 0.f);
    }
    return r;
}

// LDS carve of the assembly: float4 positions of the patch vertices, the
// ribbon's linear ids, the EV slab, per-edge half-edge terms (half-edge 2e + dir
// starts at the edge's (dir ? hi16 : lo16) endpoint; cot = the clamped cotangent
// of the angle opposite it in its face, vor = the partial Voronoi area of its
// start in that face; zeros where no face of the patch holds it), and the
// patch's pattern: row starts (nvo + 1) and half-edge entries (nent).
struct PlanCOT
{
    float4*   pos;
    float2 *  cot, *vor;  // per edge: the two half-edges' opposite cotangents / start Voronoi terms
    uint32_t *rid, *ev;
    uint16_t *ro, *ent;
};
__host__ __device__ inline PlanCOT plan_cot(Bump& b, uint32_t nv, uint32_t ne, uint32_t nvo, uint32_t nent)
{
    PlanCOT p{};
    p.pos = b.alloc<float4>(nv);
    p.cot = b.alloc<float2>(ne);
    p.vor = b.alloc<float2>(ne);
    p.rid = b.alloc<uint32_t>(nv);
    p.ev  = b.alloc<uint32_t>(r4(ne));
    p.ro  = b.alloc<uint16_t>((nvo + 1u + 7u) & ~7u);
    p.ent = b.alloc<uint16_t>((nent + 7u) & ~7u);
    return p;
}

// Rows of A = M + dt L over linear ids (apps/MCF/mcf_kernels.cuh:354-426,
// mcf_A_setup): the diagonal, then the neighbours in VV query order
// (ascending local id of the connecting edge), the column order SparseMatrix
// fills (sparse_matrix_kernels.cuh:75-140); mass[v] = 1 / v_weight.
// The pattern is static, like the reference's SparseMatrix: the VV plan's rows
// (roff) and half-edge entries (ent); the patch's run of the system starts at
// vv_base (the VV query's per-patch base) + the vertex prefix, one diagonal
// per owned row.
// Every face of the patch is evaluated once and stores, for each of its
// half-edges, the cotangent opposite it and the Voronoi term of its start
// (plain stores: a half-edge has one face on a consistently oriented
// manifold). An edge's weight is cot(2e) + cot(2e + 1) -- the reference's
// part(q) + part(s), in an order floating-point addition does not see --
// and a row's area sums the Voronoi terms of its outgoing half-edges. This
// equals the reference's walk over the oriented ring for every vertex whose
// ring is one closed fan; the rows of other vertices (boundary, several
// fans) take wedges across the ring's gaps, as the reference's cyclic walk
// does, and are rewritten afterwards by k_cot_ring_rows.
// CSR false: values, mass and, by vertex, the diagonal only (the weights of the
// matrix-free solve); row_ptr and col are not written.
// All loads of the staging are issued before the first is waited for, with
// 16-byte loads of the pattern: 27.6 -> 24.8 us on
// 654k vertices. Bound: the face pass's arithmetic and the rows' LDS gathers.
template <uint32_t T, bool CSR = true>
__global__ __launch_bounds__(T) void k_cot_assemble(DevMesh m, const uint32_t* __restrict__ vv_base,
                                                    const uint32_t* __restrict__ rbase,
                                                    const uint32_t* __restrict__ nbase,
                                                    const uint16_t* __restrict__ roff,
                                                    const uint16_t* __restrict__ ent, const float* __restrict__ pos,
                                                    float dt, int32_t* __restrict__ row_ptr,
                                                    int32_t* __restrict__ col, float* __restrict__ val,
                                                    float* __restrict__ mass, float* __restrict__ diag)
{
    extern __shared__ uint4 smem[];
    const uint32_t p = patch_of_block(m.P);  // XCD-contiguous patch ranges
    if (p >= m.P) return;
    const PatchDesc d   = load_desc(m.patch, p);
    const uint32_t  vb  = vv_base[p], nent = vv_base[p + 1] - vb;
    const uint32_t  bse = vb + d.vp;  // first entry of the patch's rows
    Bump            b(reinterpret_cast<char*>(smem));
    const PlanCOT   L = plan_cot(b, d.nv, d.ne, d.nvo, nent);
    const uint32_t  t = threadIdx.x;
    // the FE words of this thread's faces, loaded with the staging's loads
    constexpr uint32_t RF = (1024u + T - 1u) / T;
    const uint16_t*    fe = m.fe + 3u * d.f_off;
    const u32x4 *      evs = reinterpret_cast<const u32x4*>(m.ev + d.e_off), *ros = as_words(roff + rbase[p]),
                *ens = as_words(ent + nbase[p]);
    FaceWords                           fw[RF];
    HeldVerts<T, 3>                     hv_;
    Held<T, (384u + T - 1u) / T, u32x4> h_ev;
    Held<T, (256u + T - 1u) / T, u32x4> h_ent;
    Held<T, 1, u32x4>                   h_ro;
    hv_.ids(m, d);
#pragma unroll
    for (uint32_t r = 0; r < RF; ++r)
        if (r == 0 || r * T < d.nf) fw[r].load(fe, min(t + r * T, d.nf - 1u));
    h_ev.load(evs, r4(d.ne) >> 2);
    h_ro.load(ros, words8(d.nvo + 1));
    h_ent.load(ens, words8(nent));
    hv_.owned(pos, m, d);
    hv_.ribbon(pos, m, d);
    for (uint32_t i = t; i < d.ne; i += T) {
        L.cot[i] = make_float2(0.f, 0.f);
        L.vor[i] = make_float2(0.f, 0.f);
    }
    if constexpr (CSR) {
#pragma unroll
        for (uint32_t k = 0; k < HeldVerts<T, 3>::RR; ++k)
            if (d.nvo + t + k * T < d.nv) L.rid[t + k * T] = hv_.g[k];
        for (uint32_t l = d.nvo + t + HeldVerts<T, 3>::RR * T; l < d.nv; l += T) L.rid[l - d.nvo] = m.v_lin[d.v_off + l];
    }
    h_ev.store(reinterpret_cast<u32x4*>(L.ev), evs, r4(d.ne) >> 2);
    h_ro.store(as_words(L.ro), ros, words8(d.nvo + 1));
    h_ent.store(as_words(L.ent), ens, words8(nent));
    hv_.store(pos, m, d, [&](uint32_t l, const float (&w)[3]) { L.pos[l] = make_float4(w[0], w[1], w[2], 0.f); });
    __syncthreads();
    // per face: the terms of its half-edges, stored at the half-edge's FE
    // word 2 e + dir (float half dir of edge e's pair)
    float* hc = reinterpret_cast<float*>(L.cot);
    float* hv = reinterpret_cast<float*>(L.vor);
    auto   face = [&](const uint32_t (&x)[3]) {
        uint32_t a[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const uint32_t e = L.ev[x[j] >> 1];
            a[j]             = (x[j] & 1u) ? hi16(e) : lo16(e);
        }
        const float4  q0 = L.pos[a[0]], q1 = L.pos[a[1]], q2 = L.pos[a[2]];
        const FaceCot c  = face_cot(f3{q0.x, q0.y, q0.z}, f3{q1.x, q1.y, q1.z}, f3{q2.x, q2.y, q2.z});
        // slot j runs a_j -> a_{j+1}: opposite corner a_{j+2}, start a_j
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            hc[x[j]] = c.cot[(j + 2) % 3];
            hv[x[j]] = c.vor[j];
        }
    };
#pragma unroll
    for (uint32_t r = 0; r < RF; ++r)
        if (t + r * T < d.nf) {
            uint32_t x[3];
            fw[r].get(x);
            face(x);
        }
    for (uint32_t f = t + RF * T; f < d.nf; f += T) {
        const uint32_t x[3] = {fe[3 * f], fe[3 * f + 1], fe[3 * f + 2]};
        face(x);
    }
    __syncthreads();
    // rows: diagonal and mass (entries in pattern order)
    for (uint32_t v = threadIdx.x; v < d.nvo; v += T) {
        const uint32_t k0 = L.ro[v], k1 = L.ro[v + 1];
        float          sum_w = 0.f, vw = 0.f;
        for (uint32_t k = k0; k < k1; ++k) {
            const uint32_t u = L.ent[k];  // the half-edge leaving v
            const float2   c = L.cot[u >> 1];
            const float    w = c.x + c.y;
            sum_w += ((w >= 0.f) ? w : 0.f) * dt;
            vw += hv[u];
        }
        const float    ms = 1.0f / (0.5f / vw);
        const uint32_t o  = bse + k0 + v;
        if constexpr (CSR) {
            row_ptr[d.vp + v] = static_cast<int32_t>(o);
            col[o]            = static_cast<int32_t>(d.vp + v);
        } else {
            diag[d.vp + v] = ms + sum_w;
        }
        mass[d.vp + v] = ms;
        val[o]         = ms + sum_w;
    }
    if (CSR && threadIdx.x == 0) row_ptr[d.vp + d.nvo] = static_cast<int32_t>(bse + nent + d.nvo);
    // off-diagonal entries, contiguous over the patch's output range
    for (uint32_t k = threadIdx.x; k < nent; k += T) {
        const uint32_t u = L.ent[k], e = u >> 1, x = L.ev[e], v = (u & 1u) ? hi16(x) : lo16(x);
        const float2   c = L.cot[e];
        const float    w = c.x + c.y;
        const uint32_t o = bse + k + v + 1;
        if constexpr (CSR) {
            const uint32_t q = (u & 1u) ? lo16(x) : hi16(x), r = L.rid[max(q, d.nvo) - d.nvo];
            col[o]           = static_cast<int32_t>((q < d.nvo) ? d.vp + q : r);
        }
        val[o] = -(((w >= 0.f) ? w : 0.f) * dt);
    }
}

// Which owned vertices have a ring of one closed fan (the successors of a vertex's
// half-edges -- v -> a of face (v, a, b) is followed by v -> b -- are one cycle
// through all of them): bit per linear vertex into `closed` (cleared before),
// ring[patch] = 1 where one has not. Successors as in k_query_vx_oriented, from the
// FE words alone; a walk of at most K steps per vertex. Needs a consistently
// oriented edge-manifold mesh. (Looking each successor up among the K neighbours
// took 224 ms where a vertex has 2000 of them; the first assembly takes 0.6 now.)
template <uint32_t T>
__global__ __launch_bounds__(T) void k_closed_fans(DevMesh m, const uint32_t* __restrict__ rbase,
                                                   const uint32_t* __restrict__ nbase,
                                                   const uint16_t* __restrict__ roff, const uint16_t* __restrict__ ent,
                                                   uint32_t* __restrict__ closed, uint32_t* __restrict__ ring)
{
    extern __shared__ uint4 smem[];
    const uint32_t  p = blockIdx.x;
    const PatchDesc d = load_desc(m.patch, p);
    Bump            b(reinterpret_cast<char*>(smem));
    uint16_t*       nh = b.alloc<uint16_t>(2 * d.ne);
    const uint16_t* fe = m.fe + 3u * d.f_off;
    for (uint32_t i = threadIdx.x; i < d.ne; i += T) reinterpret_cast<uint32_t*>(nh)[i] = 0xFFFFFFFFu;
    __syncthreads();
    for (uint32_t f = threadIdx.x; f < d.nf; f += T) {
        const uint32_t x[3] = {fe[3 * f], fe[3 * f + 1], fe[3 * f + 2]};
#pragma unroll
        for (uint32_t i = 0; i < 3; ++i) nh[x[i]] = static_cast<uint16_t>(x[(i + 2u) % 3u] ^ 1u);
    }
    __syncthreads();
    const uint16_t* ro = roff + rbase[p];
    for (uint32_t v = threadIdx.x; v < d.nvo; v += T) {
        const uint32_t k0 = ro[v], K = ro[v + 1] - k0;
        uint32_t       steps = 0;
        bool           ok    = K > 0;
        if (ok) {
            const uint32_t s = ent[nbase[p] + k0];  // a half-edge leaving v
            uint32_t       h = s;
            do {
                h = nh[h];
                ++steps;
            } while (h != kInv16 && h != s && steps < K);
            ok = h == s && steps == K;
        }
        const uint32_t lv = d.vp + v;
        if (ok) atomicOr(&closed[lv >> 5], 1u << (lv & 31u));
        else ring[p] = 1u;
    }
}

// LDS carve of the ring-row pass: EV, FE, half-edge successors, global ids,
// column offsets, the owned rows (sorted) and a scratch copy of one row's
// edges per row (ordered into the canonical ring in place).
struct PlanCOTR
{
    uint32_t *ev, *gid, *off, *wave, *slots, *ring;
    uint16_t *fe, *hn;
};
__host__ __device__ inline PlanCOTR plan_cot_ring(Bump& b, uint32_t nv, uint32_t ne, uint32_t nf, uint32_t nvo,
                                                  uint32_t nrow)
{
    PlanCOTR p{};
    p.ev    = b.alloc<uint32_t>(r4(ne));
    p.gid   = b.alloc<uint32_t>(nv);
    p.off   = b.alloc<uint32_t>(nvo + 1);
    p.wave  = b.alloc<uint32_t>(20);
    p.slots = b.alloc<uint32_t>(nrow);
    p.ring  = b.alloc<uint32_t>(nrow);
    p.fe    = b.alloc<uint16_t>(r4(3 * nf));
    p.hn    = b.alloc<uint16_t>(2 * ne);
    return p;
}

// Rows of the vertices whose ring is not one closed fan (flag bit clear in
// `closed`, per linear id), for the patches listed in `plist`: the
// reference's cyclic walk over the canonical oriented ring (wedge (p, r_i,
// r_{i+1}) for every consecutive pair, the last one wrapping to the first),
// each weight written to its neighbour's column of the row k_cot_assemble
// laid out (neighbours ascending by local id of the connecting edge). Positions come from global
// memory: these rows are few.
template <uint32_t T>
__global__ __launch_bounds__(T) void k_cot_ring_rows(DevMesh m, const uint32_t* __restrict__ base,
                                                     const uint32_t* __restrict__ plist,
                                                     const uint32_t* __restrict__ closed,
                                                     const float* __restrict__ pos, float dt,
                                                     float* __restrict__ val, float* __restrict__ mass)
{
    extern __shared__ uint4 smem[];
    const uint32_t  p   = plist[blockIdx.x];
    const PatchDesc d   = load_desc(m.patch, p);
    const uint32_t  bse = base[p], nrow = base[p + 1] - bse;
    Bump            b(reinterpret_cast<char*>(smem));
    const PlanCOTR  L = plan_cot_ring(b, d.nv, d.ne, d.nf, d.nvo, nrow);
    const uint32_t  N = m.nV;
    stage_u32(L.ev, m.ev + d.e_off, d.ne);
    stage_fe(L.fe, m.fe + 3u * d.f_off, d.nf);
    for (uint32_t v = threadIdx.x; v < d.nv; v += T) L.gid[v] = m.ltog_v[d.v_off + v];
    for (uint32_t i = threadIdx.x; i < d.ne; i += T) reinterpret_cast<uint32_t*>(L.hn)[i] = 0xFFFFFFFFu;
    __syncthreads();
    build_half_next(L.fe, L.ev, d.nf, L.hn);
    fill_columns<T>(
        2 * d.ne, d.nvo,
        [&](uint32_t i) {
            const uint32_t x = L.ev[i >> 1];
            return (i & 1u) ? hi16(x) : lo16(x);
        },
        [&](uint32_t i) {
            const uint32_t x = L.ev[i >> 1];
            return ((i >> 1) << 16) | ((i & 1u) ? lo16(x) : hi16(x));
        },
        L.off, L.slots, L.wave);
    if (L.off[d.nvo] + d.nvo != nrow) return;
    for (uint32_t v = threadIdx.x; v < d.nvo; v += T) {
        const uint32_t lv = d.vp + v;
        if ((closed[lv >> 5] >> (lv & 31u)) & 1u) continue;
        const uint32_t k0 = L.off[v], K = L.off[v + 1] - k0;
        sort_row(L.slots + k0, K, [&](uint32_t j, uint32_t s) {
            L.slots[k0 + j] = s;
            L.ring[k0 + j]  = s >> 16;
        });
        orient_ring<12, true>(v, k0, k0 + K, L.ring, L.ring, L.ev, L.hn, L.gid);
        auto P3 = [&](uint32_t l) {
            const uint32_t g = lin_of(l, d.nvo, d.vp, m.v_lin + d.v_off);
            return f3{pos[g], pos[N + g], pos[2 * N + g]};
        };
        // column of neighbour r: its position in the sorted row
        auto rank = [&](uint32_t r) {
            uint32_t c = 0;
            for (uint32_t j = 0; j < K; ++j) c = ((L.slots[k0 + j] & 0xFFFFu) == r) ? j : c;
            return c;
        };
        const uint32_t o  = bse + k0 + v;
        const f3       pp = P3(v);
        float          sum_w = 0.f, vw = 0.f;
        if (K > 0) {
            // wedge i = (p, r_i, r_{i+1}); edge p-r_i takes the angle at
            // r_{i-1} of wedge i-1 and the angle at r_{i+1} of wedge i
            uint32_t    rc = L.ring[k0];
            f3          Pc = P3(rc);
            const Wedge wl = wedge(pp, P3(L.ring[k0 + K - 1]), Pc);
            float       ca_prev = wl.ca;
            vw                  = wl.vor;
            for (uint32_t i = 0; i < K; ++i) {
                uint32_t rn = 0;
                f3       Pn{};
                Wedge    w = wl;
                if (i + 1 < K) {
                    rn = L.ring[k0 + i + 1];
                    Pn = P3(rn);
                    w  = wedge(pp, Pc, Pn);
                    vw += w.vor;
                }
                float wt = ca_prev + w.cb;
                wt       = ((wt >= 0.f) ? wt : 0.f) * dt;
                sum_w += wt;
                val[o + 1 + rank(rc)] = -wt;
                ca_prev = w.ca;
                rc      = rn;
                Pc      = Pn;
            }
        }
        const float ms = 1.0f / (0.5f / vw);
        mass[lv]       = ms;
        val[o]         = ms + sum_w;
    }
}

// ---- SpMV over 3 SoA columns, optionally fused with the explicit MCF step --
// LANES consecutive lanes share a row (rows hold ~7 entries), so the col /
// val loads of a wave are contiguous; partial sums meet through a fixed
// xor-shuffle tree (deterministic).
//   FUSED == false: y = A x
//   FUSED == true : y = x + (M x - A x) / M
template <uint32_t LANES, bool FUSED>
__global__ __launch_bounds__(256) void k_spmv3(uint32_t n, const int32_t* __restrict__ row_ptr,
                                               const int32_t* __restrict__ col, const float* __restrict__ val,
                                               const float* __restrict__ mass, const float* __restrict__ x,
                                               float* __restrict__ y)
{
    const uint32_t gid  = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t row  = gid / LANES;
    const uint32_t lane = gid % LANES;
    float          ax = 0.f, ay = 0.f, az = 0.f;
    const bool     ok = row < n;
    if (ok) {
        const int32_t s = row_ptr[row], e = row_ptr[row + 1];
        for (int32_t k = s + static_cast<int32_t>(lane); k < e; k += LANES) {
            const uint32_t c = static_cast<uint32_t>(col[k]);
            const float    w = val[k];
            ax += w * x[c];
            ay += w * x[n + c];
            az += w * x[2 * n + c];
        }
    }
#pragma unroll
    for (uint32_t o = LANES / 2; o > 0; o >>= 1) {
        ax += __shfl_xor(ax, o, 64);
        ay += __shfl_xor(ay, o, 64);
        az += __shfl_xor(az, o, 64);
    }
    if (ok && lane == 0) {
        if constexpr (FUSED) {
            const float M = mass[row];
            const float px = x[row], py = x[n + row], pz = x[2 * n + row];
            y[row]         = px + (M * px - ax) / M;
            y[n + row]     = py + (M * py - ay) / M;
            y[2 * n + row] = pz + (M * pz - az) / M;
        } else {
            y[row]         = ax;
            y[n + row]     = ay;
            y[2 * n + row] = az;
        }
    }
}

// ---- explicit MCF step, patch-local ------------------------------------------
// y = x + (M x - A x) / M on the mesh's cotangent system (rxm_cot_csr_assemble
// layout: each patch's rows are one contiguous run, diagonal first, then the
// neighbours in VV query order). The pattern is the patch-local VV plan
// (u16 row offsets and local neighbour ids, the same order), so a workgroup
// stages its patch's positions (owned + ribbon), plan rows and the run of
// values in LDS and the matrix's column indices are never read: a row's
// neighbours come from LDS instead of one global gather per entry. Rows sum
// the diagonal term first, then the neighbours in row order.
template <uint32_t T>
__global__ __launch_bounds__(T) void k_mcf_patch(DevMesh m, const uint32_t* __restrict__ vv_base,
                                                 const uint32_t* __restrict__ rbase,
                                                 const uint32_t* __restrict__ nbase,
                                                 const uint16_t* __restrict__ roff, const uint16_t* __restrict__ nbr,
                                                 const float* __restrict__ val, const float* __restrict__ mass,
                                                 const float* __restrict__ x, float* __restrict__ y)
{
    extern __shared__ uint4 smem[];
    const uint32_t p = patch_of_block(m.P);  // XCD-contiguous patch ranges
    if (p >= m.P) return;
    const PatchDesc d    = load_desc(m.patch, p);
    // nbase runs are padded to 8 entries; the system's run is not: nent is
    // the patch's true VV entry count
    const uint32_t  rb   = rbase[p], nbb = nbase[p], nent = vv_base[p + 1] - vv_base[p];
    const uint32_t  bse  = vv_base[p] + d.vp;  // the patch's run in the system
    const uint32_t  N    = m.nV;
    Bump            b(reinterpret_cast<char*>(smem));
    const PlanSL    L = plan_sl(b, d.nv, d.nvo, nent, false);
    float*          wl = b.alloc<float>(nent + d.nvo + 3u);
    const float*    vsrc = val + bse;
    const uint32_t  t = threadIdx.x;
    HeldVerts<T, 3>                     hv;
    HeldFloats<T, (512u + T - 1u) / T>  hw;
    Held<T, (256u + T - 1u) / T, u32x4> h_nb;
    Held<T, 1, u32x4>                   h_ro;
    float                               M[HeldVerts<T, 3>::RO];
    hv.ids(m, d);
    h_ro.load(as_words(roff + rb), words8(d.nvo + 1));
    h_nb.load(as_words(nbr + nbb), words8(nent));
    hw.load(vsrc, nent + d.nvo);
    hv.owned(x, m, d);
#pragma unroll
    for (uint32_t k = 0; k < HeldVerts<T, 3>::RO; ++k)
        if (k == 0 || k * T < d.nvo) M[k] = mass[min(d.vp + t + k * T, N - 1u)];
    hv.ribbon(x, m, d);
    h_ro.store(as_words(L.ro), as_words(roff + rb), words8(d.nvo + 1));
    h_nb.store(as_words(L.nb), as_words(nbr + nbb), words8(nent));
    hw.store(wl, vsrc, nent + d.nvo);
    hv.store(x, m, d, [&](uint32_t l, const float (&q)[3]) {
        L.x[l] = q[0];
        L.y[l] = q[1];
        L.z[l] = q[2];
    });
    const float* w = wl + hw.shift(vsrc);
    __syncthreads();
    auto row = [&](uint32_t v, float Mv) {
        const uint32_t k0 = L.ro[v], k1 = L.ro[v + 1];
        const float*   wr = w + k0 + v;  // diagonal, then the row's neighbours
        const float    px = L.x[v], py = L.y[v], pz = L.z[v];
        float          ax = wr[0] * px, ay = wr[0] * py, az = wr[0] * pz;
        for (uint32_t k = k0; k < k1; ++k) {
            const uint32_t q = L.nb[k];
            const float    c = wr[1 + k - k0];
            ax += c * L.x[q];
            ay += c * L.y[q];
            az += c * L.z[q];
        }
        const uint32_t g = d.vp + v;
        y[g]             = px + (Mv * px - ax) / Mv;
        y[N + g]         = py + (Mv * py - ay) / Mv;
        y[2 * N + g]     = pz + (Mv * pz - az) / Mv;
    };
#pragma unroll
    for (uint32_t k = 0; k < HeldVerts<T, 3>::RO; ++k)
        if (t + k * T < d.nvo) row(t + k * T, M[k]);
    for (uint32_t v = t + HeldVerts<T, 3>::RO * T; v < d.nvo; v += T) row(v, mass[d.vp + v]);
}

// ---- implicit MCF: conjugate gradients on the cotangent system ---------------
// Restates the reference's CGSolver (include/rxmesh/matrix/cg_solver.h:37-125)
// on A X = B with B = M x (apps/MCF/mcf_kernels.cuh:302-352, mcf_B_setup) for
// the three coordinate columns at once: dot products and norms run over all
// 3V entries, as the reference's cuBLAS calls over the whole V x 3 matrix do.
// The loop runs on the device and the host enqueues max_iter iterations of two
// launches without reading anything back:
//   k_cg_apply   sums the update's partials (<r, r>), takes beta and the
//                stopping decision from them, adds the last alpha p to x,
//                forms p = r + beta p and s = A p, partial <s, p> per patch;
//   k_cg_update  sums those partials, takes alpha, r -= alpha s, partial
//                <r, r> per workgroup.
// Every workgroup sums the partials itself, in the same fixed order and in
// FP64, so all of them hold the same scalar, two solves are bit-identical and
// no launch of its own (a single workgroup, 2.5-4.4 us each, twice per
// iteration) stands between the passes. The update runs in at most
// kCgUpdateGroups workgroups so that the product's workgroups have few
// partials to sum. Adding alpha p to x in the product, which has p in
// registers, instead of in the update saves one read of p (12 V bytes).
// Bound: 160 V bytes of vectors and values per iteration from the Infinity
// Cache, and the product's four dependent round trips (descriptor, ids and
// plan, ribbon words, stores). Assembly + 20 iterations, 1201 x 401 torus
// (482k vertices): 647 -> 494 us; an iteration 15.5 + 8.8 and two sums of 4.3 +
// 3.6 us -> 14.5 + 7.7 us.
// Scalars pass through two states: the product reads `upd` and writes `app`,
// the update reads `app` and writes `upd`, so no launch reads what it writes.
struct CgState
{
    float    delta, alpha, beta, start;
    uint32_t iters, done;
};
constexpr uint32_t kCgUpdateThreads = 1024, kCgUpdateGroups = 512;

// component stride of the solver's vectors: whole 256-byte lines
__host__ __device__ inline size_t cg_stride(uint32_t n) { return (size_t(n) + 63u) & ~size_t(63); }

// Sum over the wave, in lane 63: rows of 16 lanes by DPP shifts, then the row
// totals broadcast upwards (a fixed order; no LDS round trip per step).
__device__ __forceinline__ double wave_sum63(double v)
{
    auto step = [&](auto ctrl, auto rows) {
        const uint64_t u = __double_as_longlong(v);
        const uint32_t lo = __builtin_amdgcn_update_dpp(0u, uint32_t(u), decltype(ctrl)::value, decltype(rows)::value, 0xf, false);
        const uint32_t hi = __builtin_amdgcn_update_dpp(0u, uint32_t(u >> 32), decltype(ctrl)::value, decltype(rows)::value, 0xf, false);
        v += __longlong_as_double(static_cast<long long>((uint64_t(hi) << 32) | lo));
    };
    using r1 = std::integral_constant<int, 0x111>;  // row_shr 1, 2, 4, 8
    using r2 = std::integral_constant<int, 0x112>;
    using r4 = std::integral_constant<int, 0x114>;
    using r8 = std::integral_constant<int, 0x118>;
    using b15 = std::integral_constant<int, 0x142>;  // row_bcast 15, 31
    using b31 = std::integral_constant<int, 0x143>;
    using all = std::integral_constant<int, 0xf>;
    step(r1{}, all{});
    step(r2{}, all{});
    step(r4{}, all{});
    step(r8{}, all{});
    step(b15{}, std::integral_constant<int, 0xa>{});
    step(b31{}, std::integral_constant<int, 0xc>{});
    return v;
}

// Sum over the workgroup, the same value in every thread: wave sums, then the
// wave totals in order. red: T / 64 doubles, used once per kernel.
template <uint32_t T>
__device__ __forceinline__ double block_sum(double v, double* red)
{
    v = wave_sum63(v);
    if ((threadIdx.x & 63u) == 63u) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (uint32_t i = 0; i < T / 64u; ++i) t += red[i];
    return t;
}

// States are read and written field by field: a struct copied whole under a
// branch became a private array, which the compiler placed in LDS with the
// workgroup size read from the dispatch packet in host memory by every
// workgroup (the update took 17-20 us instead of 8).
__device__ __forceinline__ CgState cg_load(const CgState* __restrict__ q)
{
    CgState s;
    s.delta = q->delta;
    s.alpha = q->alpha;
    s.beta  = q->beta;
    s.start = q->start;
    s.iters = q->iters;
    s.done  = q->done;
    return s;
}
__device__ __forceinline__ void cg_store(CgState* __restrict__ q, const CgState& s)
{
    q->delta = s.delta;
    q->alpha = s.alpha;
    q->beta  = s.beta;
    q->start = s.start;
    q->iters = s.iters;
    q->done  = s.done;
}

// Scalar step on sum = <r, r> (<r, r / diag> with the preconditioner) after the
// set-up (FIRST) or an update: stop when it is below abs_tol or, relative to
// the start, below rel_tol; else beta = delta / delta_old and one more
// iteration taken.
template <bool FIRST>
__device__ __forceinline__ CgState cg_next(CgState s, double total, float abs_tol, float rel_tol)
{
    const float sum = static_cast<float>(total);
    if constexpr (FIRST) {
        s.start = sum;
        s.iters = 0;
        s.alpha = s.beta = 0.f;
        s.done = (sum < abs_tol || sum / sum < rel_tol) ? 1u : 0u;
    } else if (sum < abs_tol || sum / s.start < rel_tol) {
        s.done = 1u;
    } else {
        s.beta = sum / s.delta;
        s.iters += 1u;
        s.done = 0u;
    }
    s.delta = sum;
    return s;
}

// LDS carve of the product: the plan rows and direction (plan_sl), the values
// (none with uniform weights) and the wave totals.
struct PlanCG
{
    PlanSL  sl;
    float*  w;
    double* red;
};
__host__ __device__ inline PlanCG plan_cg(Bump& b, uint32_t nv, uint32_t nvo, uint32_t nent, bool uniform,
                                          uint32_t threads)
{
    PlanCG p{};
    p.sl  = plan_sl(b, nv, nvo, nent, false);
    p.w   = uniform ? nullptr : b.alloc<float>(nent + nvo + 3u);
    p.red = b.alloc<double>(threads / 64u);
    return p;
}

// MODE 0 (set-up): y = A x, x the caller's start vector (component stride nV).
// MODE 1 (first iteration) / 2: p = z, or z + beta p_old, z = r, or r / diag
// with the Jacobi preconditioner (PRE, the reference's precond_matvec,
// mcf_kernels.cuh:219-299); p written for the owned rows, y = A p, <y, p>
// into partial[patch], and (MODE 2) sol += alpha p_old of the iteration
// before. UNI: uniform weights (off-diagonals -dt, diagonal valence + the
// row's dt), val unread. The pattern is the patch-local VV plan.
template <uint32_t T, int MODE, bool PRE, bool UNI>
__global__ __launch_bounds__(T) void k_cg_apply(DevMesh m, const uint32_t* __restrict__ vv_base,
                                                const uint32_t* __restrict__ rbase,
                                                const uint32_t* __restrict__ nbase,
                                                const uint16_t* __restrict__ roff, const uint16_t* __restrict__ nbr,
                                                const float* __restrict__ val, float dt, const float* __restrict__ x,
                                                const float* __restrict__ r, const float* __restrict__ diag,
                                                float* __restrict__ sol, float* __restrict__ p_new,
                                                float* __restrict__ y, float* __restrict__ partial,
                                                const double* __restrict__ part_in, uint32_t nin,
                                                const CgState* __restrict__ upd, CgState* __restrict__ app,
                                                float abs_tol, float rel_tol)
{
    extern __shared__ uint4 smem[];
    const uint32_t p = patch_of_block(m.P);  // XCD-contiguous patch ranges
    if (p >= m.P) return;
    CgState         st{};
    const PatchDesc d = load_desc(m.patch, p);
    // true VV entry count (nbase runs are padded to 8; the system's run is not)
    const uint32_t rb = rbase[p], nbb = nbase[p], vb = vv_base[p], nent = vv_base[p + 1] - vb;
    if constexpr (MODE == 2) st = cg_load(upd);
    if (MODE == 2 && st.done) return;
    const size_t   N = m.nV, S = cg_stride(m.nV);
    Bump           b(reinterpret_cast<char*>(smem));
    const PlanCG   L  = plan_cg(b, d.nv, d.nvo, nent, UNI, T);
    const uint32_t  t = threadIdx.x, nvo = d.nvo, nr = d.nv - nvo;  // nr: ribbon vertices
    const uint32_t* vl   = m.v_lin + d.v_off;
    const float*    vsrc = UNI ? nullptr : val + vb + d.vp;
    // first round trip: ribbon ids, plan rows, values, partials and the owned
    // vertices' words; second: the ribbon's words. Clamped indices read a
    // valid element whose value is not used.
    constexpr uint32_t         RO = (512u + T - 1u) / T;
    HeldFloats<T, UNI ? 1 : 2> hw;
    Held<T, 1, u32x4>          hro, hnb;
    const uint32_t             nro = (nvo + 1u + 7u) >> 3, nnb = (nent + 7u) >> 3;
    const u32x4 *ros = reinterpret_cast<const u32x4*>(roff + rb), *nbs = reinterpret_cast<const u32x4*>(nbr + nbb);
    const uint32_t gr = vl[min(nvo + t, d.nv - 1u)];
    hro.load(ros, nro);
    hnb.load(nbs, nnb);
    if constexpr (!UNI) hw.load(vsrc, nent + nvo);
    double acc0 = 0.0, acc1 = 0.0;
    if constexpr (MODE != 0) {
        static_assert(2 * T >= kCgUpdateGroups, "two rounds hold every partial");
        acc0 = part_in[min(t, nin - 1u)];
        acc1 = part_in[min(t + T, nin - 1u)];
    }
    float a[RO][3], po[RO][3], xs[RO][3], dg[RO];
#pragma unroll
    for (uint32_t k = 0; k < RO; ++k) {
        if (k * T >= nvo && k) continue;
        const size_t gg = min(d.vp + t + k * T, m.nV - 1u);
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) {
            a[k][c] = (MODE == 0) ? x[c * N + gg] : r[c * S + gg];
            if constexpr (MODE == 2) {
                po[k][c] = x[c * S + gg];  // x holds p_old
                xs[k][c] = sol[c * N + gg];
            }
        }
        if constexpr (MODE != 0 && PRE) dg[k] = diag[gg];
    }
    float ar[3], pr[3], dr = 1.f;
#pragma unroll
    for (uint32_t c = 0; c < 3; ++c) {
        ar[c] = (MODE == 0) ? x[c * N + gr] : r[c * S + gr];
        if constexpr (MODE == 2) pr[c] = x[c * S + gr];
    }
    if constexpr (MODE != 0 && PRE) dr = diag[gr];
    hro.store(reinterpret_cast<u32x4*>(L.sl.ro), ros, nro);
    hnb.store(reinterpret_cast<u32x4*>(L.sl.nb), nbs, nnb);
    uint32_t mis = 0;
    if constexpr (!UNI) {
        hw.store(L.w, vsrc, nent + nvo);
        mis = hw.shift(vsrc);
    }
    if constexpr (MODE != 0) {
        const double acc = (t < nin ? acc0 : 0.0) + (t + T < nin ? acc1 : 0.0);
        st = cg_next<MODE == 1>(st, block_sum<T>(acc, L.red), abs_tol, rel_tol);
        if (p == 0 && t == 0) cg_store(app, st);
    }
    // direction of a vertex from its words into LDS
    const float alpha = st.alpha, beta = st.beta;
    auto        put   = [&](uint32_t l, const float (&av)[3], const float (&pv)[3], float dv) {
        float* const o[3] = {L.sl.x, L.sl.y, L.sl.z};
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) {
            const float z = (MODE != 0 && PRE) ? av[c] / dv : av[c];
            o[c][l]       = (MODE == 2) ? z + beta * pv[c] : z;
        }
    };
    auto finish = [&](size_t gg, const float (&pv)[3], const float (&xv)[3]) {  // the last iteration's step of x
        if constexpr (MODE == 2)
#pragma unroll
            for (uint32_t c = 0; c < 3; ++c) sol[c * N + gg] = xv[c] + alpha * pv[c];
    };
#pragma unroll
    for (uint32_t k = 0; k < RO; ++k)
        if (t + k * T < nvo) {
            finish(d.vp + t + k * T, po[k], xs[k]);
            put(t + k * T, a[k], po[k], dg[k]);
        }
    if (t < nr) put(nvo + t, ar, pr, dr);
    auto direct = [&](uint32_t l, size_t gg, bool owned) {  // vertices beyond the register rounds
        float av[3], pv[3] = {}, xv[3] = {};
        for (uint32_t c = 0; c < 3; ++c) {
            av[c] = (MODE == 0) ? x[c * N + gg] : r[c * S + gg];
            if constexpr (MODE == 2) {
                pv[c] = x[c * S + gg];
                if (owned) xv[c] = sol[c * N + gg];
            }
        }
        if (owned) finish(gg, pv, xv);
        put(l, av, pv, (MODE != 0 && PRE) ? diag[gg] : 1.f);
    };
    for (uint32_t l = t + RO * T; l < nvo; l += T) direct(l, d.vp + l, true);
    for (uint32_t l = nvo + t + T; l < d.nv; l += T) direct(l, vl[l], false);
    if (MODE != 0 && st.done) return;  // converged: x is complete (the same decision in every workgroup)
    __syncthreads();
    float dotp = 0.f;
    for (uint32_t v = t; v < d.nvo; v += T) {
        const uint32_t k0 = L.sl.ro[v], k1 = L.sl.ro[v + 1];
        const float*   wr = L.w + mis + k0 + v;  // diagonal, then the row's neighbours
        const float    px = L.sl.x[v], py = L.sl.y[v], pz = L.sl.z[v];
        float          w0;
        if constexpr (UNI) {
            float sum_w = 0.f;
            for (uint32_t k = k0; k < k1; ++k) sum_w += dt;
            w0 = static_cast<float>(k1 - k0) + sum_w;
        } else {
            w0 = wr[0];
        }
        float ax = w0 * px, ay = w0 * py, az = w0 * pz;
        for (uint32_t k = k0; k < k1; ++k) {
            const uint32_t q = L.sl.nb[k];
            const float    c = UNI ? -dt : wr[1 + k - k0];
            ax += c * L.sl.x[q];
            ay += c * L.sl.y[q];
            az += c * L.sl.z[q];
        }
        const size_t gg = d.vp + v;
        y[gg]           = ax;
        y[S + gg]       = ay;
        y[2 * S + gg]   = az;
        if constexpr (MODE != 0) {
            p_new[gg]         = px;
            p_new[S + gg]     = py;
            p_new[2 * S + gg] = pz;
            dotp += ax * px + ay * py + az * pz;
        }
    }
    if constexpr (MODE != 0) {
        // fixed-order workgroup sum: wave shuffles, then wave totals in order
        // (every thread has read the first sum's totals: a barrier lies between)
        float* red = reinterpret_cast<float*>(L.red);
        for (uint32_t o = 32; o > 0; o >>= 1) dotp += __shfl_xor(dotp, o, 64);
        if ((t & 63u) == 0) red[t >> 6] = dotp;
        __syncthreads();
        if (t == 0) {
            float s = 0.f;
            for (uint32_t i = 0; i < T / 64u; ++i) s += red[i];
            partial[p] = s;
        }
    }
}

// Set-up of the matrix-free solve with uniform weights: mass = valence (the
// reference's init_B scale) and, for the preconditioner, the diagonal the
// product uses.
__global__ __launch_bounds__(256) void k_uniform_diag(DevMesh m, const uint32_t* __restrict__ rbase,
                                                      const uint16_t* __restrict__ roff, float dt,
                                                      float* __restrict__ mass, float* __restrict__ diag)
{
    const uint32_t  p = blockIdx.x;
    const PatchDesc d = load_desc(m.patch, p);
    const uint16_t* ro = roff + rbase[p];
    for (uint32_t v = threadIdx.x; v < d.nvo; v += 256u) {
        const uint32_t k = ro[v + 1] - ro[v];
        float          sum_w = 0.f;
        for (uint32_t i = 0; i < k; ++i) sum_w += dt;
        mass[d.vp + v] = static_cast<float>(k);
        diag[d.vp + v] = static_cast<float>(k) + sum_w;
    }
}

// MODE 0 (set-up): r = b - s with b = mass * x0, x = x0 and the workgroup's
// partial <r, r> (<r, r / diag> with the Jacobi preconditioner, diag
// non-null). MODE 1 (iteration): alpha = delta / <s, p> from the product's
// npart partials, r -= alpha s, partial <r, r>. r and s are the solver's own
// (stride cg_stride, 16-byte quads); the pad past n is masked out.
template <int MODE>
__global__ __launch_bounds__(kCgUpdateThreads) void k_cg_update(uint32_t n, const float* __restrict__ mass,
                                                                const float* __restrict__ x0, float* __restrict__ x,
                                                                float* __restrict__ r, const float* __restrict__ s,
                                                                const float* __restrict__ diag,
                                                                const float* __restrict__ part_in, uint32_t npart,
                                                                double* __restrict__ partial,
                                                                const CgState* __restrict__ app,
                                                                CgState* __restrict__ upd)
{
    constexpr uint32_t T = kCgUpdateThreads;
    __shared__ double  red[2][T / 64u];
    const size_t       S  = cg_stride(n);
    const uint32_t     t0 = blockIdx.x * T + threadIdx.x, step = gridDim.x * T;
    double             acc = 0.0;
    if constexpr (MODE == 0) {
        // b = M x0 rounded on its own (the reference stores B, then forms
        // B - A x): no fused multiply-subtract here
#pragma clang fp contract(off)
        for (uint32_t i = t0; i < n; i += step) {
            const float M = mass[i], D = diag ? diag[i] : 1.f;
#pragma unroll
            for (uint32_t c = 0; c < 3; ++c) {
                const float x0v = x0[c * size_t(n) + i];
                const float v   = M * x0v - s[c * S + i];
                r[c * S + i]    = v;
                x[c * size_t(n) + i] = x0v;
                acc += static_cast<double>(diag ? v * (v / D) : v * v);
            }
        }
    } else {
        CgState st = cg_load(app);
        if (st.done) {  // the product has finished x; pass the decision on
            if (blockIdx.x == 0 && threadIdx.x == 0) cg_store(upd, st);
            return;
        }
        const uint32_t nq = static_cast<uint32_t>(S >> 2);  // quads per component
        float4*        r4 = reinterpret_cast<float4*>(r);
        const float4*  s4 = reinterpret_cast<const float4*>(s);
        // the first quad's loads go out before the partials are summed
        uint32_t     q  = t0;
        const bool   on = q < 3u * nq;
        float4       rv = on ? r4[q] : float4{}, sv = on ? s4[q] : float4{};
        double       sp = 0.0;
        for (uint32_t i = threadIdx.x; i < npart; i += T) sp += static_cast<double>(part_in[i]);
        sp       = block_sum<T>(sp, red[0]);
        st.alpha = st.delta / static_cast<float>(sp);
        if (t0 == 0) cg_store(upd, st);
        const float alpha = st.alpha;
        while (q < 3u * nq) {
            const uint32_t qn = q + step;
            float4         rn{}, sn{};
            if (qn < 3u * nq) {
                rn = r4[qn];
                sn = s4[qn];
            }
            const uint32_t c = (q >= nq ? 1u : 0u) + (q >= 2u * nq ? 1u : 0u), i = 4u * (q - c * nq);
            float          v[4] = {rv.x - alpha * sv.x, rv.y - alpha * sv.y, rv.z - alpha * sv.z, rv.w - alpha * sv.w};
            r4[q]               = make_float4(v[0], v[1], v[2], v[3]);
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                if (i + j < n) acc += static_cast<double>(diag ? v[j] * (v[j] / diag[i + j]) : v[j] * v[j]);
            q  = qn;
            rv = rn;
            sv = sn;
        }
    }
    acc = block_sum<T>(acc, red[1]);
    if (threadIdx.x == 0) partial[blockIdx.x] = acc;
}

// After the last iteration (FIRST: none was asked for): the scalar step on the
// update's partials and, unless an earlier product found the solve converged,
// x += alpha p.
template <bool FIRST>
__global__ __launch_bounds__(256) void k_cg_finish(uint32_t n, const double* __restrict__ part_in, uint32_t nin,
                                                   const float* __restrict__ pvec, float* __restrict__ x,
                                                   const CgState* __restrict__ upd, CgState* __restrict__ app,
                                                   float abs_tol, float rel_tol)
{
    __shared__ double red[4];
    CgState           st{};
    if constexpr (!FIRST) st = cg_load(upd);
    if (!FIRST && st.done) return;
    if (blockIdx.x == 0) {
        double acc = 0.0;
        for (uint32_t i = threadIdx.x; i < nin; i += 256u) acc += part_in[i];
        const CgState e = cg_next<FIRST>(st, block_sum<256>(acc, red), abs_tol, rel_tol);
        if (threadIdx.x == 0) cg_store(app, e);
    }
    if constexpr (!FIRST) {
        const uint32_t i = blockIdx.x * 256u + threadIdx.x;
        const size_t   S = cg_stride(n);
        if (i < n)
#pragma unroll
            for (uint32_t c = 0; c < 3; ++c) x[c * size_t(n) + i] += st.alpha * pvec[c * S + i];
    }
}

// ---- uniform smoothing over a materialised VV CSR ---------------------------
// One Jacobi step x' = x + lambda (mean of row neighbours - x) over the CSR of
// a VV query (linear ids). LANES lanes share a row; fixed xor-tree reduction
// (LANES = 1: the row summed in order).
template <uint32_t LANES>
__global__ __launch_bounds__(256) void k_smooth_csr(uint32_t n, const int32_t* __restrict__ row_ptr,
                                                    const int32_t* __restrict__ col, float lambda,
                                                    const float* __restrict__ x, float* __restrict__ y)
{
    const uint32_t gid  = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t row  = gid / LANES;
    const uint32_t lane = gid % LANES;
    float          sx = 0.f, sy = 0.f, sz = 0.f;
    const bool     ok = row < n;
    int32_t        s = 0, e = 0;
    if (ok) {
        s = row_ptr[row];
        e = row_ptr[row + 1];
        for (int32_t k = s + static_cast<int32_t>(lane); k < e; k += LANES) {
            const uint32_t c = static_cast<uint32_t>(col[k]);
            sx += x[c];
            sy += x[n + c];
            sz += x[2 * n + c];
        }
    }
#pragma unroll
    for (uint32_t o = LANES / 2; o > 0; o >>= 1) {
        sx += __shfl_xor(sx, o, 64);
        sy += __shfl_xor(sy, o, 64);
        sz += __shfl_xor(sz, o, 64);
    }
    if (ok && lane == 0) {
        const float px = x[row], py = x[n + row], pz = x[2 * n + row];
        if (e > s) {
            const float inv = 1.0f / static_cast<float>(e - s);
            y[row]          = px + lambda * (sx * inv - px);
            y[n + row]      = py + lambda * (sy * inv - py);
            y[2 * n + row]  = pz + lambda * (sz * inv - pz);
        } else {
            y[row]         = px;
            y[n + row]     = py;
            y[2 * n + row] = pz;
        }
    }
}

// ---- symmetric Dirichlet ----------------------------------------------------
// Rest shape of a face: apps/Param/param.cu:113-141. Mr is stored SoA over
// linear face ids: Mr[c * F + f], c = (m00, m10, m01, m11), columns b-a, c-a
// in the face's local 2D frame.
struct PlanFV
{
    uint32_t* ev;
    uint16_t* fe;
};
__host__ __device__ inline PlanFV plan_fv(Bump& b, uint32_t ne, uint32_t nf)
{
    PlanFV p{};
    p.ev = b.alloc<uint32_t>(r4(ne));
    p.fe = b.alloc<uint16_t>(r4(3 * nf));
    return p;
}

__global__ __launch_bounds__(kGeomThreads) void k_symdir_rest(DevMesh m, const float* __restrict__ pos,
                                                              float* __restrict__ Mr)
{
    extern __shared__ uint4 smem[];
    const uint32_t  p = blockIdx.x;
    const PatchDesc d = load_desc(m.patch, p);
    Bump            b(reinterpret_cast<char*>(smem));
    const PlanFV    L = plan_fv(b, d.ne, d.nf);
    stage_u32(L.ev, m.ev + d.e_off, d.ne);
    stage_fe(L.fe, m.fe + 3u * d.f_off, d.nf);
    __syncthreads();
    const uint32_t N = m.nV, F = m.nF;
    for (uint32_t f = threadIdx.x; f < d.nfo; f += blockDim.x) {
        f3 P[3];
        for (uint32_t i = 0; i < 3; ++i) {
            const uint32_t g = lin_of(face_vertex(L.fe, L.ev, f, i), d.nvo, d.vp, m.v_lin + d.v_off);
            P[i] = f3{pos[g], pos[N + g], pos[2 * N + g]};
        }
        const f3    e1 = sub(P[1], P[0]), e2 = sub(P[2], P[0]);
        const f3    n  = cross(e1, e2);
        const float l1 = sqrtf(dot(e1, e1));
        const f3    b1 = {e1.x / l1, e1.y / l1, e1.z / l1};
        const f3    t  = cross(n, b1);
        const float lt = sqrtf(dot(t, t));
        const f3    b2 = {t.x / lt, t.y / lt, t.z / lt};
        const uint32_t lf = d.fp + f;
        Mr[lf]         = dot(e1, b1);
        Mr[F + lf]     = 0.f;
        Mr[2 * F + lf] = dot(e2, b1);
        Mr[3 * F + lf] = dot(e2, b2);
    }
}

// Energy and (optionally) corner gradients of one face. uv corners a, b, c;
// R = Mr (m00, m10, m01, m11). Returns FLT_MAX (and zero gradient) for a
// face whose UV triangle is not positively oriented (param.cu:165-168).
// E = A (|J|^2 + |J^-1|^2), J = M R^-1, A = det(R) / 2; for 2x2 J,
// |J^-1|^2 = |J|^2 / det(J)^2. Gradient (closed form):
// dE/dJ = A (2 (1 + 1/d^2) J - 2 |J|^2 / d^3 cof(J)), dE/dM = dE/dJ R^-T.
// a*d - b*c with one rounding error at most a few ulps (Kahan's FMA
// algorithm), so near-degenerate faces keep their relative accuracy
__device__ __forceinline__ float det2(float a, float d, float b, float c)
{
    const float w = b * c;
    const float e = fmaf(-b, c, w);
    const float f = fmaf(a, d, -w);
    return f + e;
}

template <bool GRAD>
__device__ __forceinline__ float symdir_face(const float* a, const float* b, const float* c, const float* R,
                                             float* g /* 6: da, db, dc */)
{
    const float M00 = b[0] - a[0], M10 = b[1] - a[1], M01 = c[0] - a[0], M11 = c[1] - a[1];
    const float dm  = det2(M00, M11, M01, M10);
    if (dm <= 0.f) {
        if (GRAD)
            for (int i = 0; i < 6; ++i) g[i] = 0.f;
        return FLT_MAX;
    }
    const float dr = det2(R[0], R[3], R[2], R[1]);
    const float A  = 0.5f * dr;
    const float i00 = R[3] / dr, i01 = -R[2] / dr, i10 = -R[1] / dr, i11 = R[0] / dr;
    const float J00 = M00 * i00 + M01 * i10, J01 = M00 * i01 + M01 * i11;
    const float J10 = M10 * i00 + M11 * i10, J11 = M10 * i01 + M11 * i11;
    const float n2 = J00 * J00 + J01 * J01 + J10 * J10 + J11 * J11;
    const float dj = dm / dr;  // det J = det M / det R
    const float id2 = 1.0f / (dj * dj);
    if (GRAD) {
        const float s1 = 2.0f * (1.0f + id2), s2 = -2.0f * n2 * id2 / dj;
        const float G00 = A * (s1 * J00 + s2 * J11), G01 = A * (s1 * J01 - s2 * J10);
        const float G10 = A * (s1 * J10 - s2 * J01), G11 = A * (s1 * J11 + s2 * J00);
        const float D00 = G00 * i00 + G01 * i01, D01 = G00 * i10 + G01 * i11;
        const float D10 = G10 * i00 + G11 * i01, D11 = G10 * i10 + G11 * i11;
        g[2] = D00;
        g[3] = D10;
        g[4] = D01;
        g[5] = D11;
        g[0] = -(D00 + D01);
        g[1] = -(D10 + D11);
    }
    return A * (n2 + n2 * id2);
}

// Per owned face energy into energy[linear face]; each workgroup also writes
// its patch's sum (fixed-order tree) into partial[p].
__global__ __launch_bounds__(kGeomThreads) void k_symdir_energy(DevMesh m, const float* __restrict__ Mr,
                                                                const float* __restrict__ uv,
                                                                float* __restrict__ energy,
                                                                float* __restrict__ partial)
{
    extern __shared__ uint4 smem[];
    const uint32_t  p = blockIdx.x;
    const PatchDesc d = load_desc(m.patch, p);
    Bump            b(reinterpret_cast<char*>(smem));
    const PlanFV    L  = plan_fv(b, d.ne, d.nf);
    float*          sr = b.alloc<float>(kGeomThreads);
    stage_u32(L.ev, m.ev + d.e_off, d.ne);
    stage_fe(L.fe, m.fe + 3u * d.f_off, d.nf);
    __syncthreads();
    const uint32_t N = m.nV, F = m.nF;
    float          acc = 0.f;
    for (uint32_t f = threadIdx.x; f < d.nfo; f += blockDim.x) {
        float U[3][2];
        for (uint32_t i = 0; i < 3; ++i) {
            const uint32_t g = lin_of(face_vertex(L.fe, L.ev, f, i), d.nvo, d.vp, m.v_lin + d.v_off);
            U[i][0] = uv[g];
            U[i][1] = uv[N + g];
        }
        const uint32_t lf   = d.fp + f;
        const float    R[4] = {Mr[lf], Mr[F + lf], Mr[2 * F + lf], Mr[3 * F + lf]};
        const float    e    = symdir_face<false>(U[0], U[1], U[2], R, nullptr);
        energy[lf]          = e;
        acc += e;
    }
    sr[threadIdx.x] = acc;
    __syncthreads();
    for (uint32_t s = kGeomThreads / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) sr[threadIdx.x] += sr[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[p] = sr[0];
}

// Fixed-order sum of n floats by one workgroup of 1024 threads, in doubles. A
// chain of latencies: one round trip per 4096 values and a sum over lanes with a
// single barrier: 4.0 us with the ten of a tree in LDS, 1.9 so, at 260 to 1037
// values.
__global__ __launch_bounds__(1024) void k_reduce_sum(uint32_t n, const float* __restrict__ in, float* __restrict__ out)
{
    __shared__ double red[16];
    double            acc = 0.0;
    for (uint32_t i0 = 0; i0 < n; i0 += 4096u) {
        float v[4];
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) v[j] = in[min(i0 + j * 1024u + threadIdx.x, n - 1u)];
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) acc += (i0 + j * 1024u + threadIdx.x < n) ? v[j] : 0.f;
    }
    acc = block_sum<1024>(acc, red);
    if (threadIdx.x == 0) out[0] = static_cast<float>(acc);
}

struct PlanSG
{
    uint32_t *ev, *off, *cur, *wave;
    uint16_t *fe, *fvl, *val;
    float *   u, *v, *gc;
};
__host__ __device__ inline PlanSG plan_sg(Bump& b, uint32_t nv, uint32_t ne, uint32_t nf)
{
    PlanSG p{};
    p.ev   = b.alloc<uint32_t>(r4(ne));
    p.off  = b.alloc<uint32_t>(nv + 1);
    p.cur  = b.alloc<uint32_t>(nv);
    p.wave = b.alloc<uint32_t>(20);
    p.fe   = b.alloc<uint16_t>(r4(3 * nf));
    p.fvl  = b.alloc<uint16_t>(3 * nf);
    p.val  = b.alloc<uint16_t>(3 * nf);
    p.u    = b.alloc<float>(nv);
    p.v    = b.alloc<float>(nv);
    p.gc   = b.alloc<float>(6 * nf);
    return p;
}

// Adjoint of sum_f E_f w.r.t. UV: every local face (owned and ribbon) of the
// patch recomputes its Jacobian and corner gradients into LDS; each owned
// vertex then sums the corners of its VF row in ascending local-face order.
// No global atomics (the reference scatters with atomicAdd,
// include/rxmesh/diff/diff_query_kernel.cuh:275-282). grad = scale * dE/duv,
// scale read from device memory (1 if null).
__global__ __launch_bounds__(kGeomThreads) void k_symdir_grad(DevMesh m, const float* __restrict__ Mr,
                                                              const float* __restrict__ uv,
                                                              const float* __restrict__ scale,
                                                              float* __restrict__ grad)
{
    extern __shared__ uint4 smem[];
    const uint32_t  p = blockIdx.x;
    const PatchDesc d = load_desc(m.patch, p);
    Bump            b(reinterpret_cast<char*>(smem));
    const PlanSG    L = plan_sg(b, d.nv, d.ne, d.nf);
    const uint32_t  T = blockDim.x, N = m.nV, F = m.nF;
    stage_u32(L.ev, m.ev + d.e_off, d.ne);
    stage_fe(L.fe, m.fe + 3u * d.f_off, d.nf);
    for (uint32_t l = threadIdx.x; l < d.nv; l += T) {
        const uint32_t g = lin_of(l, d.nvo, d.vp, m.v_lin + d.v_off);
        L.u[l]           = uv[g];
        L.v[l]           = uv[N + g];
    }
    __syncthreads();
    for (uint32_t f = threadIdx.x; f < d.nf; f += T) {
        float U[3][2];
        for (uint32_t i = 0; i < 3; ++i) {
            const uint32_t l = face_vertex(L.fe, L.ev, f, i);
            L.fvl[3 * f + i] = static_cast<uint16_t>(l);
            U[i][0]          = L.u[l];
            U[i][1]          = L.v[l];
        }
        const uint32_t lf   = lin_of(f, d.nfo, d.fp, m.f_lin + d.f_off);
        const float    R[4] = {Mr[lf], Mr[F + lf], Mr[2 * F + lf], Mr[3 * F + lf]};
        symdir_face<true>(U[0], U[1], U[2], R, L.gc + 6 * f);
    }
    __syncthreads();
    lds_transpose<3>(3 * d.nf, d.nv, [&](uint32_t i) { return static_cast<uint32_t>(L.fvl[i]); }, L.off, L.cur,
                     L.val, L.wave, d.nvo);
    const float sc = scale ? scale[0] : 1.0f;
    for (uint32_t v = threadIdx.x; v < d.nvo; v += T) {
        float gu = 0.f, gv = 0.f;
        for (uint32_t k = L.off[v]; k < L.off[v + 1]; ++k) {
            const uint32_t f = L.val[k];
            const uint32_t c = (L.fvl[3 * f] == v) ? 0u : ((L.fvl[3 * f + 1] == v) ? 1u : 2u);
            gu += L.gc[6 * f + 2 * c];
            gv += L.gc[6 * f + 2 * c + 1];
        }
        grad[d.vp + v]     = sc * gu;
        grad[N + d.vp + v] = sc * gv;
    }
}

// ---- symmetric Dirichlet with 3-D positions as the variable ------------------
// For a closed surface (no UV domain) the current triangle is compared with
// its rest shape directly in 3-D: J = [b-a, c-a] Mr^{-1} is 3x2,
// |J^{-1}|^2 -> |J|^2 / G with G = det(J^T J) = |J0 x J1|^2, so
// E = A |J|^2 (1 + 1/G). Reduces to symdir_face for planar input.
// g receives the 9 corner gradients (da, db, dc); FLT_MAX when G <= 0.
__device__ __forceinline__ float symdir3_face(const f3 a, const f3 b, const f3 c, const float* R, float* g)
{
    const f3    e1 = sub(b, a), e2 = sub(c, a);
    const float dr = det2(R[0], R[3], R[2], R[1]);
    const float A  = 0.5f * dr;
    const float i00 = R[3] / dr, i01 = -R[2] / dr, i10 = -R[1] / dr, i11 = R[0] / dr;
    const f3    J0 = {e1.x * i00 + e2.x * i10, e1.y * i00 + e2.y * i10, e1.z * i00 + e2.z * i10};
    const f3    J1 = {e1.x * i01 + e2.x * i11, e1.y * i01 + e2.y * i11, e1.z * i01 + e2.z * i11};
    const float a00 = dot(J0, J0), a11 = dot(J1, J1), a01 = dot(J0, J1);
    const float n2 = a00 + a11, G = det2(a00, a11, a01, a01);
    if (G <= 0.f) {
        for (int i = 0; i < 9; ++i) g[i] = 0.f;
        return FLT_MAX;
    }
    const float iG = 1.0f / G;
    const float s1 = 2.0f * (1.0f + iG), s2 = -n2 * iG * iG;
    const float q0[3] = {J0.x, J0.y, J0.z}, q1[3] = {J1.x, J1.y, J1.z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float dG0 = 2.0f * (a11 * q0[k] - a01 * q1[k]);
        const float dG1 = 2.0f * (a00 * q1[k] - a01 * q0[k]);
        const float E0 = A * (s1 * q0[k] + s2 * dG0), E1 = A * (s1 * q1[k] + s2 * dG1);
        const float D0 = E0 * i00 + E1 * i01, D1 = E0 * i10 + E1 * i11;
        g[3 + k] = D0;
        g[6 + k] = D1;
        g[k]     = -(D0 + D1);
    }
    return A * n2 * (1.0f + iG);
}

// Work-queue counter reset (a kernel, so graphs hold no memset nodes).
__global__ void k_reset_counter(uint32_t* c) { c[0] = 0u; }
__global__ __launch_bounds__(256) void k_fill_u32(uint32_t n, uint32_t v, uint32_t* __restrict__ dst)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < n) dst[i] = v;
}

// Corner gradients (9 values: da, db, dc) of one face; zero for a degenerate
// face.
__device__ __forceinline__ void symdir3_corners(const f3 a, const f3 b, const f3 c, const float* R, float (&g)[9])
{
    const f3    e1 = sub(b, a), e2 = sub(c, a);
    const float dr = det2(R[0], R[3], R[2], R[1]);
    const float A  = 0.5f * dr;
    const float i00 = R[3] / dr, i01 = -R[2] / dr, i10 = -R[1] / dr, i11 = R[0] / dr;
    const f3    J0 = {e1.x * i00 + e2.x * i10, e1.y * i00 + e2.y * i10, e1.z * i00 + e2.z * i10};
    const f3    J1 = {e1.x * i01 + e2.x * i11, e1.y * i01 + e2.y * i11, e1.z * i01 + e2.z * i11};
    const float a00 = dot(J0, J0), a11 = dot(J1, J1), a01 = dot(J0, J1);
    const float n2 = a00 + a11, G = det2(a00, a11, a01, a01);
    const float iG = 1.0f / G;
    const float s1 = 2.0f * (1.0f + iG), s2 = -n2 * iG * iG;
    const float q0[3] = {J0.x, J0.y, J0.z}, q1[3] = {J1.x, J1.y, J1.z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float E0 = A * (s1 * q0[k] + s2 * 2.0f * (a11 * q0[k] - a01 * q1[k]));
        const float E1 = A * (s1 * q1[k] + s2 * 2.0f * (a00 * q1[k] - a01 * q0[k]));
        const float D0 = E0 * i00 + E1 * i01, D1 = E0 * i10 + E1 * i11;
        g[3 + k] = (G <= 0.f) ? 0.f : D0;
        g[6 + k] = (G <= 0.f) ? 0.f : D1;
        g[k]     = (G <= 0.f) ? 0.f : -(D0 + D1);
    }
}

// LDS carve of the gradient step: the face plan, positions and the corner
// gradients (component c of corner j of face f at g[c][3 f + j]).
struct PlanS3P
{
    uint16_t *fvl, *ro, *vf;
    float *   x, *y, *z, *g[3];
};
__host__ __device__ inline PlanS3P plan_s3p(Bump& b, uint32_t nv, uint32_t nvo, uint32_t nf, uint32_t nent,
                                            bool lean = false)
{
    PlanS3P p{};
    p.fvl = b.alloc<uint16_t>((3 * nf + 7u) & ~7u);
    p.ro  = b.alloc<uint16_t>((nvo + 1u + 7u) & ~7u);
    p.vf  = b.alloc<uint16_t>((nent + 7u) & ~7u);
    p.x   = b.alloc<float>(nv);
    p.y   = b.alloc<float>(nv);
    p.z   = b.alloc<float>(nv);
    for (int c = 0; c < 3; ++c) p.g[c] = lean ? nullptr : b.alloc<float>(3 * nf);
    return p;
}

// x_out = x - eta * dE/dx over the patch-local face plan (GRAD: x_out =
// dE/dx itself, eta unused). Face pass: every local face is evaluated once,
// its rest shape straight from HBM into registers, and stores its nine corner
// gradients in LDS; vertex pass: each owned vertex sums its corners in the
// plan's ascending order. Before, every (vertex, face) pair evaluated the whole
// face (five divisions each, 2.2 times as many evaluations) from rest shapes
// staged in LDS. 24 meshes, 941k faces in 1880 patches: 38.2 -> 16.5 us a
// launch (18.5 with 256 threads, 23.1 with 128). Bound: arithmetic of the face pass and the gathers of the ribbon's
// rest shapes (four words of as many cache lines per ribbon face).
// LEAN: no face pass; every (vertex, face) pair evaluates the face, for patches
// whose corner gradients (36 bytes a face) do not fit LDS. Same results.
template <uint32_t T, bool GRAD = false, bool LEAN = false>
__device__ __forceinline__ void symdir3_plan_patch(const DevMesh& m, uint32_t p, const uint32_t* __restrict__ fbase,
                                                   const uint32_t* __restrict__ rbase,
                                                   const uint32_t* __restrict__ nbase,
                                                   const uint16_t* __restrict__ fvl,
                                                   const uint16_t* __restrict__ roff,
                                                   const uint16_t* __restrict__ vf, const float* __restrict__ Mr,
                                                   float eta, const float* __restrict__ x, float* __restrict__ xo,
                                                   char* smem)
{
    const PatchDesc d   = load_desc(m.patch, p);
    const uint32_t  nb0 = nbase[p], nent = nbase[p + 1] - nb0, fb = fbase[p], rb = rbase[p];
    Bump            b(smem);
    const PlanS3P   L = plan_s3p(b, d.nv, d.nvo, d.nf, nent, LEAN);
    const uint32_t  N = m.nV, F = m.nF, t = threadIdx.x;
    constexpr uint32_t RF = (512u + T - 1u) / T, RG = (256u + T - 1u) / T;  // owned / ribbon faces in registers
    const uint32_t     nfr = d.nf - d.nfo;
    const u32x4 *      s_fvl = as_words(fvl + fb), *s_ro = as_words(roff + rb), *s_vf = as_words(vf + nb0);
    HeldVerts<T, 3>    hv;
    Held<T, (320u + T - 1u) / T, u32x4> h_fvl;
    Held<T, (256u + T - 1u) / T, u32x4> h_vf;
    Held<T, 1, u32x4>                   h_ro;
    uint32_t                            gf[RG];
    float                               Ro[RF][4], Rr[RG][4];
    hv.ids(m, d);
#pragma unroll
    for (uint32_t k = 0; k < RG; ++k)
        if (!LEAN && (k == 0 || k * T < nfr)) gf[k] = m.f_lin[d.f_off + min(d.nfo + t + k * T, d.nf - 1u)];
    h_fvl.load(s_fvl, words8(3 * d.nf));
    h_ro.load(s_ro, words8(d.nvo + 1));
    h_vf.load(s_vf, words8(nent));
    hv.owned(x, m, d);
#pragma unroll
    for (uint32_t k = 0; k < RF; ++k)
        if (!LEAN && (k == 0 || k * T < d.nfo))
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) Ro[k][c] = Mr[size_t(c) * F + min(d.fp + t + k * T, F - 1u)];
    hv.ribbon(x, m, d);
#pragma unroll
    for (uint32_t k = 0; k < RG; ++k)
        if (!LEAN && (k == 0 || k * T < nfr))
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) Rr[k][c] = Mr[size_t(c) * F + gf[k]];
    h_fvl.store(as_words(L.fvl), s_fvl, words8(3 * d.nf));
    h_ro.store(as_words(L.ro), s_ro, words8(d.nvo + 1));
    h_vf.store(as_words(L.vf), s_vf, words8(nent));
    hv.store(x, m, d, [&](uint32_t l, const float (&w)[3]) {
        L.x[l] = w[0];
        L.y[l] = w[1];
        L.z[l] = w[2];
    });
    __syncthreads();
    auto corners = [&](uint32_t f, const float (&R)[4], float (&g)[9]) {
        f3 P[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const uint32_t q = L.fvl[3 * f + j];
            P[j]             = f3{L.x[q], L.y[q], L.z[q]};
        }
        symdir3_corners(P[0], P[1], P[2], R, g);
    };
    auto rest = [&](uint32_t f, float (&R)[4]) {
        const size_t lf = lin_of(f, d.nfo, d.fp, m.f_lin + d.f_off);
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) R[c] = Mr[size_t(c) * F + lf];
    };
    if constexpr (!LEAN) {
        auto face = [&](uint32_t f, const float (&R)[4]) {
            float g[9];
            corners(f, R, g);
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int c = 0; c < 3; ++c) L.g[c][3 * f + j] = g[3 * j + c];
        };
#pragma unroll
        for (uint32_t k = 0; k < RF; ++k)
            if (t + k * T < d.nfo) face(t + k * T, Ro[k]);
#pragma unroll
        for (uint32_t k = 0; k < RG; ++k)
            if (t + k * T < nfr) face(d.nfo + t + k * T, Rr[k]);
        auto direct = [&](uint32_t f) {  // faces beyond the register rounds
            float R[4];
            rest(f, R);
            face(f, R);
        };
        for (uint32_t f = t + RF * T; f < d.nfo; f += T) direct(f);
        for (uint32_t f = d.nfo + t + RG * T; f < d.nf; f += T) direct(f);
        __syncthreads();
    }
    auto vertex = [&](uint32_t v, const float (&w)[3]) {
        float gx = 0.f, gy = 0.f, gz = 0.f;
        for (uint32_t k = L.ro[v]; k < L.ro[v + 1]; ++k) {
            const uint32_t s = L.vf[k], f = s >> 2, c = s & 3u;  // corner c of face f
            if constexpr (LEAN) {
                float R[4], g[9];
                rest(f, R);
                corners(f, R, g);
                gx += (c == 0u) ? g[0] : ((c == 1u) ? g[3] : g[6]);
                gy += (c == 0u) ? g[1] : ((c == 1u) ? g[4] : g[7]);
                gz += (c == 0u) ? g[2] : ((c == 1u) ? g[5] : g[8]);
            } else {
                gx += L.g[0][3u * f + c];
                gy += L.g[1][3u * f + c];
                gz += L.g[2][3u * f + c];
            }
        }
        const uint32_t gg = d.vp + v;
        xo[gg]                 = GRAD ? gx : w[0] - eta * gx;
        xo[size_t(N) + gg]     = GRAD ? gy : w[1] - eta * gy;
        xo[2 * size_t(N) + gg] = GRAD ? gz : w[2] - eta * gz;
    };
#pragma unroll
    for (uint32_t k = 0; k < HeldVerts<T, 3>::RO; ++k)
        if (t + k * T < d.nvo) vertex(t + k * T, hv.o[k]);
    for (uint32_t v = t + HeldVerts<T, 3>::RO * T; v < d.nvo; v += T) {
        const float w[3] = {L.x[v], L.y[v], L.z[v]};
        vertex(v, w);
    }
}

template <uint32_t T, bool LEAN = false>
__global__ __launch_bounds__(T) void k_symdir3_step_plan(DevMesh m, const uint32_t* __restrict__ fbase,
                                                         const uint32_t* __restrict__ rbase,
                                                         const uint32_t* __restrict__ nbase,
                                                         const uint16_t* __restrict__ fvl,
                                                         const uint16_t* __restrict__ roff,
                                                         const uint16_t* __restrict__ vf, const float* __restrict__ Mr,
                                                         float eta, const float* __restrict__ x, float* __restrict__ xo)
{
    extern __shared__ uint4 smem[];
    const uint32_t p = patch_of_block(m.P);  // XCD-contiguous patch ranges
    if (p >= m.P) return;
    symdir3_plan_patch<T, false, LEAN>(m, p, fbase, rbase, nbase, fvl, roff, vf, Mr, eta, x, xo,
                          reinterpret_cast<char*>(smem));
}

// grad = dE/dx (3 x V SoA) over the face plan, one workgroup per patch.
template <uint32_t T, bool LEAN = false>
__global__ __launch_bounds__(T) void k_symdir3_grad_plan(DevMesh m, const uint32_t* __restrict__ fbase,
                                                         const uint32_t* __restrict__ rbase,
                                                         const uint32_t* __restrict__ nbase,
                                                         const uint16_t* __restrict__ fvl,
                                                         const uint16_t* __restrict__ roff,
                                                         const uint16_t* __restrict__ vf, const float* __restrict__ Mr,
                                                         const float* __restrict__ x, float* __restrict__ grad)
{
    extern __shared__ uint4 smem[];
    const uint32_t p = patch_of_block(m.P);  // XCD-contiguous patch ranges
    if (p >= m.P) return;
    symdir3_plan_patch<T, true, LEAN>(m, p, fbase, rbase, nbase, fvl, roff, vf, Mr, 0.f, x, grad,
                                reinterpret_cast<char*>(smem));
}

// Persistent form: a grid sized to the machine pulls patch ids from a global
// work queue (one atomic ticket per patch, counter cleared by k_reset_counter
// before the launch); every workgroup exits once the queue is drained.
template <uint32_t T>
__global__ __launch_bounds__(T) void k_symdir3_step_plan_queue(
    DevMesh m, uint32_t* __restrict__ queue, const uint32_t* __restrict__ fbase, const uint32_t* __restrict__ rbase,
    const uint32_t* __restrict__ nbase, const uint16_t* __restrict__ fvl, const uint16_t* __restrict__ roff,
    const uint16_t* __restrict__ vf, const float* __restrict__ Mr, float eta, const float* __restrict__ x,
    float* __restrict__ xo)
{
    extern __shared__ uint4 smem[];
    __shared__ uint32_t s_p;
    while (true) {
        if (threadIdx.x == 0) s_p = atomicAdd(queue, 1u);
        __syncthreads();
        const uint32_t p = s_p;
        __syncthreads();
        if (p >= m.P) break;
        symdir3_plan_patch<T>(m, p, fbase, rbase, nbase, fvl, roff, vf, Mr, eta, x, xo, reinterpret_cast<char*>(smem));
        __syncthreads();
    }
}

// Per-face 3-D symmetric Dirichlet energy of owned faces (FLT_MAX if degenerate).
__global__ __launch_bounds__(kGeomThreads) void k_symdir3_energy(DevMesh m, const float* __restrict__ Mr,
                                                                 const float* __restrict__ x,
                                                                 float* __restrict__ energy)
{
    extern __shared__ uint4 smem[];
    const uint32_t  p = blockIdx.x;
    const PatchDesc d = load_desc(m.patch, p);
    Bump            b(reinterpret_cast<char*>(smem));
    const PlanFV    L = plan_fv(b, d.ne, d.nf);
    stage_u32(L.ev, m.ev + d.e_off, d.ne);
    stage_fe(L.fe, m.fe + 3u * d.f_off, d.nf);
    __syncthreads();
    const uint32_t N = m.nV, F = m.nF;
    for (uint32_t f = threadIdx.x; f < d.nfo; f += blockDim.x) {
        f3 P[3];
        for (uint32_t i = 0; i < 3; ++i) {
            const uint32_t g = lin_of(face_vertex(L.fe, L.ev, f, i), d.nvo, d.vp, m.v_lin + d.v_off);
            P[i] = f3{x[g], x[N + g], x[2 * N + g]};
        }
        const uint32_t lf   = d.fp + f;
        const float    R[4] = {Mr[lf], Mr[F + lf], Mr[2 * F + lf], Mr[3 * F + lf]};
        float          gdummy[9];
        energy[lf] = symdir3_face(P[0], P[1], P[2], R, gdummy);
    }
}

}  // namespace rxm
