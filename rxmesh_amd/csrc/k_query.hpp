// Query kernels: materialise any of the 8 relations as a CSR over linear ids.
//
// One workgroup per patch. Reference behaviour: query<op>
// (include/rxmesh/kernels/rxmesh_queries.cuh:861-1053) and the iterator's
// owner resolution (include/rxmesh/iterator.cuh:117-143). Rows are the owned
// source elements of the patch (linear ids prefix[p] + local); entries are the
// target elements' linear ids, i.e. always the owner's copy.
#pragma once
#include "lds_sort.hpp"
#include "orient.hpp"

namespace rxm {

constexpr uint32_t kQueryThreads = 256;

// FE words of a thread's faces, addresses clamped to the last face
template <uint32_t T, uint32_t RF>
__device__ __forceinline__ void load_faces(FaceWords (&fw)[RF], const uint16_t* __restrict__ fe, uint32_t nf)
{
#pragma unroll
    for (uint32_t r = 0; r < RF; ++r)
        if (r == 0 || r * T < nf) fw[r].load(fe, min(threadIdx.x + r * T, nf - 1u));
}

// ---- oriented VV / VE ----------------------------------------------------------
// LDS carve: EV slab, per half-edge the next one around its start, per owned
// vertex the best start (u64) and the row offset, the rows (nrow = entries of
// the patch's owned rows), global ids of the local vertices and linear ids of
// the ribbon's elements the rows list.
constexpr uint32_t kSeveralFans = 19;  // word of PlanVXO::wave past what the scan uses: some vertex has several fans
struct PlanVXO
{
    uint64_t* start;
    uint32_t *ev, *nh, *off, *wave, *gid, *rid;
    uint16_t* rows;
};
__host__ __device__ inline PlanVXO plan_vxo(Bump& b, uint32_t nv, uint32_t ne, uint32_t nvo, uint32_t nrow,
                                            uint32_t nrid)
{
    PlanVXO p{};
    p.start = b.alloc<uint64_t>(nvo);
    p.ev    = b.alloc<uint32_t>(r4(ne));
    p.nh    = b.alloc<uint32_t>(ne);
    p.off   = b.alloc<uint32_t>(nvo + 1);
    p.wave  = b.alloc<uint32_t>(20);
    p.gid   = b.alloc<uint32_t>(nv);
    p.rid   = b.alloc<uint32_t>(nrid + 1u);  // at least one: read at clamped indices
    p.rows  = b.alloc<uint16_t>(nrow);
    return p;
}

struct PlanFX
{
    uint32_t* ev;
    uint16_t* fe;
};
__host__ __device__ inline PlanFX plan_fx(Bump& b, uint32_t ne, uint32_t nf)
{
    PlanFX p{};
    p.ev = b.alloc<uint32_t>(r4(ne));
    p.fe = b.alloc<uint16_t>(r4(3 * nf));
    return p;
}

// The ring of a vertex of several fans, or whose fan does not start where the
// rule says: L.rows holds the half-edges leaving it, in any order; the rule of
// orient_ring_lds (selection of a start among the edges left, walk, restart),
// whose result does not depend on theirs.
template <bool NBR>
__device__ inline void ring_by_selection(uint32_t k0, uint32_t k1, const PlanVXO& L)
{
    const uint16_t* ev16 = reinterpret_cast<const uint16_t*>(L.ev);
    const uint16_t* nh   = reinterpret_cast<const uint16_t*>(L.nh);
    auto nbr       = [&](uint32_t h) { return static_cast<uint32_t>(ev16[h ^ 1u]); };
    auto startable = [&](uint32_t h) { return nh[h] != kInv16 && nh[h ^ 1u] == kInv16; };
    uint32_t pos = k0;
    while (pos < k1) {
        uint32_t best = pos;
        for (uint32_t j = pos + 1; j < k1; ++j) {
            const uint32_t hj = L.rows[j], hb = L.rows[best];
            const bool     sj = startable(hj), sb = startable(hb);
            if ((sj && !sb) || (sj == sb && L.gid[nbr(hj)] < L.gid[nbr(hb)])) best = j;
        }
        uint16_t x   = L.rows[pos];
        L.rows[pos]  = L.rows[best];
        L.rows[best] = x;
        while (true) {
            const uint32_t q = nh[L.rows[pos]];
            uint32_t       j = pos + 1;
            while (j < k1 && L.rows[j] != q) ++j;
            if (q == kInv16 || j >= k1) break;
            x               = L.rows[pos + 1];
            L.rows[pos + 1] = L.rows[j];
            L.rows[j]       = x;
            ++pos;
        }
        ++pos;
    }
    for (uint32_t k = k0; k < k1; ++k) {
        const uint32_t h = L.rows[k];
        L.rows[k]        = static_cast<uint16_t>(NBR ? nbr(h) : h >> 1);
    }
}

// Oriented VV (IS_VV) or VE: every owned vertex's canonical CCW ring (the rule is
// orient.hpp's). Face slot i holds half-edge fv[i] -> fv[i+1]; the one after it
// around fv[i] is the reverse of slot i + 2, so the FE words alone give every
// half-edge its successor (one LDS store per slot). The start -- an edge the walk
// can proceed from and no face precedes, else the smallest global id -- is one
// 64-bit LDS minimum per half-edge over (not startable, neighbour's global id,
// half-edge); the ring is then one LDS read per entry along the successors.
// Sorting each row and matching successors against it in registers took 43.7 us
// on 654k vertices and 110 on 2.6M; this takes 19.0 and 46. Bound: LDS (random
// minima and adds). A vertex the walk does not
// exhaust (several fans) takes ring_by_selection; where a patch has any, the
// workgroup first collects their half-edges in one pass (a thread that looked for
// its row's by itself held up the launch: two tori glued at one vertex, 358
// patches, 29 us with rows matched in registers, 199 so, 23 now). Needs ne < 2^15
// and a consistently oriented edge-manifold mesh (checked on the host).
template <uint32_t T, bool IS_VV>
__global__ __launch_bounds__(T) void k_query_vx_oriented(DevMesh m, uint32_t nrid, const uint32_t* __restrict__ base,
                                                         int32_t* __restrict__ row_ptr, int32_t* __restrict__ col)
{
    extern __shared__ uint4 smem[];
    const uint32_t p = patch_of_block(m.P);  // XCD-contiguous patch ranges
    if (p >= m.P) return;
    const PatchDesc d   = load_desc(m.patch, p);
    const uint32_t  bse = base[p], nent = base[p + 1] - bse;
    Bump            b(reinterpret_cast<char*>(smem));
    const PlanVXO   L = plan_vxo(b, d.nv, d.ne, d.nvo, nent, nrid);
    const uint32_t  t = threadIdx.x, nvo = d.nvo;
    const uint16_t* fe  = m.fe + 3u * d.f_off;
    const u32x4*    evs = reinterpret_cast<const u32x4*>(m.ev + d.e_off);
    const uint32_t* gs  = m.ltog_v + d.v_off;
    const uint32_t  no = IS_VV ? nvo : d.neo, nr = (IS_VV ? d.nv : d.ne) - no, pre = IS_VV ? d.vp : d.ep;
    const uint32_t* rs = (IS_VV ? m.v_lin + d.v_off : m.e_lin + d.e_off) + no;
    FaceWords                              fw[(768u + T - 1u) / T];
    Held<T, (384u + T - 1u) / T, u32x4>    h_ev;
    Held<T, (512u + T - 1u) / T, uint32_t> h_gid;
    Held<T, (256u + T - 1u) / T, uint32_t> h_rid;
    h_ev.load(evs, r4(d.ne) >> 2);
    load_faces<T>(fw, fe, d.nf);
    h_gid.load(gs, d.nv);
    h_rid.load(rs, nr);
    for (uint32_t i = t; i < d.ne; i += T) L.nh[i] = 0xFFFFFFFFu;
    for (uint32_t v = t; v < nvo; v += T) L.start[v] = ~0ull;
    for (uint32_t v = t; v <= nvo; v += T) L.off[v] = 0u;
    if (t == 0) L.wave[kSeveralFans] = 0u;
    h_ev.store(reinterpret_cast<u32x4*>(L.ev), evs, r4(d.ne) >> 2);
    h_gid.store(L.gid, gs, d.nv);
    h_rid.store(L.rid, rs, nr);
    __syncthreads();
    uint16_t* nh = reinterpret_cast<uint16_t*>(L.nh);
    auto face = [&](const uint32_t (&x)[3]) {
#pragma unroll
        for (uint32_t i = 0; i < 3; ++i) nh[x[i]] = static_cast<uint16_t>(x[(i + 2u) % 3u] ^ 1u);
    };
#pragma unroll
    for (uint32_t r = 0; r < (768u + T - 1u) / T; ++r)
        if (t + r * T < d.nf) {
            uint32_t x[3];
            fw[r].get(x);
            face(x);
        }
    for (uint32_t f = t + (768u + T - 1u) / T * T; f < d.nf; f += T) {
        const uint32_t x[3] = {fe[3 * f], fe[3 * f + 1], fe[3 * f + 2]};
        face(x);
    }
    __syncthreads();
    for (uint32_t e = t; e < d.ne; e += T) {
        const uint32_t x = L.ev[e], n = L.nh[e];
        const bool     f0 = lo16(n) != kInv16, f1 = hi16(n) != kInv16;  // half-edge 2 e / 2 e + 1 has a face
        auto half = [&](uint32_t v, uint32_t q, uint32_t h, bool startable) {
            if (v >= nvo) return;
            const uint64_t key = (uint64_t(startable ? 0u : 1u) << 63) | (uint64_t(L.gid[q]) << 16) | h;
            atomicMin(reinterpret_cast<unsigned long long*>(&L.start[v]), static_cast<unsigned long long>(key));
            atomicAdd(&L.off[v + 1u], 1u);
        };
        half(lo16(x), hi16(x), 2u * e, f0 && !f1);
        half(hi16(x), lo16(x), 2u * e + 1u, f1 && !f0);
    }
    const uint32_t total = scan_excl<T>(L.off + 1, nvo, L.wave);  // off[v + 1] = start of row v
    // the host's row counts (global valences) match the patch's owned
    // columns on every manifold patch; anything else leaves it unwritten
    if (total != nent) return;
    const uint16_t* ev16 = reinterpret_cast<const uint16_t*>(L.ev);
    auto            row0 = [&](uint32_t v) { return L.off[v + 1u]; };
    auto            row1 = [&](uint32_t v) { return v + 1u < nvo ? L.off[v + 2u] : nent; };
    for (uint32_t v = t; v < nvo; v += T) {
        const uint32_t k0 = row0(v), k1 = row1(v);
        const uint32_t s = static_cast<uint32_t>(L.start[v]) & 0xFFFFu;
        uint32_t       h = s, k = k0;
        L.start[v] = ~0ull;
        if (k0 >= k1) continue;
        do {
            L.rows[k++] = static_cast<uint16_t>(IS_VV ? static_cast<uint32_t>(ev16[h ^ 1u]) : h >> 1);
            h           = nh[h];
        } while (k < k1 && h != kInv16 && h != s);
        if (k < k1) {  // several fans: a cursor into the row (no other value is that small)
            L.start[v]           = 0ull;
            L.wave[kSeveralFans] = 1u;
        }
    }
    __syncthreads();
    if (L.wave[kSeveralFans]) {  // uniform
        auto several = [&](uint32_t v) { return L.start[v] != ~0ull; };
        for (uint32_t i = t; i < 2u * d.ne; i += T) {  // half-edge i leaves vertex ev16[i]
            const uint32_t v = ev16[i];
            if (v < nvo && several(v))
                L.rows[row0(v) + static_cast<uint32_t>(
                                     atomicAdd(reinterpret_cast<unsigned long long*>(&L.start[v]), 1ull))] =
                    static_cast<uint16_t>(i);
        }
        __syncthreads();
        for (uint32_t v = t; v < nvo; v += T)
            if (several(v)) ring_by_selection<IS_VV>(row0(v), row1(v), L);
        __syncthreads();
    }
    for (uint32_t v = t; v < nvo; v += T) row_ptr[d.vp + v] = static_cast<int32_t>(bse + row0(v));
    if (t == 0) row_ptr[d.vp + nvo] = static_cast<int32_t>(bse + nent);
    for (uint32_t k = t; k < nent; k += T) {
        const uint32_t x = L.rows[k], r = L.rid[max(x, no) - no];
        col[bse + k]     = static_cast<int32_t>((x < no) ? pre + x : r);
    }
}

// Fixed-width relations EV (2), FV (3), FE (3); OP as in the reference enum.
template <int OP>
__global__ __launch_bounds__(kQueryThreads) void k_query_fixed(DevMesh m, int32_t* __restrict__ row_ptr,
                                                               int32_t* __restrict__ col)
{
    extern __shared__ uint4 smem[];
    const uint32_t  p = blockIdx.x;
    const PatchDesc d = load_desc(m.patch, p);
    Bump            b(reinterpret_cast<char*>(smem));
    const PlanFX    L = plan_fx(b, d.ne, d.nf);
    const uint32_t  T = blockDim.x;
    if constexpr (OP == 9) {  // EV
        for (uint32_t e = threadIdx.x; e < d.neo; e += T) {
            const uint32_t x = m.ev[d.e_off + e], r = d.ep + e;
            row_ptr[r]       = static_cast<int32_t>(2 * r);
            col[2 * r]       = static_cast<int32_t>(lin_of(lo16(x), d.nvo, d.vp, m.v_lin + d.v_off));
            col[2 * r + 1]   = static_cast<int32_t>(lin_of(hi16(x), d.nvo, d.vp, m.v_lin + d.v_off));
        }
        if (p + 1 == m.P && threadIdx.x == 0) row_ptr[d.ep + d.neo] = static_cast<int32_t>(2 * (d.ep + d.neo));
    } else {
        if constexpr (OP == 6) stage_u32(L.ev, m.ev + d.e_off, d.ne);
        stage_fe(L.fe, m.fe + 3u * d.f_off, d.nf);
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < 3 * d.nfo; i += T) {
            const uint32_t r = d.fp + i / 3;
            uint32_t       out;
            if constexpr (OP == 6) out = lin_of(face_vertex(L.fe, L.ev, i / 3, i % 3), d.nvo, d.vp, m.v_lin + d.v_off);
            else out = lin_of(L.fe[i] >> 1, d.neo, d.ep, m.e_lin + d.e_off);
            col[3 * d.fp + i] = static_cast<int32_t>(out);
            if (i % 3 == 0) row_ptr[r] = static_cast<int32_t>(3 * r);
        }
        if (p + 1 == m.P && threadIdx.x == 0) row_ptr[d.fp + d.nfo] = static_cast<int32_t>(3 * (d.fp + d.nfo));
    }
}

// EVDiamond (reference e_v_diamond, rxmesh_queries.cuh:198-265): per owned
// edge [v0, the vertex closing the face that runs v0 -> v1, v1, the vertex
// closing the face that runs v1 -> v0] as linear vertex ids (v0 = lo16 of EV,
// the larger global id), -1 where the edge has no such face. Every local face
// slot names its start vertex as the opposite of the face's next slot, which
// lands in position 1 + 2 dir of that slot's edge. Owned edges' slots take a
// u32 LDS atomicMax over (face + 1) << 16 | vertex: where two faces run an
// edge the same way (non-manifold input) the larger local face index wins,
// as in a serial pass over the faces, independent of scheduling.
struct PlanEVD
{
    uint32_t *ev, *opp, *rid;
};
__host__ __device__ inline PlanEVD plan_evd(Bump& b, uint32_t nv, uint32_t ne, uint32_t nvo, uint32_t neo)
{
    PlanEVD p{};
    p.ev  = b.alloc<uint32_t>(r4(ne));
    p.opp = b.alloc<uint32_t>(2 * neo);
    p.rid = b.alloc<uint32_t>(nv - nvo + 1u);  // at least one: read at clamped indices
    return p;
}

// Opposite vertices of the patch's owned edges into opp (2 neo u32: 0 or
// (face + 1) << 16 | vertex; cleared and EV staged before a barrier by the
// caller, complete after the caller's next one). Faces come as FE words in
// registers (FaceWords), fe the patch's slab for those beyond.
template <uint32_t T, uint32_t RF>
__device__ __forceinline__ void edge_opposites(const FaceWords (&fw)[RF], const uint16_t* __restrict__ fe,
                                               const uint32_t* ev, const PatchDesc& d, uint32_t* opp)
{
    auto face = [&](uint32_t f, const uint32_t (&x)[3]) {
#pragma unroll
        for (uint32_t k = 0; k < 3; ++k) {
            const uint32_t y = x[(k + 1u) % 3u];  // the slot after k runs opposite k's start vertex
            if ((y >> 1) < d.neo) {
                const uint32_t e = ev[x[k] >> 1];
                atomicMax(&opp[y], ((f + 1u) << 16) | ((x[k] & 1u) ? hi16(e) : lo16(e)));
            }
        }
    };
#pragma unroll
    for (uint32_t r = 0; r < RF; ++r)
        if (threadIdx.x + r * T < d.nf) {
            uint32_t x[3];
            fw[r].get(x);
            face(threadIdx.x + r * T, x);
        }
    for (uint32_t f = threadIdx.x + RF * T; f < d.nf; f += T) {
        const uint32_t x[3] = {fe[3 * f], fe[3 * f + 1], fe[3 * f + 2]};
        face(f, x);
    }
}

// Rows leave as one 16-byte store per edge; vertex ids of the ribbon are staged
// (owned ids follow from the prefix); FE goes to registers and is read per face
// (no division per corner). 654k vertices 21.3 -> 11.8 us, 2.6M 65 -> 36; bound by
// the 20 bytes written per edge.
template <uint32_t T>
__global__ __launch_bounds__(T) void k_query_evd(DevMesh m, int32_t* __restrict__ row_ptr, int32_t* __restrict__ col)
{
    extern __shared__ uint4 smem[];
    const uint32_t p = patch_of_block(m.P);  // XCD-contiguous patch ranges
    if (p >= m.P) return;
    const PatchDesc d = load_desc(m.patch, p);
    Bump            b(reinterpret_cast<char*>(smem));
    const PlanEVD   L  = plan_evd(b, d.nv, d.ne, d.nvo, d.neo);
    const uint32_t  t  = threadIdx.x, nr = d.nv - d.nvo;
    const uint16_t* fe = m.fe + 3u * d.f_off;
    const u32x4*    evs = reinterpret_cast<const u32x4*>(m.ev + d.e_off);
    const uint32_t* vr  = m.v_lin + d.v_off + d.nvo;
    FaceWords                              fw[(768u + T - 1u) / T];
    Held<T, (384u + T - 1u) / T, u32x4>    h_ev;
    Held<T, (256u + T - 1u) / T, uint32_t> h_rid;
    h_ev.load(evs, r4(d.ne) >> 2);
    load_faces<T>(fw, fe, d.nf);
    h_rid.load(vr, nr);
    for (uint32_t i = t; i < 2 * d.neo; i += T) L.opp[i] = 0u;
    h_ev.store(reinterpret_cast<u32x4*>(L.ev), evs, r4(d.ne) >> 2);
    h_rid.store(L.rid, vr, nr);
    __syncthreads();
    edge_opposites<T>(fw, fe, L.ev, d, L.opp);
    __syncthreads();
    auto lin = [&](uint32_t q) {
        const uint32_t r = L.rid[max(q, d.nvo) - d.nvo];
        return static_cast<int32_t>((q < d.nvo) ? d.vp + q : r);
    };
    const bool wide = (reinterpret_cast<uintptr_t>(col) & 15u) == 0;  // uniform
    for (uint32_t e = t; e < d.neo; e += T) {
        const uint32_t x = L.ev[e], r = d.ep + e, a = L.opp[2 * e], c = L.opp[2 * e + 1];
        row_ptr[r]       = static_cast<int32_t>(4 * r);
        const int32_t o[4] = {lin(lo16(x)), a ? lin(a & 0xFFFFu) : -1, lin(hi16(x)), c ? lin(c & 0xFFFFu) : -1};
        if (wide) {
            reinterpret_cast<u32x4*>(col)[r] =
                u32x4{uint32_t(o[0]), uint32_t(o[1]), uint32_t(o[2]), uint32_t(o[3])};
        } else {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) col[4 * size_t(r) + j] = o[j];
        }
    }
    if (p + 1 == m.P && t == 0) row_ptr[d.ep + d.neo] = static_cast<int32_t>(4 * (d.ep + d.neo));
}

}  // namespace rxm
