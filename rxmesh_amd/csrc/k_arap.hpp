// ARAP-style deformation terms (reference apps/DiffARAP): cotangent edge
// weights over the EVDiamond relation, the best rotation per vertex, and the
// EV energy with its hand-written gradient. One workgroup per patch; every
// per-vertex result is gathered over the owner's rows, without atomics.
#pragma once
#include "k_numerics.hpp"
#include "k_query.hpp"

namespace rxm {

// cotangent of the angle at c of triangle (a, b, c) as arap_kernels.h:41-45
// writes it: dot(a - c, b - c) / length(cross(a - c, b - c))
__device__ __forceinline__ float arap_cot(f3 a, f3 b, f3 c)
{
    const f3 u = sub(a, c), v = sub(b, c), x = cross(u, v);
    return dot(u, v) / sqrtf(dot(x, x));
}

// ---- edge weights ------------------------------------------------------------
struct PlanAW
{
    uint32_t *ev, *opp;
    float *   x, *y, *z;
};
__host__ __device__ inline PlanAW plan_aw(Bump& b, uint32_t nv, uint32_t ne, uint32_t neo)
{
    PlanAW p{};
    p.ev  = b.alloc<uint32_t>(r4(ne));
    p.opp = b.alloc<uint32_t>(2 * neo);
    p.x   = b.alloc<float>(nv);
    p.y   = b.alloc<float>(nv);
    p.z   = b.alloc<float>(nv);
    return p;
}

// 654k vertices 18.2 -> 14.3 us, 2.6M 52 -> 40 (loads issued together, faces in
// registers; 512 threads 15.5 and 49).
// Per owned edge p-r with EVDiamond opposite vertices q and s (the slots of
// k_query_evd): w = max(0, (cot_q + cot_s) / 2) (arap_kernels.h:8-54); 0 for
// an edge that lacks a side, which the reference skips, leaving the weight at
// its reset value 0. w is indexed by linear edge id.
template <uint32_t T>
__global__ __launch_bounds__(T) void k_arap_weights(DevMesh m, const float* __restrict__ pos, float* __restrict__ w)
{
    extern __shared__ uint4 smem[];
    const uint32_t p = patch_of_block(m.P);  // XCD-contiguous patch ranges
    if (p >= m.P) return;
    const PatchDesc d = load_desc(m.patch, p);
    Bump            b(reinterpret_cast<char*>(smem));
    const PlanAW    L = plan_aw(b, d.nv, d.ne, d.neo);
    const uint16_t* fe  = m.fe + 3u * d.f_off;
    const u32x4*    evs = reinterpret_cast<const u32x4*>(m.ev + d.e_off);
    FaceWords                           fw[(768u + T - 1u) / T];
    Held<T, (384u + T - 1u) / T, u32x4> h_ev;
    HeldVerts<T, 3>                     hv;
    hv.ids(m, d);
    h_ev.load(evs, r4(d.ne) >> 2);
    load_faces<T>(fw, fe, d.nf);
    hv.owned(pos, m, d);
    hv.ribbon(pos, m, d);
    for (uint32_t i = threadIdx.x; i < 2 * d.neo; i += T) L.opp[i] = 0u;
    h_ev.store(reinterpret_cast<u32x4*>(L.ev), evs, r4(d.ne) >> 2);
    hv.store(pos, m, d, [&](uint32_t l, const float (&q)[3]) {
        L.x[l] = q[0];
        L.y[l] = q[1];
        L.z[l] = q[2];
    });
    __syncthreads();
    edge_opposites<T>(fw, fe, L.ev, d, L.opp);
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < d.neo; e += T) {
        const uint32_t qa = L.opp[2 * e], sa = L.opp[2 * e + 1];
        float          wt = 0.f;
        if (qa && sa) {
            const uint32_t x = L.ev[e], P = lo16(x), R = hi16(x), Q = qa & 0xFFFFu, S = sa & 0xFFFFu;
            const f3       pp{L.x[P], L.y[P], L.z[P]}, rr{L.x[R], L.y[R], L.z[R]};
            const f3       qq{L.x[Q], L.y[Q], L.z[Q]}, ss{L.x[S], L.y[S], L.z[S]};
            wt = (arap_cot(pp, rr, qq) + arap_cot(pp, rr, ss)) * 0.5f;
            wt = fmaxf(0.f, wt);  // also 0 for a NaN from a degenerate face, as std::max(0, NaN)
        }
        w[d.ep + e] = wt;
    }
}

// ---- best rotation -------------------------------------------------------------
// One Jacobi rotation of the symmetric 4x4 a in the (P, Q) plane (P < Q),
// zeroing a[P][Q]; v accumulates the eigenvectors as columns. Only the upper
// triangle of a is kept: a_PP -= t a_PQ, a_QQ += t a_PQ, a_PQ = 0, and the
// two other rows' (P, Q) pairs rotate. The rotation only has to be
// orthogonal, not exact (an angle off by an ulp leaves a tiny a[P][Q] that
// later sweeps remove): c = rsqrt(1 + t^2) and s = t c keep c^2 + s^2 = 1 to
// an ulp, so the hardware reciprocal and reciprocal square root serve.
template <int P, int Q>
__device__ __forceinline__ void jacobi4(float (&a)[4][4], float (&v)[4][4])
{
    static_assert(P < Q, "upper triangle");
    const float apq = a[P][Q];
    if (fabsf(apq) < 1e-30f) return;  // negligible in the unit-scaled matrix; keeps rcp away from denormals
    const float theta = 0.5f * (a[Q][Q] - a[P][P]) * __builtin_amdgcn_rcpf(apq);
    const float at    = fabsf(theta);
    // t = sign(theta) / (|theta| + sqrt(theta^2 + 1)); ~1 / (2 theta) once theta^2 would overflow
    const float den = (at < 1e18f) ? at + (at * at + 1.f) * __builtin_amdgcn_rsqf(at * at + 1.f) : 2.f * at;
    const float t   = copysignf(__builtin_amdgcn_rcpf(den), theta);
    const float c = __builtin_amdgcn_rsqf(t * t + 1.f), s = t * c;
    a[P][P] -= t * apq;
    a[Q][Q] += t * apq;
    a[P][Q] = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (k == P || k == Q) continue;
        // the upper-triangle entries (k, P) and (k, Q)
        float& akp = (k < P) ? a[k][P] : a[P][k];
        float& akq = (k < Q) ? a[k][Q] : a[Q][k];
        const float xp = akp, xq = akq;
        akp              = c * xp - s * xq;
        akq              = s * xp + c * xq;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float vkp = v[k][P], vkq = v[k][Q];
        v[k][P]         = c * vkp - s * vkq;
        v[k][Q]         = s * vkp + c * vkq;
    }
}

// The rotation R maximising tr(R S) (row-major R, S[a][b] = sum w e_a e'_b
// of rest e and deformed e' edge vectors): the reference takes R = V U^T
// from S = U Sigma V^T with a sign fix for reflections
// (arap_kernels.h:89-110). Computed here by Horn's closed form (J. Opt. Soc.
// Am. A 4(4):629, 1987): R's unit quaternion is the eigenvector of the
// largest eigenvalue of the symmetric 4x4 N(S), found by cyclic Jacobi
// sweeps; the result is a proper rotation by construction. S = 0 gives I.
__device__ inline void best_rotation(const float (&S)[3][3], float (&R)[3][3])
{
    float a[4][4], v[4][4];
    a[0][0] = S[0][0] + S[1][1] + S[2][2];
    a[1][1] = S[0][0] - S[1][1] - S[2][2];
    a[2][2] = -S[0][0] + S[1][1] - S[2][2];
    a[3][3] = -S[0][0] - S[1][1] + S[2][2];
    a[0][1] = a[1][0] = S[1][2] - S[2][1];
    a[0][2] = a[2][0] = S[2][0] - S[0][2];
    a[0][3] = a[3][0] = S[0][1] - S[1][0];
    a[1][2] = a[2][1] = S[0][1] + S[1][0];
    a[1][3] = a[3][1] = S[2][0] + S[0][2];
    a[2][3] = a[3][2] = S[1][2] + S[2][1];
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            mx      = fmaxf(mx, fabsf(a[i][j]));
            v[i][j] = (i == j) ? 1.f : 0.f;
        }
    if (mx > 0.f) {
        const float inv = 1.f / mx;  // scale: no under- or overflow in the sweeps
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) a[i][j] *= inv;
        for (int sweep = 0; sweep < 8; ++sweep) {
            // quadratic convergence: stop once the off-diagonal mass is below
            // fp32 resolution of the unit-scaled matrix (3-4 sweeps typically)
            const float off = a[0][1] * a[0][1] + a[0][2] * a[0][2] + a[0][3] * a[0][3] + a[1][2] * a[1][2] +
                              a[1][3] * a[1][3] + a[2][3] * a[2][3];
            if (off < 1e-15f) break;
            jacobi4<0, 1>(a, v);
            jacobi4<0, 2>(a, v);
            jacobi4<0, 3>(a, v);
            jacobi4<1, 2>(a, v);
            jacobi4<1, 3>(a, v);
            jacobi4<2, 3>(a, v);
        }
    }
    // eigenvector of the largest eigenvalue (static indices keep a, v in registers)
    float lk = a[0][0], q0 = v[0][0], qx = v[1][0], qy = v[2][0], qz = v[3][0];
#pragma unroll
    for (int i = 1; i < 4; ++i)
        if (a[i][i] > lk) {
            lk = a[i][i];
            q0 = v[0][i];
            qx = v[1][i];
            qy = v[2][i];
            qz = v[3][i];
        }
    const float n = 1.f / sqrtf(q0 * q0 + qx * qx + qy * qy + qz * qz);
    q0 *= n;
    qx *= n;
    qy *= n;
    qz *= n;
    R[0][0] = q0 * q0 + qx * qx - qy * qy - qz * qz;
    R[0][1] = 2.f * (qx * qy - q0 * qz);
    R[0][2] = 2.f * (qx * qz + q0 * qy);
    R[1][0] = 2.f * (qy * qx + q0 * qz);
    R[1][1] = q0 * q0 - qx * qx + qy * qy - qz * qz;
    R[1][2] = 2.f * (qy * qz - q0 * qx);
    R[2][0] = 2.f * (qz * qx - q0 * qy);
    R[2][1] = 2.f * (qz * qy + q0 * qx);
    R[2][2] = q0 * q0 - qx * qx - qy * qy + qz * qz;
}

// The same rotation without the sweeps, in FP64 (which runs at the rate of plain
// FP32 here): the largest eigenvalue of N(S) is the largest root of its
// characteristic polynomial, whose coefficients are S's invariants
// (l^4 - 2 |S|^2 l^2 - 8 det(S) l + |S|^4 - 4 |cof(S)|^2), found by Newton's
// method from the bound sqrt(3) |S| (monotone from above); its eigenvector is
// the largest column of the adjugate of N - l I (Theobald, Acta Cryst. A 61:478,
// 2005, takes the same two steps). Returns false, R unset, where the gap to the
// next eigenvalue all but cancels the adjugate (below 1e-7 of l^3), or the root
// has not settled: the sweeps decide there. What it accepts loses digits with the
// gap, but far fewer than the sweeps do in FP32: over random mirrored covariances
// the eigenvector is off by at most 8e-13, 6e-10, 1e-7, 2e-6 and 8e-6 at gaps of
// 1e-1 to 1e-5 of l, an FP32 eigenvector by 8e-7, 7e-6, 7e-5, 8e-4 and 7e-3, and
// S's own FP32 rounding moves it by 6e-8 over the gap. About 300 instructions a vertex
// against 2,000 and more of the sweeps, which bound the kernel
// (654k vertices 41 -> 30 us with the records written as one run and 256 threads,
// 2.6M 129 -> 90; now the staging). Its error against FP64 is not larger: R is
// rounded once (energy and gradient that use R: 6.9e-7 -> 3.3e-7 off).
__device__ inline bool best_rotation_direct(const float (&Sf)[3][3], float (&R)[3][3])
{
    double S[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) S[i][j] = static_cast<double>(Sf[i][j]);
    double f = 0.0, cf = 0.0, det = 0.0;  // |S|^2, |cof(S)|^2, det(S)
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int    i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
            const double c = S[i1][j1] * S[i2][j2] - S[i1][j2] * S[i2][j1];
            f += S[i][j] * S[i][j];
            cf += c * c;
            if (i == 0) det += S[0][j] * c;
        }
    const double c2 = -2.0 * f, c1 = -8.0 * det, c0 = f * f - 4.0 * cf;
    double       l = sqrt(3.0 * f);
    bool         settled = false;
    for (int it = 0; it < 24 && !settled; ++it) {
        const double l2 = l * l;
        const double p = ((l2 + c2) * l + c1) * l + c0, dp = (4.0 * l2 + 2.0 * c2) * l + c1;
        const double step = p * __builtin_amdgcn_rcp(dp);  // an approximate step only slows the last digits
        l -= step;
        settled = fabs(step) <= 1e-12 * l;
    }
    // B = N(S) - l I, upper triangle
    const double b00 = S[0][0] + S[1][1] + S[2][2] - l, b11 = S[0][0] - S[1][1] - S[2][2] - l;
    const double b22 = -S[0][0] + S[1][1] - S[2][2] - l, b33 = -S[0][0] - S[1][1] + S[2][2] - l;
    const double b01 = S[1][2] - S[2][1], b02 = S[2][0] - S[0][2], b03 = S[0][1] - S[1][0];
    const double b12 = S[0][1] + S[1][0], b13 = S[2][0] + S[0][2], b23 = S[1][2] + S[2][1];
    // 2 x 2 minors of rows (2, 3) and of rows (0, 1), columns as named
    const double m01 = b02 * b13 - b12 * b03, m02 = b02 * b23 - b22 * b03, m03 = b02 * b33 - b23 * b03;
    const double m12 = b12 * b23 - b22 * b13, m13 = b12 * b33 - b23 * b13, m23 = b22 * b33 - b23 * b23;
    const double n01 = b00 * b11 - b01 * b01, n02 = b00 * b12 - b02 * b01, n03 = b00 * b13 - b03 * b01;
    const double n12 = b01 * b12 - b02 * b11, n13 = b01 * b13 - b03 * b11;
    // cofactors (symmetric)
    const double a00 = b11 * m23 - b12 * m13 + b13 * m12, a01 = -(b01 * m23 - b12 * m03 + b13 * m02);
    const double a02 = b01 * m13 - b11 * m03 + b13 * m01, a03 = -(b01 * m12 - b11 * m02 + b12 * m01);
    const double a11 = b00 * m23 - b02 * m03 + b03 * m02, a12 = -(b00 * m13 - b01 * m03 + b03 * m01);
    const double a13 = b00 * m12 - b01 * m02 + b02 * m01;
    const double a22 = b33 * n01 - b13 * n03 + b03 * n13, a23 = -(b23 * n01 - b13 * n02 + b03 * n12);
    const double a33 = b22 * n01 - b12 * n02 + b02 * n12;
    double       dg = fabs(a00), q0 = a00, qx = a01, qy = a02, qz = a03;
    auto         take = [&](double d, double e0, double ex, double ey, double ez) {
        const bool up = fabs(d) > dg;
        dg = up ? fabs(d) : dg;
        q0 = up ? e0 : q0;
        qx = up ? ex : qx;
        qy = up ? ey : qy;
        qz = up ? ez : qz;
    };
    take(a11, a01, a11, a12, a13);
    take(a22, a02, a12, a22, a23);
    take(a33, a03, a13, a23, a33);
    // a degenerate S (l = 0) or a NaN fails the comparison
    if (!(settled && dg >= 1e-7 * l * l * l && l > 0.0)) return false;
    // unit scale: the components squared neither over- nor underflow
    const double u  = __builtin_amdgcn_rcp(dg);
    q0 *= u;
    qx *= u;
    qy *= u;
    qz *= u;
    const double n = q0 * q0 + qx * qx + qy * qy + qz * qz;
    double       v = __builtin_amdgcn_rcp(n);
    v              = v * (2.0 - n * v);
    v              = v * (2.0 - n * v);
    R[0][0] = static_cast<float>(v * (q0 * q0 + qx * qx - qy * qy - qz * qz));
    R[0][1] = static_cast<float>(2.0 * v * (qx * qy - q0 * qz));
    R[0][2] = static_cast<float>(2.0 * v * (qx * qz + q0 * qy));
    R[1][0] = static_cast<float>(2.0 * v * (qy * qx + q0 * qz));
    R[1][1] = static_cast<float>(v * (q0 * q0 - qx * qx + qy * qy - qz * qz));
    R[1][2] = static_cast<float>(2.0 * v * (qy * qz - q0 * qx));
    R[2][0] = static_cast<float>(2.0 * v * (qz * qx - q0 * qy));
    R[2][1] = static_cast<float>(2.0 * v * (qz * qy + q0 * qx));
    R[2][2] = static_cast<float>(v * (q0 * q0 - qx * qx - qy * qy + qz * qz));
    return true;
}

// Patch-local data of the rotation and energy kernels: the VV plan's rows
// (offsets, neighbours or half-edges), rest and deformed positions of every
// local vertex, weights of every local edge; for the energy also EV and the
// rotations of every local vertex, whose space then takes the residuals of the
// local edges (three floats each).
struct PlanAR
{
    uint32_t* ev;
    uint16_t *ro, *nb, *ent;
    float *   px, *py, *pz, *xx, *xy, *xz, *w, *rot;
};
__host__ __device__ inline PlanAR plan_ar(Bump& b, uint32_t nv, uint32_t ne, uint32_t nvo, uint32_t nent, bool rot)
{
    PlanAR p{};
    p.ev  = rot ? b.alloc<uint32_t>(r4(ne)) : nullptr;
    p.ro  = b.alloc<uint16_t>((nvo + 1u + 7u) & ~7u);
    p.nb  = rot ? nullptr : b.alloc<uint16_t>((nent + 7u) & ~7u);
    p.ent = b.alloc<uint16_t>((nent + 7u) & ~7u);
    p.px  = b.alloc<float>(nv);
    p.py  = b.alloc<float>(nv);
    p.pz  = b.alloc<float>(nv);
    p.xx  = b.alloc<float>(nv);
    p.xy  = b.alloc<float>(nv);
    p.xz  = b.alloc<float>(nv);
    p.w   = b.alloc<float>(ne);
    p.rot = rot ? b.alloc<float>(9 * nv + 3u > 3 * ne ? 9 * nv + 3u : 3 * ne) : nullptr;
    return p;
}

// Stage them, every load issued before the first is waited for, in two
// dependent round trips (the ribbon's ids, then its words).
// ROT: L.rot is moved to the first vertex's record.
template <uint32_t T, bool ROT>
__device__ __forceinline__ void stage_arap(const DevMesh& m, const PatchDesc& d, PlanAR& L,
                                           const uint16_t* __restrict__ roff, const uint16_t* __restrict__ nbr,
                                           const uint16_t* __restrict__ ent, uint32_t nent,
                                           const float* __restrict__ rest, const float* __restrict__ x,
                                           const float* __restrict__ w, const float* __restrict__ R)
{
    const uint32_t     t = threadIdx.x, ner = d.ne - d.neo;
    constexpr uint32_t RW = (768u + T - 1u) / T, RX = (512u + T - 1u) / T;  // owned / ribbon edges in registers
    const uint32_t*    el  = m.e_lin + d.e_off;
    const u32x4*       evs = reinterpret_cast<const u32x4*>(m.ev + d.e_off);
    HeldVerts<T, 3>                     hp, hx;
    Held<T, (384u + T - 1u) / T, u32x4> h_ev;
    Held<T, (256u + T - 1u) / T, u32x4> h_nb, h_ent;
    Held<T, 1, u32x4>                   h_ro;
    uint32_t                            ge[RX];
    float                               wo[RW], wr[RX];
    // rotations: the owned vertices' records are one run of 9 nvo floats, the
    // ribbon's are gathered word by word (record j of the ribbon at 9 (nvo + j))
    constexpr uint32_t            RQ = (1536u + T - 1u) / T;
    const uint32_t                nq = 9u * (d.nv - d.nvo);
    const float*                  Ro = R + 9ull * d.vp;
    HeldFloats<T, (768u + T - 1u) / T> h_rot;
    uint32_t                      gq[RQ];
    float                         rq[RQ];
    auto rec = [&](uint32_t i) { return min(d.nvo + i / 9u, d.nv - 1u); };
    hp.ids(m, d);
    if constexpr (ROT)
#pragma unroll
        for (uint32_t k = 0; k < RQ; ++k)
            if (k == 0 || k * T < nq) gq[k] = m.v_lin[d.v_off + rec(t + k * T)];
#pragma unroll
    for (uint32_t k = 0; k < RX; ++k)
        if (k == 0 || k * T < ner) ge[k] = el[min(d.neo + t + k * T, d.ne - 1u)];
    if constexpr (ROT) h_ev.load(evs, r4(d.ne) >> 2);
    h_ro.load(as_words(roff), words8(d.nvo + 1));
    h_ent.load(as_words(ent), words8(nent));
    if constexpr (!ROT) h_nb.load(as_words(nbr), words8(nent));
    if constexpr (ROT) h_rot.load(Ro, 9u * d.nvo);
    hp.owned(rest, m, d);
    hx.owned(x, m, d);
#pragma unroll
    for (uint32_t k = 0; k < RW; ++k)
        if (k == 0 || k * T < d.neo) wo[k] = w[min(d.ep + t + k * T, m.nE - 1u)];
#pragma unroll
    for (uint32_t k = 0; k < HeldVerts<T, 3>::RR; ++k) hx.g[k] = hp.g[k];
    hp.ribbon(rest, m, d);
    hx.ribbon(x, m, d);
#pragma unroll
    for (uint32_t k = 0; k < RX; ++k)
        if (k == 0 || k * T < ner) wr[k] = w[ge[k]];
    if constexpr (ROT) {
#pragma unroll
        for (uint32_t k = 0; k < RQ; ++k)
            if (k == 0 || k * T < nq) rq[k] = R[9ull * gq[k] + (t + k * T) % 9u];
        h_rot.store(L.rot, Ro, 9u * d.nvo);
        L.rot += h_rot.shift(Ro);
#pragma unroll
        for (uint32_t k = 0; k < RQ; ++k)
            if (t + k * T < nq) L.rot[9u * d.nvo + t + k * T] = rq[k];
        for (uint32_t i = t + RQ * T; i < nq; i += T)
            L.rot[9u * d.nvo + i] = R[9ull * m.v_lin[d.v_off + rec(i)] + i % 9u];
        h_ev.store(reinterpret_cast<u32x4*>(L.ev), evs, r4(d.ne) >> 2);
    }
    h_ro.store(as_words(L.ro), as_words(roff), words8(d.nvo + 1));
    h_ent.store(as_words(L.ent), as_words(ent), words8(nent));
    if constexpr (!ROT) h_nb.store(as_words(L.nb), as_words(nbr), words8(nent));
    hp.store(rest, m, d, [&](uint32_t l, const float (&q)[3]) {
        L.px[l] = q[0];
        L.py[l] = q[1];
        L.pz[l] = q[2];
    });
    hx.store(x, m, d, [&](uint32_t l, const float (&q)[3]) {
        L.xx[l] = q[0];
        L.xy[l] = q[1];
        L.xz[l] = q[2];
    });
#pragma unroll
    for (uint32_t k = 0; k < RW; ++k)
        if (t + k * T < d.neo) L.w[t + k * T] = wo[k];
#pragma unroll
    for (uint32_t k = 0; k < RX; ++k)
        if (t + k * T < ner) L.w[d.neo + t + k * T] = wr[k];
    for (uint32_t e = t + RW * T; e < d.neo; e += T) L.w[e] = w[d.ep + e];
    for (uint32_t e = d.neo + t + RX * T; e < d.ne; e += T) L.w[e] = w[el[e]];
}

// Best rotation per owned vertex (arap_kernels.h:60-117): S = sum over the
// vertex's VV row of w (P_v - P_j)(X_v - X_j)^T, R from best_rotation. R
// holds one row-major 3 x 3 record per vertex, R[9 v + 3 i + j] = R_v(i, j)
// (the reference's rotations(v, i * 3 + j)): a ribbon vertex's rotation is
// one or two cache lines for the energy kernel's gather, not nine.
// RUN: a round's records pass through LDS and leave as one run; without, each
// lane stores its own, for patches that leave no LDS for them.
template <uint32_t T, bool RUN = true>
__global__ __launch_bounds__(T) void k_arap_rotations(DevMesh m, const uint32_t* __restrict__ vv_base,
                                                      const uint32_t* __restrict__ rbase,
                                                      const uint32_t* __restrict__ nbase,
                                                      const uint16_t* __restrict__ roff,
                                                      const uint16_t* __restrict__ nbr,
                                                      const uint16_t* __restrict__ ent,
                                                      const float* __restrict__ rest, const float* __restrict__ x,
                                                      const float* __restrict__ w, float* __restrict__ R)
{
    extern __shared__ uint4 smem[];
    const uint32_t p = patch_of_block(m.P);  // XCD-contiguous patch ranges
    if (p >= m.P) return;
    const PatchDesc d    = load_desc(m.patch, p);
    const uint32_t  nent = vv_base[p + 1] - vv_base[p];
    Bump            b(reinterpret_cast<char*>(smem));
    PlanAR          L = plan_ar(b, d.nv, d.ne, d.nvo, nent, false);
    stage_arap<T, false>(m, d, L, roff + rbase[p], nbr + nbase[p], ent + nbase[p], nent, rest, x, w, nullptr);
    float* const out = RUN ? b.alloc<float>(9u * T) : nullptr;  // this round's records, written as one run
    __syncthreads();
    for (uint32_t v0 = 0; v0 < d.nvo; v0 += T) {
        const uint32_t v = v0 + threadIdx.x, nr = min(T, d.nvo - v0);
        float* const   dst = R + 9ull * (d.vp + v0);
        if (v < d.nvo) {
            float       S[3][3] = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
            const float p0 = L.px[v], p1 = L.py[v], p2 = L.pz[v], x0 = L.xx[v], x1 = L.xy[v], x2 = L.xz[v];
            for (uint32_t k = L.ro[v]; k < L.ro[v + 1]; ++k) {
                const uint32_t j = L.nb[k];
                const float    wt = L.w[L.ent[k] >> 1];
                const float    a[3] = {p0 - L.px[j], p1 - L.py[j], p2 - L.pz[j]};
                const float    c[3] = {x0 - L.xx[j], x1 - L.xy[j], x2 - L.xz[j]};
#pragma unroll
                for (int r = 0; r < 3; ++r)
#pragma unroll
                    for (int s = 0; s < 3; ++s) S[r][s] += wt * a[r] * c[s];
            }
            float Rv[3][3];
            if (!best_rotation_direct(S, Rv)) best_rotation(S, Rv);
            float* const rec = RUN ? out + 9u * threadIdx.x : dst + 9u * threadIdx.x;
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int s = 0; s < 3; ++s) rec[3u * r + s] = Rv[r][s];
        }
        if constexpr (RUN) {
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < 9u * nr; i += T) dst[i] = out[i];
            __syncthreads();
        }
    }
}

// edge residual d = (X_i - X_j) - R_i (P_i - P_j) for local endpoints i, j
__device__ __forceinline__ f3 arap_residual(const PlanAR& L, uint32_t i, uint32_t j)
{
    const float  e0 = L.px[i] - L.px[j], e1 = L.py[i] - L.py[j], e2 = L.pz[i] - L.pz[j];
    const float* r  = L.rot + 9 * i;
    return {(L.xx[i] - L.xx[j]) - (r[0] * e0 + r[1] * e1 + r[2] * e2),
            (L.xy[i] - L.xy[j]) - (r[3] * e0 + r[4] * e1 + r[5] * e2),
            (L.xz[i] - L.xz[j]) - (r[6] * e0 + r[7] * e1 + r[8] * e2)};
}

// Energy E = sum over owned edges, i = EV's first vertex (the larger global
// id, the reference's iter[0] of Op::EV), of w |(X_i - X_j) - R_i (P_i -
// P_j)|^2 (diff_arap.cu:87-118), one partial per patch; gradient with the
// rotations held fixed (the reference's term reads them as constants):
// dE/dX_v = sum over v's edges of +-2 w d, + where v is the edge's i.
// Every local edge's residual is evaluated once, into registers, and stored
// over the rotations once all are done; the gradient gathers them per vertex
// (patches beyond the register rounds evaluate an edge at each use). 654k
// vertices 42.8 -> 33 us, 2.6M 142 -> 112. Bound: the gathers of the ribbon's
// rotations and the residuals' LDS reads.
template <uint32_t T>
__global__ __launch_bounds__(T) void k_arap_energy_grad(DevMesh m, const uint32_t* __restrict__ vv_base,
                                                        const uint32_t* __restrict__ rbase,
                                                        const uint32_t* __restrict__ nbase,
                                                        const uint16_t* __restrict__ roff,
                                                        const uint16_t* __restrict__ ent,
                                                        const float* __restrict__ rest, const float* __restrict__ x,
                                                        const float* __restrict__ w, const float* __restrict__ R,
                                                        float* __restrict__ partial, float* __restrict__ grad)
{
    constexpr uint32_t RE = (1536u + T - 1u) / T;  // edges in registers
    extern __shared__ uint4 smem[];
    __shared__ float red[T / 64u];
    const uint32_t   p = patch_of_block(m.P);  // XCD-contiguous patch ranges
    if (p >= m.P) return;
    const PatchDesc d    = load_desc(m.patch, p);
    const uint32_t  nent = vv_base[p + 1] - vv_base[p], t = threadIdx.x;
    Bump            b(reinterpret_cast<char*>(smem));
    PlanAR          L = plan_ar(b, d.nv, d.ne, d.nvo, nent, true);
    float* const    res = L.rot;  // the residuals' space
    stage_arap<T, true>(m, d, L, roff + rbase[p], nullptr, ent + nbase[p], nent, rest, x, w, R);
    __syncthreads();
    float      acc  = 0.f;
    const bool held = d.ne <= RE * T;
    float *    rx = res, *ry = rx + d.ne, *rz = ry + d.ne;
    if (held) {
        f3 r[RE];
#pragma unroll
        for (uint32_t k = 0; k < RE; ++k) {
            const uint32_t e = t + k * T;
            if (e < d.ne) {
                const uint32_t y = L.ev[e];
                r[k]             = arap_residual(L, lo16(y), hi16(y));
                if (e < d.neo) acc += L.w[e] * dot(r[k], r[k]);
            }
        }
        __syncthreads();  // every rotation has been read
#pragma unroll
        for (uint32_t k = 0; k < RE; ++k) {
            const uint32_t e = t + k * T;
            if (e < d.ne) {
                rx[e] = r[k].x;
                ry[e] = r[k].y;
                rz[e] = r[k].z;
            }
        }
        __syncthreads();
    } else {
        for (uint32_t e = t; e < d.neo; e += T) {
            const uint32_t y = L.ev[e];
            const f3       r = arap_residual(L, lo16(y), hi16(y));
            acc += L.w[e] * dot(r, r);
        }
    }
    const uint32_t N = m.nV;
    for (uint32_t v = t; v < d.nvo; v += T) {
        float gx = 0.f, gy = 0.f, gz = 0.f;
        for (uint32_t k = L.ro[v]; k < L.ro[v + 1]; ++k) {
            const uint32_t u = L.ent[k], e = u >> 1;  // the half-edge leaving v: dir 0 where v is the edge's i
            f3             r;
            if (held) {
                r = f3{rx[e], ry[e], rz[e]};
            } else {
                const uint32_t y = L.ev[e];
                r                = arap_residual(L, lo16(y), hi16(y));
            }
            const float s = ((u & 1u) ? -2.f : 2.f) * L.w[e];
            gx += s * r.x;
            gy += s * r.y;
            gz += s * r.z;
        }
        const uint32_t g = d.vp + v;
        grad[g]          = gx;
        grad[N + g]      = gy;
        grad[2 * N + g]  = gz;
    }
    // fixed-order workgroup sum of the energy
    for (uint32_t o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((t & 63u) == 0) red[t >> 6] = acc;
    __syncthreads();
    if (t == 0) {
        float s = 0.f;
        for (uint32_t i = 0; i < T / 64u; ++i) s += red[i];
        partial[p] = s;
    }
}

}  // namespace rxm
