// Device-side integrator for continuous piecewise-affine (CPA) velocity
// fields on gfx950.
//
// Coordinates.  All integration runs in scaled coordinates q = x * nc
// (x in [0,1]^D, nc = cells per axis), where the field of cell c is
// q' = Mq q + bq with Mq = S M S^-1, bq = S b, S = diag(nc).  Facets are unit
// planes n.q + e <= 0 (inside), stored per cell with the cell across them.
//
// In-cell flow.  For v = M q + b the exact flow is
//     q(s) = q0 + sum_{k>=1} s^k / k! M^(k-1) v0 ,   v0 = M q0 + b,
// an entire series.  It is evaluated on chunks with |M|_F h <= RHO = 1/2 and
// KS = 7 terms, so the truncation (< RHO^7/8! = 1.9e-7 relative to the chunk
// displacement; 1e-9 at the typical |M|_F h ~ 0.25) is at FP32 resolution; no
// eigenvalue case analysis (real / complex / repeated) and no transcendental
// calls are needed in 2D/3D.  Cayley-Hamilton reduces the series to D scalars
// (flow_at): q(s) = q0 + sum_{i<D} al_i(s) M^i v0 and exp(s M) =
// sum_{i<D} e_i(s) M^i, with al and e from one Horner recurrence in the
// invariants of s M.  The position, the Jacobian, every facet's G and G' and
// the gradient integral share those scalars, so a chunk keeps D vectors
// instead of KS and a facet D + 1 coefficients instead of KS + 1.
// 1D uses the closed form q(s) = q0 + s*phi1(a s)*v0 and the analytic hit time
// s = (qb-q0)/v0 * log1p(r)/r, r = a (qb-q0)/v0.
//
// Boundary hits.  For each facet G(s) = n.q(s) + e is the same series.  A
// facet is skipped when a convex cubic bound on G is negative at the chunk's
// end.  Where a bound on the series tail certifies the sign of G'' or of G'
// over the chunk, G(h) decides the crossing and [0, h] brackets a unique root.  Starts on a facet,
// uncertified curvature and interior maxima are bracketed by sampling G and G'
// at NSAMP points (a local maximum with G > 0 inside a sample interval
// counts).  A bracket is solved by Newton steps safeguarded by it; a second
// facet is solved only when it is positive at (or its bracket ends before) the
// first one's root.
//
// Gradients.  The field is continuous across facets, so the sensitivity of the
// final point obeys the variational equation with the saltation matrix
// S = I + (v_next - v_prev) n^T / (n.v_prev) at every crossing (S = I for a
// continuous field; it is applied anyway so the hit-time and cell-change terms
// are part of the derivative).  Pass 1 carries J = dq(T)/dq0; the adjoint at
// t = 0 is mu0 = J^T dL/dq(T).  Pass 2 re-integrates forward carrying
// mu(s) = exp(-s M^T) mu0 and adds int_0^h mu(s) [q(s);1]^T ds to dL/dA_q of
// the cell, an exact double series.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#define CPAB_HD __host__ __device__
#include <stdint.h>
#include <limits.h>
#include <type_traits>

namespace cpab {

constexpr int NF = 4;           // facet slots per cell
constexpr int KS = 7;           // series terms
constexpr float RHO = 0.5f;     // chunk bound |M|_F * h
constexpr float GROW = 1.6488f;   // e^RHO: speed growth bound over a chunk
constexpr int NSAMP = 4;        // samples per chunk for root isolation
constexpr int MAX_ITERS = 512;  // chunks + crossings per point (termination bound; a point that
                                // has time left after them is unfinished: NaN, and counted)
constexpr float ZERO_HOP = 1e-7f;
constexpr int MAX_ZERO_HOPS = 8;
constexpr int NREC = 2;         // chunks per point the forward records for the backward (2D/3D)

template <int D>
struct CellTable {
    const float* A;      // [nC, D, D+1]  q-space affine
    const float* inv_n;  // [nC]          1 / |Mq|_F (inf for Mq = 0)
    const float4* pl;    // [nC, NF]      (n0, n1, n2, e)
    const int* nb;       // [nC, NF]      neighbour, <0: none
    const float2* hits = nullptr;  // 1D, nullable: [nC, 2] crossing a whole cell to the left, right: time, a dq / v0
};

template <int D>
struct PointState {
    float q[D];
    float T;        // remaining time
    int c;          // current cell
    int came_from;  // cell left by the last crossing
    int zero_hops;  // consecutive crossings of (near) zero length
    int iters;
};

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
// 1/x to ~1 ulp for the safeguarded iterations (their steps are clamped to a
// bracket, so the correctly rounded quotient is not needed)
CPAB_HD __forceinline__ float fast_rcp(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcpf(x);
#else
    return 1.0f / x;
#endif
}
// sqrt(x) to ~1 ulp for the chunk bounds and thresholds (their constants
// carry the margin; the correctly rounded square root costs a dozen more
// instructions per chunk)
CPAB_HD __forceinline__ float fast_sqrt(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_sqrtf(x);
#else
    return sqrtf(x);
#endif
}
// a * b of non-negative integers below 2^24 (cell numbers and table strides): a
// full-rate product; the compiler's own choice for a table address is a 64-bit
// multiply-add at a quarter of the rate
CPAB_HD __forceinline__ int mul_small(int a, int b) {
    return (int)(((unsigned)a & 0xFFFFFFu) * ((unsigned)b & 0xFFFFFFu));
}
template <int D>
CPAB_HD __forceinline__ void load_affine(const CellTable<D>& t, int c, float (&M)[D][D], float (&b)[D]) {
    const float* a = t.A + mul_small(c, D * (D + 1));
#pragma unroll
    for (int r = 0; r < D; ++r) {
#pragma unroll
        for (int k = 0; k < D; ++k) M[r][k] = a[r * (D + 1) + k];
        b[r] = a[r * (D + 1) + D];
    }
}

template <int D>
CPAB_HD __forceinline__ void affine_apply(const float (&M)[D][D], const float (&b)[D], const float (&q)[D], float (&v)[D]) {
#pragma unroll
    for (int r = 0; r < D; ++r) {
        float acc = b[r];
#pragma unroll
        for (int k = 0; k < D; ++k) acc = fmaf(M[r][k], q[k], acc);
        v[r] = acc;
    }
}

// Invariants of a cell's M: trace, (3D) second invariant, determinant.
template <int D>
struct Invariants {
    float t, sg, d;
};
template <int D>
CPAB_HD __forceinline__ Invariants<D> invariants(const float (&M)[D][D]) {
    Invariants<D> v;
    if constexpr (D == 2) {
        v.t = M[0][0] + M[1][1];
        v.sg = 0.f;
        v.d = fmaf(M[0][0], M[1][1], -(M[0][1] * M[1][0]));
    } else {
        v.t = M[0][0] + M[1][1] + M[2][2];
        const float c0 = fmaf(M[1][1], M[2][2], -(M[1][2] * M[2][1]));
        const float c1 = fmaf(M[1][0], M[2][2], -(M[1][2] * M[2][0]));
        const float c2 = fmaf(M[1][0], M[2][1], -(M[1][1] * M[2][0]));
        v.sg = c0 + fmaf(M[0][0], M[2][2], -(M[0][2] * M[2][0])) + fmaf(M[0][0], M[1][1], -(M[0][1] * M[1][0]));
        v.d = fmaf(M[0][0], c0, fmaf(-M[0][1], c1, M[0][2] * c2));
    }
    return v;
}

// The flow's scalars at time s: displacement sum_i al[i] M^i v0 and
// exp(s M) = sum_i e[i] M^i.  With N = s M, phi1(N) = sum_{k<KS} N^k/(k+1)! is
// evaluated by Horner's rule in the powers of N below D, each product by N
// reduced by the characteristic polynomial (2D: N^2 = t N - d; 3D: N^3 =
// t N^2 - sg N + d); then al_i M^i = s phi1 and exp(N) = I + N phi1.
template <int D>
struct FlowAt {
    float al[D], e[D];
};
template <int D>
CPAB_HD __forceinline__ FlowAt<D> flow_at(const Invariants<D>& iv, float s) {
    static_assert(KS == 7, "the Horner constants below are 1/(k+1)! for k < 7");
    constexpr float C[KS] = {1.f, 1.f / 2, 1.f / 6, 1.f / 24, 1.f / 120, 1.f / 720, 1.f / 5040};
    FlowAt<D> f;
    const float tt = s * iv.t, s2 = s * s;
    if constexpr (D == 2) {
        const float dd = s2 * iv.d;
        float a = C[6], b = C[5];  // a N + b
#pragma unroll
        for (int k = 4; k >= 0; --k) {
            const float an = fmaf(tt, a, b);
            b = fmaf(-dd, a, C[k]);
            a = an;
        }
        f.al[0] = s * b;
        f.al[1] = s2 * a;
        f.e[0] = fmaf(-dd, a, 1.f);
        f.e[1] = s * fmaf(tt, a, b);
    } else {
        const float s3 = s2 * s;
        const float ss = s2 * iv.sg, dd = s3 * iv.d;
        float a = C[6], b = C[5], c = C[4];  // a N^2 + b N + c
#pragma unroll
        for (int k = 3; k >= 0; --k) {
            const float an = fmaf(tt, a, b);
            b = fmaf(-ss, a, c);
            c = fmaf(dd, a, C[k]);
            a = an;
        }
        f.al[0] = s * c;
        f.al[1] = s2 * b;
        f.al[2] = s3 * a;
        f.e[0] = fmaf(dd, a, 1.f);
        f.e[1] = s * fmaf(-ss, a, c);
        f.e[2] = s2 * fmaf(tt, a, b);
    }
    return f;
}

// G(s) = n.q(s) + e along one facet: g[0] = G(0), g[i + 1] = n.M^i v0.
template <int D>
struct FacetG {
    float g[D + 1];
};
template <int D>
CPAB_HD __forceinline__ float facet_g(const FacetG<D>& F, const FlowAt<D>& f) {
    float r = F.g[0];
#pragma unroll
    for (int i = 0; i < D; ++i) r = fmaf(f.al[i], F.g[i + 1], r);
    return r;
}
template <int D>
CPAB_HD __forceinline__ float facet_dg(const FacetG<D>& F, const FlowAt<D>& f) {
    float r = f.e[0] * F.g[1];
#pragma unroll
    for (int i = 1; i < D; ++i) r = fmaf(f.e[i], F.g[i + 1], r);
    return r;
}
// G(s) and G'(s)
template <int D>
CPAB_HD __forceinline__ void facet_at(const FacetG<D>& F, const Invariants<D>& iv, float s, float& g, float& d) {
    const FlowAt<D> f = flow_at<D>(iv, s);
    g = facet_g<D>(F, f);
    d = facet_dg<D>(F, f);
}

// Root of G in [lo, hi] with G(lo) <= 0 < G(hi): Newton steps from the root of
// the quadratic model, safeguarded by bisection.  A lane stops after a Newton
// step below 1e-5 of its bracket (quadratic convergence: the error is then
// ~1e-10) or after 6 steps; its result depends on its own iterates only, not
// on the other lanes of the wave.
template <int D>
CPAB_HD __forceinline__ float solve_bracket(const FacetG<D>& F, const Invariants<D>& iv, float lo, float hi, float glo,
                                            float ghi) {
    // the root of G's quadratic model at 0 (relative error ~ (|M| h)^2 / 6; two
    // evaluations then usually end the iteration, four from the regula-falsi
    // point), where it falls inside the bracket
    float s = -2.f * F.g[0] * fast_rcp(F.g[1] + fast_sqrt(fmaf(F.g[1], F.g[1], -2.f * (F.g[2] * F.g[0]))));
    if (!(s >= lo && s <= hi)) s = lo + (hi - lo) * (glo * fast_rcp(glo - ghi));
    if (!(s >= lo && s <= hi)) s = 0.5f * (lo + hi);
    const float tol = 1e-5f * (hi - lo);
    bool fin = false;
#pragma unroll 1
    for (int it = 0; it < 6; ++it) {
        if (!fin) {
            float g, d;
            facet_at<D>(F, iv, s, g, d);
            if (g > 0.f) hi = s; else lo = s;
            float sn = s - g * fast_rcp(d);
            const bool newton = sn >= lo && sn <= hi;
            if (!newton) sn = 0.5f * (lo + hi);
            fin = newton && fabsf(sn - s) <= tol;
            s = sn;
        }
#if defined(__HIP_DEVICE_COMPILE__)
        if (__ballot(!fin) == 0) break;
#else
        if (fin) break;
#endif
    }
    return s;
}

// Zero of G' in [lo, hi] given G'(lo) and G'(hi) of opposite signs:
// Illinois-modified secant steps inside the shrinking bracket; returns the
// bracket end with the smaller |G'|.
template <int D>
CPAB_HD __forceinline__ float crit_point(const FacetG<D>& F, const Invariants<D>& iv, float lo, float hi, float dlo,
                                         float dhi) {
    int side = 0;
#pragma unroll 1
    for (int it = 0; it < 4; ++it) {
        const float m = (lo * dhi - hi * dlo) * fast_rcp(dhi - dlo);
        if (!(m > lo && m < hi)) break;
        float gm, dm;
        facet_at<D>(F, iv, m, gm, dm);
        if ((dm > 0.f) == (dlo > 0.f)) {
            lo = m;
            dlo = dm;
            if (side == -1) dhi *= 0.5f;
            side = -1;
        } else {
            hi = m;
            dhi = dm;
            if (side == 1) dlo *= 0.5f;
            side = 1;
        }
    }
    return (fabsf(dlo) < fabsf(dhi)) ? lo : hi;
}

// Bracket of the first exit through one facet within a chunk.
struct Bracket {
    float lo, hi, glo, ghi;
    int idx;  // 0: exits at the start; i: inside sample interval i; NSAMP+1: none
};

// Isolates the first time in [0, h] at which the trajectory leaves through the
// facet F (G <= 0 inside).
//  * A start on the facet (G(0) >= -tol0, taken as G(0) = 0) moving out
//    exits at 0 when allow_start: G'(0) > tol1, or 0 <= G'(0) <= tol1 (an
//    outward speed within the rounding of the field) with G''(0) > 0.
//  * A start on the facet with G'(0) < 0, however small, first dips below 0;
//    a later positive sample is bracketed from the dip's minimum (zero of
//    G').  Two cells round the normal speed of the same point differently, so
//    a point handed over by a zero-length crossing may see a tangential start
//    here that its previous cell saw as a clear exit: the dip still has to be
//    followed out.
//  * Any other start on the facet (G'(0) >= 0 with the start exit
//    disallowed) is ignored until G has gone negative.
//  * Between two negative samples a local maximum above 0 is a crossing.
template <int D>
CPAB_HD __forceinline__ void first_bracket(const FacetG<D>& F, const Invariants<D>& iv, float h, float tol0, float tol1,
                                           bool allow_start, Bracket& br) {
    br.idx = NSAMP + 1;
    const bool on = F.g[0] >= -tol0;
    if (on && allow_start && (F.g[1] > tol1 || (F.g[1] >= 0.f && F.g[2] > 0.f))) {
        br.idx = 0;
        br.lo = br.hi = 0.f;
        return;
    }
    bool skip = on && !(F.g[1] < 0.f);
    bool dip = on && !skip;
    float ps = 0.f, pg = F.g[0], pd = F.g[1];
#pragma unroll 1
    for (int i = 1; i <= NSAMP; ++i) {
        const float s = h * ((float)i * (1.0f / NSAMP));
        float g, d;
        facet_at<D>(F, iv, s, g, d);
        // 0: nothing, 1: dip minimum (G comes back above 0), 2: graze maximum
        int crit = 0;
        if (skip) {
            if (g <= 0.f) skip = false;
        } else if (dip) {
            if (g <= 0.f) dip = false;
            else if (pd < 0.f && d > 0.f) crit = 1;
        } else {
            if (g > 0.f && pg <= 0.f) {
                br.idx = i; br.lo = ps; br.hi = s; br.glo = pg; br.ghi = g;
                return;
            }
            if (pd > 0.f && d < 0.f) crit = 2;
        }
        if (crit) {
            const float m = crit_point<D>(F, iv, ps, s, pd, d);
            const float gm = facet_g<D>(F, flow_at<D>(iv, m));
            if (crit == 1 && gm < 0.f) {
                br.idx = i; br.lo = m; br.hi = s; br.glo = gm; br.ghi = g;
                return;
            }
            if (crit == 2 && gm > 0.f) {
                br.idx = i; br.lo = ps; br.hi = m; br.glo = pg; br.ghi = gm;
                return;
            }
            if (crit == 1) {  // never went inside: treat as outside until G < 0
                skip = true;
                dip = false;
            }
        }
        ps = s;
        pg = g;
        pd = d;
    }
}

// The chunk's vectors v[i] = M^i v0, i < D.
template <int D>
CPAB_HD __forceinline__ void powers(const float (&M)[D][D], const float (&v0)[D], float (&v)[D][D]) {
#pragma unroll
    for (int a = 0; a < D; ++a) v[0][a] = v0[a];
#pragma unroll
    for (int k = 1; k < D; ++k)
#pragma unroll
        for (int r = 0; r < D; ++r) {
            float acc = M[r][0] * v[k - 1][0];
#pragma unroll
            for (int a = 1; a < D; ++a) acc = fmaf(M[r][a], v[k - 1][a], acc);
            v[k][r] = acc;
        }
}

// The cells across the facets of cell c (one 16-byte load on the device, where
// the staged table is aligned)
template <int D>
CPAB_HD __forceinline__ void cell_neighbours(const CellTable<D>& tab, int c, int (&nb)[NF]) {
#if defined(__HIP_DEVICE_COMPILE__)
    const int4 v = reinterpret_cast<const int4*>(tab.nb)[c];
    nb[0] = v.x;
    nb[1] = v.y;
    nb[2] = v.z;
    nb[3] = v.w;
#else
    for (int f = 0; f < NF; ++f) nb[f] = tab.nb[c * NF + f];
#endif
}

// Coefficients of facet f of cell c.  A start within tol0 of the facet is a
// start on it: G(0) = 0 exactly, so the sign of G just after the start is that
// of G'(0) (and, for a shallow dip into the cell, of the dip) rather than that
// of the rounding in n.q + e.
template <int D>
CPAB_HD __forceinline__ FacetG<D> facet_coeffs(const CellTable<D>& tab, int c, int f, const float (&q)[D],
                                               const float (&v)[D][D], float tol0) {
    const float4 P = tab.pl[c * NF + f];
    const float n[3] = {P.x, P.y, P.z};
    FacetG<D> F;
    float g0 = P.w;
#pragma unroll
    for (int a = 0; a < D; ++a) g0 = fmaf(n[a], q[a], g0);
    F.g[0] = (g0 >= -tol0) ? 0.f : g0;
#pragma unroll
    for (int k = 0; k < D; ++k) {
        float acc = n[0] * v[k][0];
#pragma unroll
        for (int a = 1; a < D; ++a) acc = fmaf(n[a], v[k][a], acc);
        F.g[k + 1] = acc;
    }
    return F;
}

// What one chunk did; handed to the pass callbacks.
template <int D>
struct Chunk {
    float M[D][D];
    float b[D];
    float q0[D];
    float v[D][D];     // v[i] = M^i v0
    Invariants<D> iv;
    FlowAt<D> f;       // the flow's scalars at h
    float h;           // time advanced
    int cell;
    int facet;         // crossed facet (-1: none)
    int next;          // cell entered (== cell if no crossing)
    float q1[D];       // end point
};

// End of a chunk of duration step that crosses facet bf (-1: none): end point,
// chunk record and the point's state (ch.M, ch.b, ch.v and ch.f are set).
template <int D>
CPAB_HD __forceinline__ void finish_chunk(PointState<D>& st, const CellTable<D>& tab, float step, int bf,
                                          Chunk<D>& ch) {
    const int c = st.c;
#pragma unroll
    for (int a = 0; a < D; ++a) ch.q0[a] = st.q[a];
#pragma unroll
    for (int a = 0; a < D; ++a) {
        float acc = ch.f.al[D - 1] * ch.v[D - 1][a];
#pragma unroll
        for (int k = D - 2; k >= 0; --k) acc = fmaf(ch.f.al[k], ch.v[k][a], acc);
        ch.q1[a] = ch.q0[a] + acc;
    }
    ch.h = step;
    ch.cell = c;
    ch.facet = bf;
    ch.next = (bf >= 0) ? tab.nb[c * NF + bf] : c;
#pragma unroll
    for (int a = 0; a < D; ++a) st.q[a] = ch.q1[a];
    st.T = (bf >= 0) ? fmaxf(st.T - step, 0.f) : st.T - step;
    if (bf < 0 && st.T < 0.f) st.T = 0.f;
    if (bf >= 0) {
        st.zero_hops = (step <= ZERO_HOP) ? st.zero_hops + 1 : 0;
        st.came_from = c;
        st.c = ch.next;
    } else if (step > ZERO_HOP) {
        // time went by inside the cell: the guard against crossing straight
        // back only covers a run of zero-length crossings
        st.zero_hops = 0;
    }
    st.iters++;
}

// The first NREC chunks of a point's trajectory: durations and crossed facets.
// code: bits 0-1 chunks recorded; bits 2+3i..4+3i facet crossed by chunk i, + 1
// (0: none).
struct ChunkLog {
    float h[NREC];
    int code;
};

CPAB_HD __forceinline__ void log_chunk(ChunkLog& lg, float h, int facet) {
    const int n = lg.code & 3;
#pragma unroll
    for (int k = 0; k < NREC; ++k)
        if (k == n) lg.h[k] = h;
    if (n < NREC) lg.code = ((lg.code & ~3) | (n + 1)) | ((facet + 1) << (2 + 3 * n));
}

// Sink for the forward's chunk log: durations go straight to memory (h[k] of
// point i at base[k * stride + i], base common to the wave) as the chunks end;
// only the facet code stays in a register.  On the device the store is a raw
// buffer store with a 32-bit lane offset, bounded by the log rows, so a point's
// log has to end below 4 GiB: up to LOG_POINTS points an instance.
constexpr int LOG_POINTS = (int)((1LL << 32) / (NREC * 4)) - 1;
struct LogSink {
    float* base;
    int stride;
    int i;
    int code;
#if defined(__HIP_DEVICE_COMPILE__)
    __amdgpu_buffer_rsrc_t rsrc;
#endif
    CPAB_HD void init(float* b, int s, int idx) {
        base = b;
        stride = s;
        i = idx;
        code = 0;
#if defined(__HIP_DEVICE_COMPILE__)
        rsrc = __builtin_amdgcn_make_buffer_rsrc(b, 0, NREC * 4u * (unsigned)s, 0x00020000);
#endif
    }
};

// n: index of the chunk just finished (the point's chunk count - 1).
CPAB_HD __forceinline__ void sink_chunk(LogSink& lg, int n, float h, int facet) {
    if (n < NREC) {
#if defined(__HIP_DEVICE_COMPILE__)
        // the builtin's data operand is an integer: pass the bits, not the value
        const unsigned at = ((unsigned)n * (unsigned)lg.stride + (unsigned)lg.i) * 4u;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(h), lg.rsrc, at, 0, 0);
#else
        lg.base[(size_t)n * lg.stride + lg.i] = h;
#endif
        lg.code = ((lg.code & ~3) | (n + 1)) | ((facet + 1) << (2 + 3 * n));
    }
}

CPAB_HD __forceinline__ void logged_chunk(const ChunkLog& lg, int k, float& h, int& facet) {
    h = lg.h[0];
#pragma unroll
    for (int j = 1; j < NREC; ++j)
        if (k == j) h = lg.h[j];
    facet = ((lg.code >> (2 + 3 * k)) & 7) - 1;
}

// ---------------------------------------------------------------------------
// one chunk of integration, D = 2, 3
//
// VALU issue bounds it (85-90% of the nominal rate in the plain 2D grid
// transform, transcendentals counted once), so what counts is instructions per
// wave and chunk, and a branch costs its whole body whenever one of 64 lanes
// takes it.  Hence the shared scalars of flow_at instead of a series vector and
// a polynomial per facet, one straight cull for all facets, then a loop over
// each lane's own remaining facet (0.5 trips per chunk on [4, 4] images) instead
// of four branches, and a root search that starts from the quadratic model (1.0
// Newton steps per chunk and wave instead of 2-3) and samples only where neither
// G'' nor G' has a certified sign (2% of a wave's chunks).  VALU instructions
// per wave of the 2D grid transform (4 points a lane): 2600 with the scalars
// alone, 2030 now.  [4, 4], 64 x 256^2 points, us per launch before / after:
// grid transform 88 / 63, its recomputing backward 208 / 144; fused with 3
// channels and 256 thetas: forward 491 / 448, backward 790 / 730-740;
// [3, 3, 3], 16 x 64^3: forward 192 / 162, backward 293 / 234.
// ---------------------------------------------------------------------------
template <int D>
CPAB_HD __forceinline__ void advance(PointState<D>& st, const CellTable<D>& tab, float tol0, Chunk<D>& ch) {
    const int c = st.c;
    load_affine<D>(tab, c, ch.M, ch.b);
    float v0[D];
    affine_apply<D>(ch.M, ch.b, st.q, v0);
    const float h = fminf(st.T, RHO * tab.inv_n[c]);
    powers<D>(ch.M, v0, ch.v);
    ch.iv = invariants<D>(ch.M);
    ch.f = flow_at<D>(ch.iv, h);
    float vn2 = 0.f;
#pragma unroll
    for (int a = 0; a < D; ++a) vn2 = fmaf(v0[a], v0[a], vn2);
    const float vn = fast_sqrt(vn2);
    // Bounds on the chunk (|n| = 1, |M| <= |M|_F, |M|_F h <= RHO, |cf_k| <=
    // |M|^(k-1) |v0| / k!):  the terms of G from s^3 on sum to at most
    // K3 s^3, K3 = |M|_F^2 |v0| e^RHO / 6, their derivative to 3 K3 s^2, and
    // |G''(s) - 2 cf2 - 6 cf3 s| <= K4 = |M|_F^3 |v0| h^2 e^RHO / 2.
    const float nrm = fast_rcp(tab.inv_n[c]);  // |M|_F (the bounds below carry margin for its last bit)
    const float mh = h * nrm;
    const float K = GROW * vn * nrm;
    const float K3 = K * nrm * (1.0f / 6.0f);

    // phase 1: cull, the same straight code for every facet slot (a wave runs
    // it once; a branch per facet would run nearly every body of a wave with
    // most lanes off)
    const float hK3 = h * h * K3, hh = 0.5f * h;
    unsigned live = 0u;
    int nbs[NF];
    cell_neighbours(tab, c, nbs);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
#if defined(__HIP_DEVICE_COMPILE__)
        // a 2D cell has a fourth facet only at the domain's boundary
        if (D == 2 && f == 3 && __ballot(nbs[3] >= 0) == 0) break;
#endif
        const float4 P = tab.pl[c * NF + f];
        const float n[3] = {P.x, P.y, P.z};
        float g0 = P.w, g1 = n[0] * v0[0], g2 = n[0] * ch.v[1][0];
#pragma unroll
        for (int a = 0; a < D; ++a) g0 = fmaf(n[a], st.q[a], g0);
#pragma unroll
        for (int a = 1; a < D; ++a) {
            g1 = fmaf(n[a], v0[a], g1);
            g2 = fmaf(n[a], ch.v[1][a], g2);
        }
        // G(s) <= g0 + g1 s + max(cf2, 0) s^2 + K3 s^3 on [0, h] (cf2 = g2 / 2),
        // a convex bound (its s^2 and s^3 coefficients are >= 0), so no
        // crossing when it is below 0 at h; a start on the facet counts as
        // G(0) = 0, and a convex bound that is 0 at 0 and below 0 at h is
        // below 0 in between
        const float bound = fmaf(h, fmaf(hh, fmaxf(g2, 0.f), hK3) + g1, g0 >= -tol0 ? 0.f : g0);
        live |= (!(bound < 0.f) & (nbs[f] >= 0)) ? 1u << f : 0u;
    }
    float tol1 = 0.f;
    if (live) {
        // Tangential band for an outward normal speed G'(0): the neighbouring
        // cells' FP32 fields agree on a shared facet only up to the rounding of
        // M q + b, whose terms can be much larger than |v0| where they cancel,
        // so both may round a vanishing normal speed to a small exit.  Inside
        // the band a start exit also needs G'' > 0 (the same side from both
        // cells for a tangent velocity); an inward G'(0) always follows the dip.
        float vabs = 0.f;
#pragma unroll
        for (int r = 0; r < D; ++r) {
            float t = fabsf(ch.b[r]);
#pragma unroll
            for (int a = 0; a < D; ++a) t = fmaf(fabsf(ch.M[r][a]), fabsf(st.q[a]), t);
            vabs += t;
        }
        tol1 = 1e-6f * vabs;
        // A velocity inside that band is rounding noise: the point sits on a
        // fixed point of the field at FP32 resolution (e.g. a domain corner
        // under zero_boundary) and moves by at most e^RHO |v0| h over the
        // chunk.  It crosses no facet in this chunk (otherwise the noise could
        // carry it back and forth across a facet through the fixed point, a
        // hop per chunk, until the chunk budget ran out).
        if (vn <= tol1) live = 0u;
    }
    // phase 2: the facets left, one of each lane at a time, keep the earliest
    // crossing (best, bf).  A facet whose first crossing lies in [0, h] with a
    // certified unique root has that bracket; starts on a facet, and facets
    // whose curvature and slope have no certified sign, are sampled for theirs.
    // A later facet is solved only where it is outside at the best root so far.
    // (One site each for the sampling and the root search: a second copy of
    // either costs scalar registers for its nested lane masks, which then
    // spill into vector lanes.)
    const float K4 = 0.5f * K * mh * mh;
    float best = h;
    int bf = -1;
#pragma unroll 1
    while (live) {
        const int f = __builtin_ctz(live);
        live &= live - 1u;
        const FacetG<D> F = facet_coeffs<D>(tab, c, f, st.q, ch.v, tol0);
        // G''(s) = 2 cf2 + 6 cf3 s + R(s), |R| <= K4, 6 cf3 = n.M^2 v0: the sign
        // of G'' is certified when the linear part keeps one sign with margin K4
        float g3;
        if constexpr (D == 2) g3 = fmaf(ch.iv.t, F.g[2], -(ch.iv.d * F.g[1]));
        else g3 = F.g[3];
        const float l0 = F.g[2], l1 = fmaf(g3, h, l0);
        const bool bent = fminf(l0, l1) > K4 || fmaxf(l0, l1) < -K4;
        // likewise G' = g1 + g2 s + R, |R| <= 3 K3 s^2, for a G that is too
        // straight for its curvature to have a certified sign
        const float e1 = fmaf(l0, h, F.g[1]), r1 = 3.f * hK3;
        const bool rising = fminf(F.g[1], e1) > r1, falling = fmaxf(F.g[1], e1) < -r1;
        float lo = 0.f, hi = h, glo = F.g[0], ghi = facet_g<D>(F, ch.f);
        const bool allow_start =
            !(st.zero_hops > 0 && tab.nb[c * NF + f] == st.came_from) && st.zero_hops < MAX_ZERO_HOPS;
        bool take = ghi > 0.f, sample;
        if (F.g[0] >= -tol0) {
            if (allow_start && (F.g[1] > tol1 || (F.g[1] >= 0.f && F.g[2] > 0.f))) {
                if (best > 0.f) {
                    best = 0.f;
                    bf = f;
                }
                continue;
            }
            // a clear start inwards that ends inside has no crossing in between
            // when G is convex or concave on the chunk
            sample = !(F.g[1] < -tol1 && bent && !take);
        } else {
            // G convex, concave or monotonic on [0, h], G(0) < 0: a positive G(h)
            // means exactly one crossing; otherwise only a concave G rising and
            // falling inside the chunk can cross
            sample = !(bent || rising || falling) ||
                     (!take && l0 < 0.f && F.g[1] > 0.f && !rising && facet_dg<D>(F, ch.f) < 0.f);
        }
        if (sample) {
            Bracket br;
            first_bracket<D>(F, ch.iv, h, tol0, tol1, allow_start, br);
            take = br.idx >= 1 && br.idx <= NSAMP;
            lo = br.lo;
            hi = br.hi;
            glo = br.glo;
            ghi = br.ghi;
        }
        if (!take || !(lo < best)) continue;
        if (best < hi) {
            hi = best;
            ghi = facet_g<D>(F, flow_at<D>(ch.iv, hi));
        }
        if (ghi > 0.f) {
            const float s = solve_bracket<D>(F, ch.iv, lo, hi, glo, ghi);
            if (s < best || bf < 0) {
                best = s;
                bf = f;
            }
        }
    }
    if (bf >= 0) ch.f = flow_at<D>(ch.iv, best);
    finish_chunk<D>(st, tab, best, bf, ch);
}

// Replays a chunk whose duration h and crossed facet bf (-1: none) are known
// (recorded by the forward): the same series and the same end-of-chunk update
// as advance, without the facet search, so the state comes out bit for bit
// as in the forward.
template <int D>
CPAB_HD __forceinline__ void replay(PointState<D>& st, const CellTable<D>& tab, float h, int bf, Chunk<D>& ch) {
    load_affine<D>(tab, st.c, ch.M, ch.b);
    float v0[D];
    affine_apply<D>(ch.M, ch.b, st.q, v0);
    powers<D>(ch.M, v0, ch.v);
    ch.iv = invariants<D>(ch.M);
    ch.f = flow_at<D>(ch.iv, h);
    finish_chunk<D>(st, tab, h, bf, ch);
}

// ---------------------------------------------------------------------------
// 1D: closed form
// ---------------------------------------------------------------------------
//
// Instruction bound like the others: 2.7 chunks per wave and point on 1024-point
// signals over 50 cells, most of it the library's expm1, log1p and exp and IEEE
// quotients.  The growth of a chunk that ends on a cell edge is the velocity
// ratio 1 + r.  The gradient's pass takes phi1 and phi2 from one Taylor sum for
// |z| <= 1 (nearly every chunk; at most 9.1e-8 off, the library's quotients 1.2e-7
// and 3.9e-7).  Hit times and positions are the forward's, bit for bit, in every
// pass, and the exponentials the library's: e^z from the Taylor sum would be 1.9e-7
// off at z = -1, a hit time by the hardware's logarithm and reciprocal 2.8e-7.
// us per launch, 4096 signals of 1024 points, before / after, with the table of
// whole-cell crossings: forward 74 / 50, backward 115 / 86.
// ---------------------------------------------------------------------------
// p1 = (e^z - 1)/z, p2 = (e^z - 1 - z)/z^2
CPAB_HD __forceinline__ void phis(float z, float& p1, float& p2) {
    if (fabsf(z) <= 1.f) {
        // sum_k z^k/(k+2)!, k < 10: the next term is below 1/12! = 2.1e-9
        constexpr float C[10] = {1.f / 2,    1.f / 6,     1.f / 24,     1.f / 120,     1.f / 720,
                                 1.f / 5040, 1.f / 40320, 1.f / 362880, 1.f / 3628800, 1.f / 39916800};
        float acc = C[9];
#pragma unroll
        for (int k = 8; k >= 0; --k) acc = fmaf(acc, z, C[k]);
        p2 = acc;
        p1 = fmaf(z, acc, 1.f);
    } else {
        const float em = expm1f(z);
        p1 = em / z;
        p2 = (em - z) / (z * z);
    }
}
CPAB_HD __forceinline__ float phi1(float z) {  // (e^z - 1)/z
    return (fabsf(z) < 1e-4f) ? fmaf(z, fmaf(z, 1.0f / 6.0f, 0.5f), 1.0f) : expm1f(z) / z;
}
CPAB_HD __forceinline__ float log1p_over(float r) {  // log1p(r)/r
    return (fabsf(r) < 1e-4f) ? fmaf(r, fmaf(r, 1.0f / 3.0f, -0.5f), 1.0f) : log1pf(r) / r;
}

// The point's cell map and whether it crosses the edge qb it moves towards in
// the time left: after th, into cell next, grown by e^(a th) = 1 + r.
struct Hit1 {
    float a, b, v0, qb, th, r;
    int next;
    bool right, crosses;
};
CPAB_HD __forceinline__ Hit1 hit1(const PointState<1>& st, const CellTable<1>& tab, int nx) {
    Hit1 h;
    const int c = st.c;
    const float q0 = st.q[0];
    h.a = tab.A[2 * c];
    h.b = tab.A[2 * c + 1];
    h.v0 = fmaf(h.a, q0, h.b);
    h.right = h.v0 > 0.f;
    h.next = h.right ? c + 1 : c - 1;
    h.qb = h.right ? (float)(c + 1) : (float)c;
    h.th = 0.f;
    h.r = 0.f;
    h.crosses = false;
    if (h.v0 != 0.f && h.next >= 0 && h.next < nx) {
        if (tab.hits && q0 == (h.right ? (float)c : (float)(c + 1))) {
            // from edge to edge: the same for every point
            const float2 f = tab.hits[2 * c + (h.right ? 1 : 0)];
            h.th = f.x;
            h.r = f.y;
            const bool back = (st.zero_hops > 0 && h.next == st.came_from && h.th <= ZERO_HOP);
            h.crosses = h.th < st.T && !back;
            return h;
        }
        const float dq = h.qb - q0;
        h.r = h.a * dq / h.v0;
        if (1.0f + h.r > 0.f && h.r < INFINITY) {  // infinite: beside a fixed point, for longer than any T
            h.th = fmaxf(dq / h.v0 * log1p_over(h.r), 0.f);
            const bool back = (st.zero_hops > 0 && h.next == st.came_from && h.th <= ZERO_HOP);
            h.crosses = h.th < st.T && !back;
        }
    }
    return h;
}
// Entry of CellTable::hits: the crossing of the whole cell c to the left (dir 0) or
// right, operation for operation that of a point that starts on the edge; a time
// beyond any where there is none.
CPAB_HD __forceinline__ float2 whole_cell(const CellTable<1>& tab, int c, int dir, int nx) {
    PointState<1> st;
    st.q[0] = dir ? (float)c : (float)(c + 1);
    st.T = INFINITY;
    st.c = c;
    st.came_from = -1;
    st.zero_hops = 0;
    st.iters = 0;
    const Hit1 h = hit1(st, tab, nx);
    float2 f;
    f.x = h.crosses && h.right == (dir == 1) ? h.th : INFINITY;
    f.y = h.r;
    return f;
}
CPAB_HD __forceinline__ void hop1(PointState<1>& st, const Hit1& h) {
    st.T = fmaxf(st.T - h.th, 0.f);
    st.zero_hops = (h.th <= ZERO_HOP) ? st.zero_hops + 1 : 0;
    st.came_from = st.c;
    st.c = h.next;
    st.q[0] = h.qb;
}
// The last chunk: the time left, inside the cell; returns e^(a T).
CPAB_HD __forceinline__ float end1(PointState<1>& st, const Hit1& h) {
    const float z = h.a * st.T;
    st.q[0] = fmaf(st.T * phi1(z), h.v0, st.q[0]);
    st.T = 0.f;
    return expf(z);
}

struct Chunk1 {
    float a, b, q0, h;
    int cell, facet, next;
    float q1;
};
CPAB_HD __forceinline__ void advance1(PointState<1>& st, const CellTable<1>& tab, int nx, Chunk1& ch) {
    const Hit1 h = hit1(st, tab, nx);
    ch.a = h.a; ch.b = h.b; ch.q0 = st.q[0];
    ch.cell = st.c;
    ch.h = h.crosses ? h.th : st.T;
    ch.facet = h.crosses ? (h.right ? 1 : 0) : -1;
    ch.next = h.crosses ? h.next : st.c;
    if (h.crosses) hop1(st, h);
    else end1(st, h);
    ch.q1 = st.q[0];
    st.iters++;
}

// The saltation factor v_next / v_prev of a crossing (1 for a continuous field), or
// its inverse for the adjoint; 1 where the divisor vanishes beside the other.  A
// quotient: the reciprocal of a subnormal velocity (theta near zero) overflows.
CPAB_HD __forceinline__ float saltation1(float vnum, float vden) {
    return fabsf(vden) > 1e-6f * fabsf(vnum) && vden != 0.f ? vnum / vden : 1.f;
}

// ---------------------------------------------------------------------------
// initial cell (the reference's lookup, libcpab/numpy/findcellidx.py, in FP32)
// ---------------------------------------------------------------------------
CPAB_HD __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

CPAB_HD __forceinline__ int find_cell1(float x, int nx) {
    float f = floorf(x * (float)nx);
    f = fminf(fmaxf(f, 0.f), (float)(nx - 1));
    return (int)f;
}

CPAB_HD __forceinline__ int find_cell2(float x, float y, int nx, int ny) {
    const float qx = x * (float)nx, qy = y * (float)ny;
    const int i = clampi((int)floorf(fminf(fmaxf(qx, 0.f), (float)nx)), 0, nx - 1);
    const int j = clampi((int)floorf(fminf(fmaxf(qy, 0.f), (float)ny)), 0, ny - 1);
    const int base = 4 * (i + j * nx);
    if (x <= 0.f) {
        if (y <= 0.f && qy < qx) return base;
        if (y >= 1.f && qy - (float)ny > -qx) return base + 2;
        return base + 3;
    }
    if (x >= 1.f) {
        if (y <= 0.f && -qy > qx - (float)nx) return base;
        if (y >= 1.f && qy - (float)ny > qx - (float)nx) return base + 2;
        return base + 1;
    }
    if (y <= 0.f) return base;
    if (y >= 1.f) return base + 2;
    const float fx = qx - (float)i, fy = qy - (float)j;
    if (fx < fy) return base + ((1.f - fx < fy) ? 2 : 3);
    return base + ((1.f - fx < fy) ? 1 : 0);
}

// top: largest coordinate the lookup keeps (libcpab/numpy/findcellidx.py
// clamps to 1 - 1e-8, which is 1 in FP32; the torch lookup of the reference's
// use_slow path clamps to 1 - 1e-4, libcpab/pytorch/findcellidx.py:112-114)
CPAB_HD __forceinline__ int find_cell3(float x, float y, float z, int nx, int ny, int nz, float top = 1.f) {
    float p[3] = {x, y, z};
    const int n[3] = {nx, ny, nz};
    const bool outside = x < 0.f || x > 1.f || y < 0.f || y > 1.f || z < 0.f || z > 1.f;
    if (outside) {
        // libcpab/numpy/findcellidx.py:85-108: push the point onto the boundary
        const float half = 0.5f;
        float d[3] = {x - half, y - half, z - half};
        const float ax = fabsf(d[0]), ay = fabsf(d[1]), az = fabsf(d[2]);
        const float push[3] = {(ax < ay && ax < az) ? half / nx : 0.f, (ay < ax && ax < az) ? half / ny : 0.f,
                               (az < ax && ax < ay) ? half / nz : 0.f};
        const float ab[3] = {ax, ay, az};
#pragma unroll
        for (int a = 0; a < 3; ++a)
            if (ab[a] > half) d[a] = copysignf(half - push[a], d[a]);
#pragma unroll
        for (int a = 0; a < 3; ++a) p[a] = d[a] + half;
    }
    int ijk[3];
    float loc[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float q = fminf(fmaxf(p[a], 0.f), top) * (float)n[a];
        ijk[a] = clampi((int)floorf(q), 0, n[a] - 1);
        loc[a] = q - (float)ijk[a];
    }
    int idx = 5 * (ijk[0] + ijk[1] * nx + ijk[2] * nx * ny);
    float lx = loc[0], ly = loc[1], lz = loc[2];
    if ((ijk[0] + ijk[1] + ijk[2]) & 1) {
        const float t = lx;
        lx = ly;
        ly = 1.f - t;
    }
    if (-lx - ly + lz >= 0.f) idx += 1;
    else if (lx + ly + lz - 2.f >= 0.f) idx += 2;
    else if (-lx + ly - lz >= 0.f) idx += 3;
    else if (lx - ly - lz >= 0.f) idx += 4;
    return idx;
}

template <int D>
CPAB_HD __forceinline__ int find_cell(const float (&x)[D], const int* nc) {
    if constexpr (D == 1) return find_cell1(x[0], nc[0]);
    else if constexpr (D == 2) return find_cell2(x[0], x[1], nc[0], nc[1]);
    else return find_cell3(x[0], x[1], x[2], nc[0], nc[1], nc[2]);
}

// ---------------------------------------------------------------------------
// per-point integration with optional Jacobian (pass 1)
// ---------------------------------------------------------------------------
template <int D>
CPAB_HD __forceinline__ void saltation_fwd(const CellTable<D>& tab, const Chunk<D>& ch, float (&J)[D][D]) {
    // J <- S J,  S = I + (v_next - v_prev) n^T / (n . v_prev)
    float Mn[D][D], bn[D], vp[D], vn[D];
    load_affine<D>(tab, ch.next, Mn, bn);
    affine_apply<D>(ch.M, ch.b, ch.q1, vp);
    affine_apply<D>(Mn, bn, ch.q1, vn);
    const float4 P = tab.pl[ch.cell * NF + ch.facet];
    const float n[3] = {P.x, P.y, P.z};
    float nv = 0.f, vv = 0.f;
#pragma unroll
    for (int a = 0; a < D; ++a) {
        nv = fmaf(n[a], vp[a], nv);
        vv = fmaf(vp[a], vp[a], vv);
    }
    if (fabsf(nv) <= 1e-6f * fast_sqrt(vv)) return;
    const float inv = fast_rcp(nv);
#pragma unroll
    for (int j = 0; j < D; ++j) {
        float nj = 0.f;
#pragma unroll
        for (int a = 0; a < D; ++a) nj = fmaf(n[a], J[a][j], nj);
#pragma unroll
        for (int r = 0; r < D; ++r) J[r][j] = fmaf((vn[r] - vp[r]) * inv, nj, J[r][j]);
    }
}

template <int D>
CPAB_HD __forceinline__ void saltation_adj(const CellTable<D>& tab, const Chunk<D>& ch, float (&mu)[D]) {
    // mu <- S^-T mu = mu - n ((v_next - v_prev) . mu) / (n . v_next)
    float Mn[D][D], bn[D], vp[D], vn[D];
    load_affine<D>(tab, ch.next, Mn, bn);
    affine_apply<D>(ch.M, ch.b, ch.q1, vp);
    affine_apply<D>(Mn, bn, ch.q1, vn);
    const float4 P = tab.pl[ch.cell * NF + ch.facet];
    const float n[3] = {P.x, P.y, P.z};
    float nv = 0.f, vv = 0.f, um = 0.f;
#pragma unroll
    for (int a = 0; a < D; ++a) {
        nv = fmaf(n[a], vn[a], nv);
        vv = fmaf(vn[a], vn[a], vv);
        um = fmaf(vn[a] - vp[a], mu[a], um);
    }
    if (fabsf(nv) <= 1e-6f * fast_sqrt(vv)) return;
    const float f = um * fast_rcp(nv);
#pragma unroll
    for (int a = 0; a < D; ++a) mu[a] = fmaf(-n[a], f, mu[a]);
}

// J <- exp(h M) J = sum_i e_i M^i J
template <int D>
CPAB_HD __forceinline__ void carry_jacobian(const Chunk<D>& ch, float (&J)[D][D]) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
        float w[D], acc[D];
#pragma unroll
        for (int r = 0; r < D; ++r) {
            w[r] = J[r][j];
            acc[r] = ch.f.e[0] * w[r];
        }
#pragma unroll
        for (int k = 1; k < D; ++k) {
            float m[D];
#pragma unroll
            for (int r = 0; r < D; ++r) {
                float t = ch.M[r][0] * w[0];
#pragma unroll
                for (int a = 1; a < D; ++a) t = fmaf(ch.M[r][a], w[a], t);
                m[r] = t;
            }
#pragma unroll
            for (int r = 0; r < D; ++r) {
                w[r] = m[r];
                acc[r] = fmaf(ch.f.e[k], m[r], acc[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < D; ++r) J[r][j] = acc[r];
    }
}

template <int D>
CPAB_HD __forceinline__ void init_point(PointState<D>& st, const float (&q)[D], int c0, float T) {
#pragma unroll
    for (int a = 0; a < D; ++a) st.q[a] = q[a];
    st.T = T;
    st.c = c0;
    st.came_from = -1;
    st.zero_hops = 0;
    st.iters = 0;
}

template <int D>
CPAB_HD __forceinline__ bool point_active(const PointState<D>& st) {
    return st.T > 0.f && st.iters < MAX_ITERS;
}

// One chunk of pass 1 (2D/3D): advance the point and carry J = dq(T)/dq0; with
// LOG the chunk goes into lg (a ChunkLog or a LogSink).
template <int D, bool WITHJ, bool LOG = false, class Log = ChunkLog>
CPAB_HD __forceinline__ void step_point(PointState<D>& st, const CellTable<D>& tab, int nx, float tol0,
                                        float (&J)[D][D], Log& lg) {
    static_assert(D > 1, "integrate carries 1D points itself");
    Chunk<D> ch;
    advance<D>(st, tab, tol0, ch);
    if constexpr (WITHJ) {
        carry_jacobian<D>(ch, J);
        if (ch.facet >= 0) saltation_fwd<D>(tab, ch, J);
    }
    // logged last, when the chunk's temporaries are dead
    if constexpr (LOG) {
        if constexpr (std::is_same<Log, LogSink>::value)
            sink_chunk(lg, st.iters - 1, ch.h, ch.facet);
        else
            log_chunk(lg, ch.h, ch.facet);
    }
}

template <int D>
CPAB_HD __forceinline__ void identity(float (&J)[D][D]) {
#pragma unroll
    for (int r = 0; r < D; ++r)
#pragma unroll
        for (int k = 0; k < D; ++k) J[r][k] = (r == k) ? 1.f : 0.f;
}

// A point that used up MAX_ITERS with time left: NaN, and counted.
template <int D, bool WITHJ>
CPAB_HD __forceinline__ void give_up(PointState<D>& st, float (&J)[D][D], int* unfinished) {
    const float nan = __builtin_nanf("");
    st.T = 0.f;
#pragma unroll
    for (int a = 0; a < D; ++a) st.q[a] = nan;
    if constexpr (WITHJ) {
#pragma unroll
        for (int r = 0; r < D; ++r)
#pragma unroll
            for (int k = 0; k < D; ++k) J[r][k] = nan;
    }
    if (unfinished) {
#if defined(__HIP_DEVICE_COMPILE__)
        // the operand is made opaque so that its register is set here, on the
        // rare path, and not hoisted out of the loop
        int one = 1;
        asm volatile("" : "+v"(one));
        atomicAdd(unfinished, one);
#else
        ++*unfinished;
#endif
    }
}

// Integrate one point for time T (pass 1 if WITHJ); with LOG its first NREC
// chunks go into lg for the backward to replay.  A point that uses up
// MAX_ITERS with time left ends as NaN (q and J) rather than short of its end,
// and adds 1 to *unfinished (nullable).  The check sits in the rare branch
// only, so the common path carries no extra live state.
template <int D, bool WITHJ, bool LOG = false, class Log = ChunkLog>
CPAB_HD __forceinline__ void integrate(float (&q)[D], int c0, float T, const CellTable<D>& tab, int nx, float tol0,
                                       float (&J)[D][D], Log& lg, int* unfinished = nullptr) {
    PointState<D> st;
    init_point<D>(st, q, c0, T);
    if constexpr (WITHJ) identity<D>(J);
    lg.code = 0;
    if constexpr (D == 1) {
        // the last chunk after the loop: its exponential runs once for all lanes,
        // whichever crossing each of them stopped after
        Hit1 h;
        bool last = false;
        while (st.T > 0.f) {
            h = hit1(st, tab, nx);
            last = !h.crosses;
            if (last) break;
            hop1(st, h);
            st.iters++;
            if constexpr (WITHJ) {
                const float vn = fmaf(tab.A[2 * st.c], h.qb, tab.A[2 * st.c + 1]);
                const float vp = fmaf(h.a, h.qb, h.b);
                J[0][0] *= (1.f + h.r) * saltation1(vn, vp);
            }
            if (st.iters >= MAX_ITERS && st.T > 0.f) give_up<D, WITHJ>(st, J, unfinished);
        }
        if (last) {
            const float grow = end1(st, h);
            if constexpr (WITHJ) J[0][0] *= grow;
        }
    } else {
        while (st.T > 0.f) {
            step_point<D, WITHJ, LOG, Log>(st, tab, nx, tol0, J, lg);
            if (st.iters >= MAX_ITERS && st.T > 0.f) give_up<D, WITHJ>(st, J, unfinished);
        }
    }
#pragma unroll
    for (int a = 0; a < D; ++a) q[a] = st.q[a];
}

template <int D, bool WITHJ>
CPAB_HD __forceinline__ void integrate(float (&q)[D], int c0, float T, const CellTable<D>& tab, int nx, float tol0,
                                       float (&J)[D][D], int* unfinished = nullptr) {
    ChunkLog lg;
    integrate<D, WITHJ, false>(q, c0, T, tab, nx, tol0, J, lg, unfinished);
}

// ---------------------------------------------------------------------------
// pass 2: gradient contribution of one chunk
// ---------------------------------------------------------------------------
// K[i][j] = int_0^h e_i(-s) al_j(s) ds: with mu(s) = exp(-s M^T) mu0 =
// sum_i e_i(-s) (M^T)^i mu0 and q(s) = q0 + sum_j al_j(s) M^j v0, the integral
// of mu(s) (q(s) - q0)^T over the chunk is sum_ij K[i][j] (M^T)^i mu0 (M^j v0)^T.
// Each K is h^(2+i+j) times a polynomial in the invariants of h M, the terms of
// total degree below KS in h M of the double series sum_{j,m} (-1)^j N^j (x) N^m
// / (j! (m+1)! (j+m+2)) with every power reduced by Cayley-Hamilton (exact
// rational coefficients, rounded to FP32).
template <int D>
CPAB_HD __forceinline__ void chunk_moments(const Invariants<D>& iv, float h, float (&K)[D][D]) {
    const float h2 = h * h, h3 = h2 * h, h4 = h2 * h2, tt = h * iv.t;
    if constexpr (D == 2) {
        const float dd = h2 * iv.d;
        K[0][0] = h2 * fmaf(dd, fmaf(dd, fmaf(dd, -0.00158730159f, fmaf(tt, fmaf(tt, 0.00111607143f,
                  -0.00297619048f), 0.0222222222f)), fmaf(tt, fmaf(tt, fmaf(tt, fmaf(tt, -0.000198412698f,
                  0.000992063492f), -0.00833333333f), 0.025f), -0.166666667f)), 0.5f);
        K[0][1] = h3 * fmaf(dd, fmaf(dd, fmaf(tt, 7.44047619e-05f, 0.00615079365f), fmaf(tt, fmaf(tt, fmaf(tt,
                  -9.92063492e-05f, -0.00257936508f), -0.00277777778f), -0.0583333333f)), fmaf(tt, fmaf(tt, fmaf(tt,
                  fmaf(tt, fmaf(tt, 2.48015873e-05f, 0.000198412698f), 0.00138888889f), 0.00833333333f),
                  0.0416666667f), 0.166666667f));
        K[1][0] = h3 * fmaf(dd, fmaf(dd, fmaf(tt, 0.0015625f, -0.00634920635f), fmaf(tt, fmaf(tt, fmaf(tt,
                  -0.00104166667f, 0.00575396825f), -0.0208333333f), 0.0666666667f)), fmaf(tt, fmaf(tt, fmaf(tt,
                  fmaf(tt, fmaf(tt, 0.000173611111f, -0.00119047619f), 0.00694444444f), -0.0333333333f), 0.125f),
                  -0.333333333f));
        K[1][1] = h4 * fmaf(dd, fmaf(dd, -0.0015625f, fmaf(tt, fmaf(tt, 0.00104166667f, -0.00257936508f),
                  0.0208333333f)), fmaf(tt, fmaf(tt, fmaf(tt, fmaf(tt, -0.000173611111f, 0.000793650794f),
                  -0.00694444444f), 0.0166666667f), -0.125f));
    } else {
        const float h5 = h4 * h, h6 = h3 * h3, ss = h2 * iv.sg, dd = h3 * iv.d;
        K[0][0] = h2 * fmaf(dd, fmaf(dd, -0.000669642857f, fmaf(ss, fmaf(tt, -0.000396825397f, 0.000992063492f),
                  fmaf(tt, fmaf(tt, fmaf(tt, 0.000198412698f, -0.000992063492f), 0.00833333333f), -0.025f))), 0.5f);
        K[0][1] = h3 * fmaf(dd, fmaf(ss, 0.00133928571f, fmaf(tt, fmaf(tt, -0.000496031746f, 0.00317460317f),
                  -0.0125f)), fmaf(ss, fmaf(ss, fmaf(tt, 4.96031746e-05f, 0.000198412698f), fmaf(tt, fmaf(tt,
                  fmaf(tt, -2.48015873e-05f, -0.000198412698f), -0.00138888889f), -0.00833333333f)), 0.166666667f));
        K[0][2] = h4 * fmaf(dd, fmaf(tt, 4.96031746e-05f, -0.00376984127f), fmaf(ss, fmaf(ss, 2.48015873e-05f,
                  fmaf(tt, fmaf(tt, -7.44047619e-05f, -0.000396825397f), -0.00138888889f)), fmaf(tt, fmaf(tt,
                  fmaf(tt, fmaf(tt, 2.48015873e-05f, 0.000198412698f), 0.00138888889f), 0.00833333333f),
                  0.0416666667f)));
        K[1][0] = h3 * fmaf(dd, fmaf(ss, 0.000694444444f, (tt * -0.00238095238f)), fmaf(ss, fmaf(ss, fmaf(tt,
                  0.000347222222f, -0.00119047619f), fmaf(tt, fmaf(tt, fmaf(tt, -0.000173611111f, 0.00119047619f),
                  -0.00694444444f), 0.0333333333f)), -0.333333333f));
        K[1][1] = h4 * fmaf(dd, fmaf(tt, -0.000694444444f, 0.00178571429f), fmaf(ss, fmaf(ss, -0.0015625f, fmaf(tt,
                  fmaf(tt, 0.000694444444f, -0.00178571429f), 0.0208333333f)), -0.125f));
        K[1][2] = h5 * fmaf(dd, 0.000694444444f, fmaf(ss, fmaf(tt, 0.000347222222f, 0.00515873016f), fmaf(tt,
                  fmaf(tt, fmaf(tt, -0.000173611111f, -0.00119047619f), -0.00694444444f), -0.0333333333f)));
        K[2][0] = h4 * fmaf(dd, 0.00178571429f, fmaf(ss, fmaf(ss, 0.000173611111f, fmaf(tt, fmaf(tt,
                  -0.000520833333f, 0.00238095238f), -0.00694444444f)), fmaf(tt, fmaf(tt, fmaf(tt, fmaf(tt,
                  0.000173611111f, -0.00119047619f), 0.00694444444f), -0.0333333333f), 0.125f)));
        K[2][1] = h5 * fmaf(ss, fmaf(tt, 0.00138888889f, -0.00595238095f), fmaf(tt, fmaf(tt, fmaf(tt,
                  -0.000520833333f, 0.00297619048f), -0.0138888889f), 0.05f));
        K[2][2] = h6 * fmaf(ss, -0.00138888889f, fmaf(tt, fmaf(tt, 0.000520833333f, -0.000992063492f),
                  0.0138888889f));
    }
}

// A chunk's dL/dA_q in G; carries mu to the chunk's end.
template <int D>
CPAB_HD __forceinline__ void chunk_grad(const Chunk<D>& ch, float (&mu)[D], float (&G)[D * (D + 1)]) {
    const FlowAt<D> fb = flow_at<D>(ch.iv, -ch.h);  // exp(-h M) and -int_0^h exp(-s M) ds
    float K[D][D];
    chunk_moments<D>(ch.iv, ch.h, K);
    float m[D], gbar[D], mend[D];
#pragma unroll
    for (int a = 0; a < D; ++a) {
        m[a] = mu[a];
        gbar[a] = -fb.al[0] * mu[a];
        mend[a] = fb.e[0] * mu[a];
    }
#pragma unroll
    for (int i = 0; i < D; ++i) {
        // m = (M^T)^i mu0, u = sum_j K[i][j] M^j v0
        float u[D];
#pragma unroll
        for (int a = 0; a < D; ++a) {
            float acc = K[i][0] * ch.v[0][a];
#pragma unroll
            for (int k = 1; k < D; ++k) acc = fmaf(K[i][k], ch.v[k][a], acc);
            u[a] = acc;
        }
#pragma unroll
        for (int r = 0; r < D; ++r)
#pragma unroll
            for (int a = 0; a < D; ++a)
                G[r * (D + 1) + a] = (i == 0) ? m[r] * u[a] : fmaf(m[r], u[a], G[r * (D + 1) + a]);
        if (i + 1 < D) {
            float t[D];
#pragma unroll
            for (int r = 0; r < D; ++r) {
                float acc = ch.M[0][r] * m[0];
#pragma unroll
                for (int a = 1; a < D; ++a) acc = fmaf(ch.M[a][r], m[a], acc);
                t[r] = acc;
            }
#pragma unroll
            for (int r = 0; r < D; ++r) {
                m[r] = t[r];
                gbar[r] = fmaf(-fb.al[i + 1], t[r], gbar[r]);
                mend[r] = fmaf(fb.e[i + 1], t[r], mend[r]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < D; ++r) {
#pragma unroll
        for (int a = 0; a < D; ++a) G[r * (D + 1) + a] = fmaf(gbar[r], ch.q0[a], G[r * (D + 1) + a]);
        G[r * (D + 1) + D] = gbar[r];
    }
#pragma unroll
    for (int a = 0; a < D; ++a) mu[a] = mend[a];
}

CPAB_HD __forceinline__ void chunk_grad1(const Chunk1& ch, float& mu, float (&G)[2]) {
    const float z = -ch.a * ch.h;
    float p1, p2;
    phis(z, p1, p2);
    G[0] = mu * fmaf(ch.h * ch.h, ch.b * p2, ch.q0 * ch.h);
    G[1] = mu * ch.h * p1;
    mu *= expf(z);
}

// ---------------------------------------------------------------------------
// wave-level deterministic accumulation of per-lane cell contributions
// ---------------------------------------------------------------------------
// Inclusive prefix sum over the 64 lanes (lane i gets lanes 0..i): scans
// inside each row of 16 (row_shr 1, 2, 4, 8), then the row totals carried by
// row_bcast:15 and row_bcast:31.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_take_int(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, true);
}
__device__ __forceinline__ int wave_inclusive_scan(int v) {
    v += dpp_take_int<0x111, 0xF>(v);
    v += dpp_take_int<0x112, 0xF>(v);
    v += dpp_take_int<0x114, 0xF>(v);
    v += dpp_take_int<0x118, 0xF>(v);
    v += dpp_take_int<0x142, 0xA>(v);
    v += dpp_take_int<0x143, 0xC>(v);
    return v;
}

// Minimum / maximum over the 64 lanes (same DPP pattern; lanes without a
// source keep the identity), read into a scalar.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_keep(int ident, int v) {
    return __builtin_amdgcn_update_dpp(ident, v, CTRL, ROWS, 0xF, false);
}
__device__ __forceinline__ int wave_min(int v) {
    v = min(v, dpp_keep<0x111, 0xF>(INT_MAX, v));
    v = min(v, dpp_keep<0x112, 0xF>(INT_MAX, v));
    v = min(v, dpp_keep<0x114, 0xF>(INT_MAX, v));
    v = min(v, dpp_keep<0x118, 0xF>(INT_MAX, v));
    v = min(v, dpp_keep<0x142, 0xA>(INT_MAX, v));
    v = min(v, dpp_keep<0x143, 0xC>(INT_MAX, v));
    return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_max(int v) {
    v = max(v, dpp_keep<0x111, 0xF>(INT_MIN, v));
    v = max(v, dpp_keep<0x112, 0xF>(INT_MIN, v));
    v = max(v, dpp_keep<0x114, 0xF>(INT_MIN, v));
    v = max(v, dpp_keep<0x118, 0xF>(INT_MIN, v));
    v = max(v, dpp_keep<0x142, 0xA>(INT_MIN, v));
    v = max(v, dpp_keep<0x143, 0xC>(INT_MIN, v));
    return __builtin_amdgcn_readlane(v, 63);
}

// ---------------------------------------------------------------------------
// Sums of P values over the 64 lanes, P = 2, 6 or 12 (D (D + 1)).
//
// Values are folded pairwise instead of one by one: a half-wave swap of two
// registers (v_permlane32_swap) and one add leave the first value's partial
// sums in lanes 0-31 and the second's in 32-63, a row swap (v_permlane16_swap)
// does the same between neighbouring rows of 16, and inside the rows two
// registers share one by a select on a lane bit.  12 instructions for P = 6
// and 27 for P = 12 instead of 36 and 72 DPP adds, and the totals end in
// different lanes, so one LDS add stores them all.  Every step is a fixed
// order of additions.  us per launch, DPP adds / this: backward of [3, 3, 3] on
// 16 x 64^3 points (5.5 cells per wave and round) 260 / 237, of [2, 2, 2] on
// 16 clouds of 25001 points (every lane its own cell) 71 / 51; 2D (2.7 cells)
// 732 / 730.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float fold_halves(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float fold_rows(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// v plus w of the lane CTRL pairs this one with
template <int CTRL>
__device__ __forceinline__ float pair_add(float v, float w) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(w), CTRL, 0xF, 0xF, true));
}
constexpr int PAIR_8 = 0x128;  // row_ror:8          lane ^ 8
constexpr int PAIR_7 = 0x141;  // row_half_mirror    lane ^ 7
constexpr int PAIR_2 = 0x4E;   // quad_perm 2,3,0,1  lane ^ 2
constexpr int PAIR_1 = 0xB1;   // quad_perm 1,0,3,2  lane ^ 1

// The value index whose total fold_values leaves in this lane, if the lane is
// the one that stores it, else -1.
template <int P>
__device__ __forceinline__ int fold_id() {
    const int lane = __lane_id(), row = lane >> 4, in = lane & 15;
    if constexpr (P == 2) {
        return (in == 0 && !(row & 1)) ? row >> 1 : -1;
    } else if constexpr (P == 6) {
        if (in == 0) return 2 * (row & 1) + (row >> 1);
        return (in == 8 && !(row & 1)) ? 4 + (row >> 1) : -1;
    } else {
        static_assert(P == 12, "P = D (D + 1)");
        const int k = 2 * (row & 1) + (row >> 1);
        return in == 0 ? k : (in == 8 ? 4 + k : (in == 4 ? 8 + k : -1));
    }
}
template <int P>
__device__ __forceinline__ float fold_values(const float (&v)[P]) {
    float w[P / 2];
#pragma unroll
    for (int i = 0; i < P / 2; ++i) w[i] = fold_halves(v[2 * i], v[2 * i + 1]);
    float y;
    if constexpr (P == 2) {
        y = fold_rows(w[0], w[0]);
        y = pair_add<PAIR_8>(y, y);
        y = pair_add<PAIR_7>(y, y);
    } else {
        const int lane = __lane_id();
        const float x0 = fold_rows(w[0], w[1]);
        const float x1 = P == 6 ? fold_rows(w[2], w[2]) : fold_rows(w[2], w[3 % (P / 2)]);
        y = pair_add<PAIR_8>((lane & 8) ? x1 : x0, (lane & 8) ? x0 : x1);
        if constexpr (P == 6) {
            y = pair_add<PAIR_7>(y, y);
        } else {
            float x2 = fold_rows(w[4 % (P / 2)], w[5 % (P / 2)]);
            x2 = pair_add<PAIR_8>(x2, x2);
            y = pair_add<PAIR_7>((lane & 4) ? x2 : y, (lane & 4) ? y : x2);
        }
    }
    y = pair_add<PAIR_2>(y, y);
    return pair_add<PAIR_1>(y, y);
}

// Adds g (P values) of every lane with cell >= 0 into acc[cell*P + p] of this
// wave's LDS region; the lanes sharing a cell are summed across the wave in a
// fixed order, and each total is added by the lane that holds it (LDS float
// adds, one lane per address, in program order).  Must be reached by all
// lanes of the wave.
template <int P>
__device__ __forceinline__ void wave_accumulate(float* acc, int cell, const float (&g)[P]) {
    const int id = fold_id<P>();
    float* mine_acc = acc + id;
    uint64_t pending = __ballot(cell >= 0);
    while (pending) {
        const int leader = __ffsll((unsigned long long)pending) - 1;
        const int c0 = __builtin_amdgcn_readlane(cell, leader);
        const bool mine = (cell == c0);
        pending &= ~__ballot(mine);
        float v[P];
#pragma unroll
        for (int p = 0; p < P; ++p) v[p] = mine ? g[p] : 0.f;
        const float tot = fold_values<P>(v);
        int off = c0 * P;
        // the product stays scalar: folded into the lane address it would be a
        // 64-bit multiply-add in every lane
        asm volatile("" : "+s"(off));
        if (id >= 0) atomicAdd(mine_acc + off, tot);
    }
}

}  // namespace cpab
