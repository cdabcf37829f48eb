// mpm_diff.hip -- reverse pass of one CPUDIFF substep on gfx950.
//
// Follows mpm_adjoint.rs backward_step (:142-496) for the forward of
// mpm_cpu_diff.rs step_once_record (:421-588): corotated-SVK stress, floor
// plane, explicit APIC.  The forward substep is
//   P2G (mass, momentum + stress) -> grid (v = p/m, gravity, floor)
//   -> G2P (v, C) -> x += dt v, F = (I + dt C) F,
// and its reverse runs as three launches over the substep's pre-state, which
// the host recomputes from a checkpoint (k_adj_fused merges the reverse P2G
// of one substep with the reverse G2P of the previous one):
//   k_adj_g2p   reverse of G2P and of the x/F advance.  Gathers grid v like
//               G2P and scatters dJ/d(grid v) = sum w (gv' + 4/dx^2 gC' d)
//               with the forward's block scatter (the same form as P2G's
//               w (m v + A d), with m = 0), so it reuses the LDS fixed-point
//               partials and the sorted chunk list.
//   k_adj_grid  reverse of the grid update per active cell:
//               dJ/dp = M(dJ/dv) / m, dJ/dm = -p . M(dJ/dv) / m^2, where M is
//               the floor's mask replayed from the pre-update momentum.
//   k_adj_p2g   reverse of P2G, of the stress and of the SVD: gathers
//               (dJ/dm, dJ/dp), and runs the PK1 and SVD adjoints in FP64
//               (mpm_cpu_diff.rs:330-379, dense3.rs:321-372).
// Particle adjoints live in NADJ planes in the state's slot order; the
// per-particle dJ/dE and the per-chunk (dJ/dmu, dJ/dlambda) sums accumulate
// over substeps (StateAdjoint's g_mu/g_lambda, mpm_adjoint.rs:76-113).
#include "mpm_scatter.hpp"

namespace mpm {

namespace {

// 1/x in f64 from the f32 reciprocal and two Newton steps (x > 0, normal f32).
__device__ __forceinline__ double rcp_f64(double x) {
    double r = (double)__frcp_rn((float)x);
    r = r * (2.0 - x * r);
    r = r * (2.0 - x * r);
    return r;
}

// safe_inv_sq_diff (dense3.rs:496-499) with ADJ_SVD_EPS = 1e-12 (:295).
__device__ __forceinline__ double safe_inv_sq_diff(double a, double b) {
    const double d = b * b - a * a;
    return d * rcp_f64(d * d + 1.0e-24);
}

struct Dm3 {
    double a[9];
    __device__ double& operator()(int i, int j) { return a[3 * i + j]; }
    __device__ double operator()(int i, int j) const { return a[3 * i + j]; }
};

__device__ __forceinline__ double warp_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

}  // namespace

// A block's box of grid cells in LDS for the gathers of its particles: the
// bounding box of their stencils, cells outside the grid as zeros (which add
// nothing to any of the gathers' sums).  `cells` null: not staged.
struct Staged {
    const float4* cells;
    int o[3], d[3];
    // index of the node (0, 0, 0) of a stencil at b, or -1 when not inside
    __device__ __forceinline__ int find(const int* b) const {
        bool in = cells != nullptr;
#pragma unroll
        for (int k = 0; k < 3; ++k) in = in && b[k] >= o[k] && b[k] + 2 < o[k] + d[k];
        return in ? (b[0] - o[0]) + d[0] * ((b[1] - o[1]) + d[1] * (b[2] - o[2])) : -1;
    }
};

// Stencil base of the particle in `slot` of planes ps; `on`: the particle is
// the block's and its stencil has not left its sorted neighbourhood (an
// escaped one reads global memory and would blow up the box).
__device__ __forceinline__ bool staged_base(const StepArgs& a, const SceneDev& sc, const Chunk& ch, const float* ps,
                                            uint32_t slot, bool active, int* b) {
    b[0] = b[1] = b[2] = 0;
    if (!active) return false;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        b[k] = int(floorf(fmaf(ps[(size_t)(CX + k) * a.cap + slot] - sc.origin[k], sc.inv_dx, -0.5f)));
    return !stencil_escapes(sc, ch, a.sorted_keys[slot], b);
}

// Joins the waves' stencil boxes (min and max base per axis) of up to two
// gathers through `red`.  Every thread calls it.
constexpr int NO_BASE = 0x3fffffff;
template <int N>
__device__ __forceinline__ void block_boxes(const bool (&on)[N], const int (&b)[N][3], int (*red)[WAVES][6],
                                            int (&lo)[N][3], int (&hi)[N][3]) {
    const int lane = threadIdx.x & 63, wave = wave_id();
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int l = wave_min(on[n] ? b[n][k] : NO_BASE), h = wave_max(on[n] ? b[n][k] : -NO_BASE);
            if (lane == 0) {
                red[n][wave][k] = l;
                red[n][wave][3 + k] = h;
            }
        }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[n][k] = red[n][0][k];
            hi[n][k] = red[n][0][3 + k];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) {
                lo[n][k] = min(lo[n][k], red[n][w][k]);
                hi[n][k] = max(hi[n][k], red[n][w][3 + k]);
            }
            lo[n][k] = __builtin_amdgcn_readfirstlane(lo[n][k]);
            hi[n][k] = __builtin_amdgcn_readfirstlane(hi[n][k]);
        }
}

// Loads the cells of stencils with bases lo .. hi into `to` (LDS_CELLS); the
// caller puts a barrier before the first read.
__device__ __forceinline__ Staged stage_box(const SceneDev& sc, const float4* __restrict__ grid, const int* lo,
                                            const int* hi, float4* to) {
    Staged s;
    s.cells = nullptr;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        s.o[k] = lo[k];
        s.d[k] = hi[k] - lo[k] + 3;
    }
    // no base at all (hi < lo), or a box that cannot fit
    if (s.d[0] < 3 || s.d[1] < 3 || s.d[2] < 3 || s.d[0] > LDS_CELLS || s.d[1] > LDS_CELLS || s.d[2] > LDS_CELLS ||
        s.d[0] * s.d[1] > LDS_CELLS || s.d[0] * s.d[1] * s.d[2] > LDS_CELLS)
        return s;
    const int vol = s.d[0] * s.d[1] * s.d[2];
    const float inv_x = 1.0f / float(s.d[0]), inv_y = 1.0f / float(s.d[1]);
    constexpr int PER = 4;  // loads in flight per thread
#pragma unroll 1
    for (int i0 = 0; i0 < vol; i0 += PER * BLOCK) {
        float4 v[PER];
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int i = i0 + int(threadIdx.x) + u * BLOCK;
            v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            // exact for the box's small integers, as in stage_gather_box
            const int r = int((float(i) + 0.5f) * inv_x), z = int((float(r) + 0.5f) * inv_y);
            const int ix = s.o[0] + (i - r * s.d[0]), iy = s.o[1] + (r - z * s.d[1]), iz = s.o[2] + z;
            if (i < vol && in_grid(sc, ix, iy, iz)) v[u] = grid[cell_index(sc, ix, iy, iz)];
        }
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int i = i0 + int(threadIdx.x) + u * BLOCK;
            if (i < vol) to[i] = v[u];
        }
    }
    s.cells = to;
    return s;
}

// The gathers' arithmetic is written out with its fused operations (and the
// compiler's own fusing switched off): a gradient's last bits depend on which
// products are rounded, and as the compiler fuses within a basic block only,
// they would change with every change of the code around the sums.
__device__ __forceinline__ float dot3(float a0, float b0, float a1, float b1, float a2, float b2) {
#pragma clang fp contract(off)
    return fmaf(a2, b2, fmaf(a0, b0, a1 * b1));
}

// Quadratic stencil of a position: first node, offset, weights, derivatives.
struct AdjStencil {
    int b[3];
    float fx[3], w[3][3], dw[3][3];
    __device__ __forceinline__ AdjStencil(const SceneDev& sc, const float* x) {
#pragma clang fp contract(off)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float r = x[k] - sc.origin[k];
            const float bf = floorf(fmaf(r, sc.inv_dx, -0.5f));
            b[k] = int(bf);
            fx[k] = fmaf(r, sc.inv_dx, -bf);
            const float p = 1.5f - fx[k], q = fx[k] - 1.0f, s = fx[k] - 0.5f;
            w[k][0] = 0.5f * p * p;
            w[k][1] = fmaf(-q, q, 0.75f);
            w[k][2] = 0.5f * s * s;
            dw[k][0] = -p;
            dw[k][1] = -2.0f * q;
            dw[k][2] = s;
        }
    }
};

// One z-plane of the sums over a stencil's nodes g, row by row (fixed j, k):
// with the node term
// u_jk + i c0, u_jk = u0 + j c1 + k c2, and h = (MASS ? m g.x : 0) + G . u,
// G the node's vector (MASS: g.yzw, else g.xyz),
//   S = sum w G,  M = sum w G (i, j, k)^T,
//   acc = (sum w1 w2 Sdw, sum dw1 w2 Sw, sum w1 dw2 Sw),
// Sw = sum_i w0 h, Sdw = sum_i dw0 h.  fetch(i, j, k) gives a node, zero
// outside the grid.
template <bool MASS, class Fetch>
__device__ __forceinline__ void adj_plane(int k, float wk, float dwk, const AdjStencil& st, float m, const float* u0,
                                          const float* c0, const float* c1, const float* c2, Fetch fetch, float* S,
                                          float* M, float* acc) {
#pragma clang fp contract(off)
    const float wi[3] = {0.f, st.w[0][1], 2.0f * st.w[0][2]};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const float wjk = st.w[1][j] * wk;
        float u[3], rs[3] = {0.f, 0.f, 0.f}, ri[3] = {0.f, 0.f, 0.f}, Sw = 0.f, Sdw = 0.f;
#pragma unroll
        for (int r = 0; r < 3; ++r) u[r] = fmaf(float(k), c2[r], fmaf(float(j), c1[r], u0[r]));
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const float4 g = fetch(i, j, k);
            const float G[3] = {MASS ? g.y : g.x, MASS ? g.z : g.y, MASS ? g.w : g.z};
            float v[3], h;
#pragma unroll
            for (int r = 0; r < 3; ++r) v[r] = fmaf(float(i), c0[r], u[r]);
            if (!MASS) {
                h = dot3(v[0], G[0], v[1], G[1], v[2], G[2]);
            } else {
                h = i == 0 ? fmaf(m, g.x, v[0] * G[0]) : fmaf(v[0], G[0], m * g.x);
                h = fmaf(v[2], G[2], fmaf(v[1], G[1], h));
            }
            Sw = fmaf(st.w[0][i], h, Sw);
            Sdw = fmaf(st.dw[0][i], h, Sdw);
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                rs[r] = fmaf(st.w[0][i], G[r], rs[r]);
                if (i > 0) ri[r] = fmaf(wi[i], G[r], ri[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            S[r] = fmaf(wjk, rs[r], S[r]);
            M[3 * r] = fmaf(wjk, ri[r], M[3 * r]);
            M[3 * r + 1] = fmaf(float(j) * wjk, rs[r], M[3 * r + 1]);
            M[3 * r + 2] = fmaf(float(k) * wjk, rs[r], M[3 * r + 2]);
        }
        acc[0] = fmaf(wjk, Sdw, acc[0]);
        acc[1] = fmaf(st.dw[1][j] * wk, Sw, acc[1]);
        acc[2] = fmaf(st.w[1][j] * dwk, Sw, acc[2]);
    }
}

// The sums over a stencil from the block's staged cells, or from global memory
// for waves with a stencil outside them (rolled: it is rare, and 27 nodes of
// code twice crowd the instruction cache: 340 us of k_adj_fused instead of 367;
// the common one rolled as well costs 26 instead of 13 us of k_adj_p2g on one
// scene of 65,536 particles).
template <bool MASS>
__device__ __forceinline__ void adj_gather(const SceneDev& sc, const float4* __restrict__ grid, const Staged& box,
                                           const AdjStencil& st, float m, const float* u0, const float* c0,
                                           const float* c1, const float* c2, float* S, float* M, float* acc) {
#pragma unroll
    for (int r = 0; r < 3; ++r) S[r] = acc[r] = M[3 * r] = M[3 * r + 1] = M[3 * r + 2] = 0.f;
    const int at = box.find(st.b);
    if (__all(at >= 0)) {
        const int dx = box.d[0], dxy = box.d[0] * box.d[1];
        const auto fetch = [&](int i, int j, int k) { return box.cells[at + i + dx * j + dxy * k]; };
#pragma unroll
        for (int k = 0; k < 3; ++k)
            adj_plane<MASS>(k, st.w[2][k], st.dw[2][k], st, m, u0, c0, c1, c2, fetch, S, M, acc);
    } else {
        const auto fetch = [&](int i, int j, int k) {
            const int ix = st.b[0] + i, iy = st.b[1] + j, iz = st.b[2] + k;
            return in_grid(sc, ix, iy, iz) ? grid[cell_index(sc, ix, iy, iz)] : make_float4(0.f, 0.f, 0.f, 0.f);
        };
        float w0 = st.w[2][0], w1 = st.w[2][1], d0 = st.dw[2][0], d1 = st.dw[2][1];
#pragma unroll 1
        for (int k = 0; k < 3; ++k) {
            adj_plane<MASS>(k, w0, d0, st, m, u0, c0, c1, c2, fetch, S, M, acc);
            w0 = w1;
            d0 = d1;
            w1 = st.w[2][2];
            d1 = st.dw[2][2];
        }
    }
}

// Reverse of G2P and of the x/F advance for the particle in `slot` of the
// pre-state a.ps with grid velocity a.gv (mpm_adjoint.rs:196-305).  On entry
// gx, gv, gC, gF are dJ/d(post-state); on return gx holds the G2P part of
// dJ/dx (plus the pass-through), gF = (I + dt C')^T dJ/dF', and sp the
// scatter of dJ/d(grid v).
__device__ __forceinline__ void adj_g2p_particle(const StepArgs& a, const SceneDev& sc, const Chunk& ch, uint32_t slot,
                                                 float* gx, const float* gv, const float* gC, float* gF, Scatter& sp,
                                                 const Staged& box) {
#pragma clang fp contract(off)
    const uint32_t cap = a.cap;
    const float* __restrict__ ps = a.ps;
    const float dt = a.dt;
    float x[3], F[9];
#pragma unroll
    for (int k = 0; k < 3; ++k) x[k] = ps[(size_t)(CX + k) * cap + slot];
#pragma unroll
    for (int k = 0; k < 9; ++k) F[k] = ps[(size_t)(CF + k) * cap + slot];
    // x' = x + dt v', F' = (I + dt C') F  =>  dJ/dv' += dt dJ/dx',
    // dJ/dC' += dt dJ/dF' F^T (mpm_adjoint.rs:196-247)
    float gvp[3], B[9];
    const float s4 = 4.0f * sc.inv_dx * sc.inv_dx;
#pragma unroll
    for (int k = 0; k < 3; ++k) gvp[k] = fmaf(gx[k], dt, gv[k]);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            B[3 * i + j] = s4 * fmaf(dt, dot3(gF[3 * i], F[3 * j], gF[3 * i + 1], F[3 * j + 1], gF[3 * i + 2],
                                              F[3 * j + 2]),
                                     gC[3 * i + j]);
    const AdjStencil st(sc, x);
    // G2P reverse (mpm_adjoint.rs:249-305): with B = 4/dx^2 dJ/dC',
    //   dJ/dx += sum grad(w) (v_i . (dJ/dv' + B d)) - B^T sum w v_i
    // in adj_gather's rows: d = ((i, j, k) - fx) dx, the gradient sum is
    // idx acc, and C' = 4/dx^2 sum w v_i d^T = 4/dx (M - S fx^T).
    const float dx = sc.dx, idx = sc.inv_dx;
    float c0[3], c1[3], c2[3], u0[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        c0[r] = dx * B[3 * r];
        c1[r] = dx * B[3 * r + 1];
        c2[r] = dx * B[3 * r + 2];
        u0[r] = gvp[r] - dot3(c0[r], st.fx[0], c1[r], st.fx[1], c2[r], st.fx[2]);
    }
    float vn[3], Mv[9], acc[3];
    adj_gather<false>(sc, a.gv, box, st, 0.f, u0, c0, c1, c2, vn, Mv, acc);
    float Cn[9];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) Cn[3 * r + c] = s4 * dx * fmaf(-vn[r], st.fx[c], Mv[3 * r + c]);
#pragma unroll
    for (int k = 0; k < 3; ++k) gx[k] += fmaf(acc[k], idx, -dot3(B[k], vn[0], B[3 + k], vn[1], B[6 + k], vn[2]));
    // dJ/dF (pre) = (I + dt C')^T dJ/dF'
    float nF[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            nF[3 * i + j] = fmaf(dt, dot3(Cn[i], gF[j], Cn[3 + i], gF[3 + j], Cn[6 + i], gF[6 + j]), gF[3 * i + j]);
#pragma unroll
    for (int k = 0; k < 9; ++k) gF[k] = nF[k];
    // dJ/d(grid v_i) += w (dJ/dv' + B d): the P2G form with m = 0
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        sp.b[k] = st.b[k];
        sp.fx[k] = st.fx[k];
        sp.mv[k] = gvp[k];
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) sp.A[k] = B[k];
    sp.m = 0.f;
    sp.on = true;
    sp.esc = stencil_escapes(sc, ch, a.sorted_keys[slot], sp.b);
}

// P2G reverse (mpm_adjoint.rs:389-487): with gw = sum w dJ/dp_i and
// T = sum w dJ/dp_i d^T:  dJ/dv = m gw, dJ/dC = m T, dJ/dstress = 4/dx^2 T,
// dJ/dx = sum grad(w) (dJ/dp_i . (m v + A d) + m dJ/dm_i) - A^T gw, in
// adj_gather's rows with T = dx (M - gw fx^T).  A = m C + 4/dx^2 stress
// (stress = -dt vol P F^T) as the forward scattered it: the tape holds it in
// the planes `aff`, so the FP64 SVD is not live across the gather.
__device__ __forceinline__ void adj_p2g_gather(const StepArgs& a, const float4* __restrict__ gadj,
                                               const float* __restrict__ aff, const SceneDev& sc, uint32_t slot, float m,
                                               float* gx, float* gv, float* T, const Staged& box) {
#pragma clang fp contract(off)
    const uint32_t cap = a.cap;
    const float* __restrict__ ps = a.ps;
    float x[3], v[3], A[9];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        x[k] = ps[(size_t)(CX + k) * cap + slot];
        v[k] = ps[(size_t)(CV + k) * cap + slot];
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) A[k] = aff[(size_t)k * cap + slot];
    const AdjStencil st(sc, x);
    const float dx = sc.dx, idx = sc.inv_dx;
    float c0[3], c1[3], c2[3], u0[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        c0[r] = dx * A[3 * r];
        c1[r] = dx * A[3 * r + 1];
        c2[r] = dx * A[3 * r + 2];
        u0[r] = fmaf(v[r], m, -dot3(c0[r], st.fx[0], c1[r], st.fx[1], c2[r], st.fx[2]));
    }
    float gw[3], Mt[9], acc[3];
    adj_gather<true>(sc, gadj, box, st, m, u0, c0, c1, c2, gw, Mt, acc);
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) T[3 * r + c] = dx * fmaf(-gw[r], st.fx[c], Mt[3 * r + c]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        gx[k] += fmaf(acc[k], idx, -dot3(A[k], gw[0], A[3 + k], gw[1], A[6 + k], gw[2]));
        gv[k] = m * gw[k];
    }
}

// Reverse of P2G, of the stress and of the SVD for the particle in `slot`
// of the pre-state a.ps, gathering (dJ/dm, dJ/dp) from gadj
// (mpm_adjoint.rs:389-487, mpm_cpu_diff.rs:330-379, dense3.rs:321-372).  On
// entry gx, gF hold the reverse G2P's output; on return gx, gv, gC, gF are
// dJ/d(pre-state), gE has dJ/dE_p added, and (amu, alam) are the particle's
// dJ/dmu, dJ/dlambda.
__device__ __forceinline__ void adj_p2g_particle(const StepArgs& a, const float4* __restrict__ gadj,
                                                 const float* __restrict__ aff, const SceneDev& sc, uint32_t slot,
                                                 float* gx, float* gF, float* gv, float* gC, float& gE, double& amu,
                                                 double& alam, const Staged& box) {
    const uint32_t cap = a.cap;
    const float* __restrict__ ps = a.ps;
    const float dt = a.dt;
    const float m = ps[(size_t)CMASS * cap + slot];
    float T[9];
    adj_p2g_gather(a, gadj, aff, sc, slot, m, gx, gv, T, box);
    // corotated-SVK PK1 from the FP64 SVD (mpm_cpu_diff.rs:279-287)
    float F[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) F[k] = ps[(size_t)(CF + k) * cap + slot];
    const float vol = ps[(size_t)CVOL * cap + slot];
    float mu = sc.mu, lam = sc.lam;
    if (a.has_E) {
        const float E = ps[(size_t)CE * cap + slot];
        mu = E / (2.0f * (1.0f + sc.poisson));
        lam = E * sc.poisson / ((1.0f + sc.poisson) * (1.0f - 2.0f * sc.poisson));
    }
    double U[9], s[3], V[9];
    svd3_f64_raw(F, U, s, V);
    svd3_signs<MODEL_CPUDIFF>(U, s, V);
    const double dmu = mu, dlam = lam;
    const double trsi = s[0] + s[1] + s[2] - 3.0;
    Dm3 P;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double r = U[3 * i] * V[3 * j] + U[3 * i + 1] * V[3 * j + 1] + U[3 * i + 2] * V[3 * j + 2];
            const double fr = U[3 * i] * s[0] * V[3 * j] + U[3 * i + 1] * s[1] * V[3 * j + 1] +
                              U[3 * i + 2] * s[2] * V[3 * j + 2];
            P(i, j) = 2.0 * dmu * (fr - r) + dlam * trsi * r;
        }
    const float s4 = 4.0f * sc.inv_dx * sc.inv_dx;
    const double coef = -(double)dt * (double)vol;
#pragma unroll
    for (int k = 0; k < 9; ++k) gC[k] = m * T[k];
    // stress = coef P F^T with dJ/dstress = s4 T:
    //   dJ/dP = coef s4 T F,  dJ/dF += coef s4 T^T P
    Dm3 aP, gf;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            aP(i, j) = coef * (double)s4 *
                       ((double)T[3 * i] * F[j] + (double)T[3 * i + 1] * F[3 + j] + (double)T[3 * i + 2] * F[6 + j]);
            gf(i, j) = (double)gF[3 * i + j] +
                       coef * (double)s4 *
                           ((double)T[i] * P(0, j) + (double)T[3 + i] * P(1, j) + (double)T[6 + i] * P(2, j));
        }
    // corotated_pk1_adjoint (mpm_cpu_diff.rs:330-379), in the rotated
    // frame: with Ut aP V = Q, aU = aP V (2mu Sd + cr I) - ..., the SVD
    // adjoint only needs Ut aU, Vt aV, so form them directly.
    Dm3 Q;  // U^T aP V
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            double acc = 0.0;
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const double pv = aP(r, 0) * V[j] + aP(r, 1) * V[3 + j] + aP(r, 2) * V[6 + j];
                acc += U[3 * r + i] * pv;
            }
            Q(i, j) = acc;
        }
    const double cr = -2.0 * dmu + dlam * trsi;
    const double r_dot = Q(0, 0) + Q(1, 1) + Q(2, 2);  // <R, aP> = tr(U^T aP V)
    // aU = aP V (2mu Sd) + cr aP V  ->  Ut aU = Q (2mu Sd + cr I)
    // aV = aP^T U (2mu Sd) + cr aP^T U  ->  Vt aV = Q^T (2mu Sd + cr I)
    Dm3 UaU, VaV;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double dj = 2.0 * dmu * s[j] + cr;
            UaU(i, j) = Q(i, j) * dj;
            VaV(i, j) = Q(j, i) * dj;
        }
    double aS[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) aS[i] = 2.0 * dmu * Q(i, i) + dlam * r_dot;
    // <Fr - R, aP> = sum_i (s_i - 1) Q_ii
    amu = 2.0 * ((s[0] - 1.0) * Q(0, 0) + (s[1] - 1.0) * Q(1, 1) + (s[2] - 1.0) * Q(2, 2));
    alam = trsi * r_dot;
    // adj_svd3 (dense3.rs:321-372): dJ/dF += U M V^T,
    //   M = diag(aS) + (f o om_u) Sd + Sd (f o om_v),
    //   om_u = Ut aU - aU^T U = UaU - UaU^T, om_v = VaV - VaV^T
    const double f01 = safe_inv_sq_diff(s[0], s[1]);
    const double f02 = safe_inv_sq_diff(s[0], s[2]);
    const double f12 = safe_inv_sq_diff(s[1], s[2]);
    Dm3 Mx;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            double f = 0.0;
            if (i == 0 && j == 1) f = f01;
            if (i == 0 && j == 2) f = f02;
            if (i == 1 && j == 2) f = f12;
            if (i == 1 && j == 0) f = -f01;
            if (i == 2 && j == 0) f = -f02;
            if (i == 2 && j == 1) f = -f12;
            const double omu = UaU(i, j) - UaU(j, i);
            const double omv = VaV(i, j) - VaV(j, i);
            Mx(i, j) = (i == j ? aS[i] : 0.0) + f * omu * s[j] + s[i] * f * omv;
        }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            double acc = gf(i, j);
#pragma unroll
            for (int r = 0; r < 3; ++r)
                acc += U[3 * i + r] * (Mx(r, 0) * V[3 * j] + Mx(r, 1) * V[3 * j + 1] + Mx(r, 2) * V[3 * j + 2]);
            gF[3 * i + j] = (float)acc;
        }
    // dJ/dE_p (per-particle E, chain rule through lame, mpm_cpu_diff.rs:217-222)
    const double nu = sc.poisson;
    const double ge = amu / (2.0 * (1.0 + nu)) + alam * nu / ((1.0 + nu) * (1.0 - 2.0 * nu));
    gE += (float)ge;
}

// Block sum of the particles' (dJ/dmu, dJ/dlambda) added to chunk ci's
// accumulator: one block owns a chunk, so the order is fixed.  Every thread
// of the block calls it.
__device__ __forceinline__ void add_chunk_mu_lambda(double* gml, uint32_t ci, double amu, double alam,
                                                    double (*red)[WAVES]) {
    const int lane = threadIdx.x & 63, wave = wave_id();
    amu = warp_sum(amu);
    alam = warp_sum(alam);
    if (lane == 0) {
        red[0][wave] = amu;
        red[1][wave] = alam;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double sm = 0.0, sl = 0.0;
        for (int w = 0; w < WAVES; ++w) {
            sm += red[0][w];
            sl += red[1][w];
        }
        gml[2 * (size_t)ci] += sm;
        gml[2 * (size_t)ci + 1] += sl;
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_adj_g2p(AdjArgs q) {
    __shared__ ScatterLdsT<true> L;
    __shared__ int red[1][WAVES][6];
    const StepArgs& a = q.a;
    const uint32_t cap = a.cap;
    float* __restrict__ adj = q.adj;
    const uint32_t nch = *a.n_chunks_dev;
    for (ChunkWalk w = chunk_walk(nch); w.ci < w.end; w.ci += w.step) {
        const uint32_t ci = w.ci;
        const Chunk ch = a.chunks[ci];
        const SceneDev sc = a.scenes[ch.scene];
        const uint32_t slot = ch.start + threadIdx.x;
        int b[1][3], lo[1][3], hi[1][3];
        const bool on[1] = {staged_base(a, sc, ch, a.ps, slot, threadIdx.x < ch.count, b[0])};
        block_boxes<1>(on, b, red, lo, hi);
        const Staged st = stage_box(sc, a.gv, lo[0], hi[0], reinterpret_cast<float4*>(&L.acc[0][0]));
        __syncthreads();
        Scatter sp;
        sp.on = false;
        sp.esc = false;
        if (threadIdx.x < ch.count) {
            float gx[3], gv[3], gC[9], gF[9];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                gx[k] = adj[(size_t)(AX + k) * cap + slot];
                gv[k] = adj[(size_t)(AV + k) * cap + slot];
            }
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                gC[k] = adj[(size_t)(AC + k) * cap + slot];
                gF[k] = adj[(size_t)(AF + k) * cap + slot];
            }
            adj_g2p_particle(a, sc, ch, slot, gx, gv, gC, gF, sp, st);
#pragma unroll
            for (int k = 0; k < 3; ++k) adj[(size_t)(AX + k) * cap + slot] = gx[k];
#pragma unroll
            for (int k = 0; k < 9; ++k) adj[(size_t)(AF + k) * cap + slot] = gF[k];
        }
        block_scatter<false, true>(a, sc, sp, ci, L);
    }
}

// ---------------------------------------------------------------------------
// Grid reverse (mpm_adjoint.rs:324-363).  gmp holds the forward's P2G total
// (m, p) of every listed tile; gadj holds the atomic part of dJ/d(grid v)
// and receives (dJ/dm, dJ/dp).
// SPLIT: the block's four waves sum four ranges of each tile's candidate
// chunks and wave 0 adds them in order (small scenes; as k_grid_update).
template <bool SPLIT>
__global__ __launch_bounds__(256) void k_adj_grid(const SceneDev* __restrict__ scenes, GridDev g, float4* gadj,
                                                  const uint32_t* __restrict__ dlist,
                                                  const uint32_t* __restrict__ dcount, float dt, int use_esc) {
    constexpr int R = 4;
    __shared__ float4 wsum[SPLIT ? R - 1 : 1][64];
    const uint32_t ns = *g.scount, nd = *dcount;
    const int lane = threadIdx.x & 63, wave = wave_id();
    const uint32_t first = SPLIT ? blockIdx.x : blockIdx.x * 4 + uint32_t(wave);
    const uint32_t stride = SPLIT ? gridDim.x : gridDim.x * 4;
    for (uint32_t i = first; i < ns + nd; i += stride) {
        TileRec r;
        load_tile_rec(g, ns, i, r);
        const uint32_t t = r.valid ? r.t : (i < ns ? g.slist[i] : dlist[i - ns]);
        const SceneDev sc = scenes[r.valid ? r.scene : g.tile_scene[t]];
        int tx, ty, tz, ix, iy, iz;
        tile_cell(sc, t, lane, tx, ty, tz, ix, iy, iz);
        const uint32_t c = (t << 6) | uint32_t(lane);
        float4 q = use_esc && (!SPLIT || wave == 0) ? gadj[c] : make_float4(0.f, 0.f, 0.f, 0.f);
        add_partials(g, sc, tx, ty, tz, ix, iy, iz, q, SPLIT ? wave : 0, SPLIT ? R : 1, r.valid, r.rng);
        if (SPLIT) {
            if (wave > 0) wsum[wave - 1][lane] = q;
            __syncthreads();
            if (wave == 0) {
#pragma unroll
                for (int r = 0; r < R - 1; ++r) {
                    const float4 v = wsum[r][lane];
                    q.x += v.x;
                    q.y += v.y;
                    q.z += v.z;
                    q.w += v.w;
                }
            }
            __syncthreads();  // wsum is reused by the next tile
            if (wave != 0) continue;
        }
        const float4 mp = g.gmp[c];
        const float m = mp.x;
        float4 out = make_float4(0.f, 0.f, 0.f, 0.f);
        if (m > 0.0f) {
            float gx = q.y, gy = q.z, gz = q.w;
            if (below_floor(sc, iy)) {
                float vy = mp.z / m;  // same operations as the forward's floor test
                vy += sc.gravity_y * dt;
                if (vy < 0.f) gy = 0.f;
                const float damp = 1.0f - sc.floor_friction;
                gx *= damp;
                gz *= damp;
            }
            const float im = 1.0f / m;
            out.y = gx * im;
            out.z = gy * im;
            out.w = gz * im;
            out.x = -(mp.y * gx + mp.z * gy + mp.w * gz) * im * im;
        }
        gadj[c] = out;
    }
}

// ---------------------------------------------------------------------------
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_adj_p2g(AdjArgs q) {
    __shared__ double red[2][WAVES];
    __shared__ float4 cells[LDS_CELLS];
    __shared__ int bred[1][WAVES][6];
    const StepArgs& a = q.a;
    const uint32_t cap = a.cap;
    float* __restrict__ adj = q.adj;
    const uint32_t nch = *a.n_chunks_dev;
    for (ChunkWalk w = chunk_walk(nch); w.ci < w.end; w.ci += w.step) {
        const uint32_t ci = w.ci;
        const Chunk ch = a.chunks[ci];
        const SceneDev sc = a.scenes[ch.scene];
        const uint32_t slot = ch.start + threadIdx.x;
        int b[1][3], lo[1][3], hi[1][3];
        const bool on[1] = {staged_base(a, sc, ch, a.ps, slot, threadIdx.x < ch.count, b[0])};
        block_boxes<1>(on, b, bred, lo, hi);
        const Staged st = stage_box(sc, q.gadj, lo[0], hi[0], cells);
        __syncthreads();
        double amu = 0.0, alam = 0.0;
        if (threadIdx.x < ch.count) {
            float gx[3], gv[3], gC[9], gF[9];
#pragma unroll
            for (int k = 0; k < 3; ++k) gx[k] = adj[(size_t)(AX + k) * cap + slot];
#pragma unroll
            for (int k = 0; k < 9; ++k) gF[k] = adj[(size_t)(AF + k) * cap + slot];
            float gE = adj[(size_t)AE * cap + slot];
            adj_p2g_particle(a, q.gadj, q.aff, sc, slot, gx, gF, gv, gC, gE, amu, alam, st);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                adj[(size_t)(AX + k) * cap + slot] = gx[k];
                adj[(size_t)(AV + k) * cap + slot] = gv[k];
            }
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                adj[(size_t)(AC + k) * cap + slot] = gC[k];
                adj[(size_t)(AF + k) * cap + slot] = gF[k];
            }
            adj[(size_t)AE * cap + slot] = gE;
        }
        add_chunk_mu_lambda(q.gml, ci, amu, alam, red);
    }
}

// Reverse P2G of substep k fused with the reverse G2P of substep k-1 for
// the same particle: dJ/d(state k) stays in registers.  Valid when no
// particle of either substep scatters with global atomics (the host checks
// the recompute's escape and fallback counters), so gadj is only read here.
// The FP64 SVD's registers leave two waves per SIMD, too few to hide 54
// dependent 16-byte gathers from L2 per particle, so both gathers' boxes are
// staged in the scatter's LDS first, with a round of coalesced loads: 128
// scenes of 4 k to 32 k particles 440 us before, 340 now, one of 65,536
// particles 29.7 and 24.3.  What is left is the FP64 arithmetic.
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_adj_fused(AdjArgs q, const float* ps_prev, const float4* gv_prev) {
    __shared__ ScatterLdsT<true> L;
    __shared__ double red[2][WAVES];
    __shared__ int bred[2][WAVES][6];
    static_assert(sizeof(L.acc) >= 2 * LDS_CELLS * sizeof(float4), "two boxes of grid cells before the scatter");
    const StepArgs& a = q.a;
    StepArgs ap = q.a;
    ap.ps = ap.ps_out = const_cast<float*>(ps_prev);
    ap.gv = const_cast<float4*>(gv_prev);
    const uint32_t cap = a.cap;
    float* __restrict__ adj = q.adj;
    const uint32_t nch = *a.n_chunks_dev;
    for (ChunkWalk w = chunk_walk(nch); w.ci < w.end; w.ci += w.step) {
        const uint32_t ci = w.ci;
        const Chunk ch = a.chunks[ci];
        const SceneDev sc = a.scenes[ch.scene];
        const uint32_t slot = ch.start + threadIdx.x;
        const bool active = threadIdx.x < ch.count;
        // both gathers' boxes (dJ/d grid of this substep, grid velocity of the
        // previous one) in the scatter's space, loaded at once
        int b[2][3], lo[2][3], hi[2][3];
        const bool on[2] = {staged_base(a, sc, ch, a.ps, slot, active, b[0]),
                            staged_base(a, sc, ch, ap.ps, slot, active, b[1])};
        block_boxes<2>(on, b, bred, lo, hi);
        float4* cells = reinterpret_cast<float4*>(&L.acc[0][0]);
        const Staged st = stage_box(sc, q.gadj, lo[0], hi[0], cells);
        const Staged stp = stage_box(sc, ap.gv, lo[1], hi[1], cells + LDS_CELLS);
        __syncthreads();
        double amu = 0.0, alam = 0.0;
        float gx[3], gv[3], gC[9], gF[9];
        if (active) {
#pragma unroll
            for (int k = 0; k < 3; ++k) gx[k] = adj[(size_t)(AX + k) * cap + slot];
#pragma unroll
            for (int k = 0; k < 9; ++k) gF[k] = adj[(size_t)(AF + k) * cap + slot];
            float gE = adj[(size_t)AE * cap + slot];
            adj_p2g_particle(a, q.gadj, q.aff, sc, slot, gx, gF, gv, gC, gE, amu, alam, st);
            adj[(size_t)AE * cap + slot] = gE;
        }
        add_chunk_mu_lambda(q.gml, ci, amu, alam, red);
        Scatter sp;
        sp.on = false;
        sp.esc = false;
        if (active) {
            adj_g2p_particle(ap, sc, ch, slot, gx, gv, gC, gF, sp, stp);
#pragma unroll
            for (int k = 0; k < 3; ++k) adj[(size_t)(AX + k) * cap + slot] = gx[k];
#pragma unroll
            for (int k = 0; k < 9; ++k) adj[(size_t)(AF + k) * cap + slot] = gF[k];
        }
        block_scatter<false, true>(ap, sc, sp, ci, L);
    }
}

hipError_t launch_adj_g2p(const AdjArgs& q, int blocks, hipStream_t s) {
    if (blocks <= 0) return hipSuccess;
    if (blocks > int(NUM_XCD)) blocks &= ~int(NUM_XCD - 1);
    hipLaunchKernelGGL(k_adj_g2p, dim3(blocks), dim3(BLOCK), 0, s, q);
    return hipGetLastError();
}

hipError_t launch_adj_grid(const SceneDev* scenes, const GridDev& g, float4* gadj, const uint32_t* dlist,
                           const uint32_t* dcount, float dt, int use_esc, int blocks, hipStream_t s, int split) {
    if (split)
        hipLaunchKernelGGL(k_adj_grid<true>, dim3(blocks), dim3(256), 0, s, scenes, g, gadj, dlist, dcount, dt,
                           use_esc);
    else
        hipLaunchKernelGGL(k_adj_grid<false>, dim3(blocks), dim3(256), 0, s, scenes, g, gadj, dlist, dcount, dt,
                           use_esc);
    return hipGetLastError();
}

hipError_t launch_adj_fused(const AdjArgs& q, const float* ps_prev, const float4* gv_prev, int blocks,
                            hipStream_t s) {
    if (blocks <= 0) return hipSuccess;
    if (blocks > int(NUM_XCD)) blocks &= ~int(NUM_XCD - 1);
    hipLaunchKernelGGL(k_adj_fused, dim3(blocks), dim3(BLOCK), 0, s, q, ps_prev, gv_prev);
    return hipGetLastError();
}

hipError_t launch_adj_p2g(const AdjArgs& q, int blocks, hipStream_t s) {
    if (blocks <= 0) return hipSuccess;
    if (blocks > int(NUM_XCD)) blocks &= ~int(NUM_XCD - 1);
    hipLaunchKernelGGL(k_adj_p2g, dim3(blocks), dim3(BLOCK), 0, s, q);
    return hipGetLastError();
}

}  // namespace mpm
