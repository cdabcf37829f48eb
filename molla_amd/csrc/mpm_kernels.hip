// mpm_kernels.hip -- HIP kernels of the MPM substep for gfx950 (MI355X).
//
// The per-substep hot path is two launches:
//   k_grid_update  over the active-tile list (mpm.wgsl grid_update :1010-1058)
//   k_particles    G2P -> x/v/C/F update -> plasticity -> stress -> P2G, fused
//                  (mpm.wgsl g2p :1241-1353, plasticity :1355-1479,
//                  p2g/p2g_two_pass :494-925) so a particle's state is read
//                  once and written once per substep and the polar/SVD of F is
//                  computed once per substep (FP64).
// The P2G half reduces the block's scatter in LDS (fixed point: 32-bit for the
// shader model, 64-bit for the differentiable model) over
// the bounding box of its particles' stencils -- particles are kept sorted by
// 4^3 tile and cut into chunks that stay inside 4 or 8 tiles of one tile row,
// so that box is small -- and stores the box as the chunk's partial with
// plain stores.  The next grid update sums the partials of the chunks around
// each active tile in ascending chunk order.  Particles that moved beyond the
// 27 tiles around their sorted tile since the last sort scatter with global
// f32 atomics instead.
#include <algorithm>

#include "mpm_blockscan.hpp"
#include "mpm_rigid.hpp"
#include "mpm_scatter.hpp"

namespace mpm {

// Kirchhoff-form stress of a particle from its SVD; returns the affine
// matrix A = m C + 4/dx^2 * (-dt vol U diag(tau) U^T).
template <int MODEL>
__device__ __forceinline__ void affine_from_svd(const SceneDev& sc, const float* mrow, const Svd32& d,
                                                float mu, float lam, float jp, float dt, float vol,
                                                float m, const float* C, float* A) {
    float tau[3];
    if (MODEL == MODEL_SHADER) {
        int rheo = int(mrow[0] + 0.5f);
        float h = 1.0f;
        if (rheo == RHEO_SNOW) h = __expf(clampf(-mrow[4] * jp, -3.0f, 3.0f));
        else if (rheo == RHEO_SAND) h = __expf(clampf(jp, -3.0f, 3.0f));
        float mu_h = mu * h, lam_h = lam * h;
        if (rheo == RHEO_FLUID) {
            mu_h = 0.0f;
            lam_h = mrow[7];
        }
        float s0 = clampf(d.s[0], 0.1f, 10.0f), s1 = clampf(d.s[1], 0.1f, 10.0f),
              s2 = clampf(d.s[2], 0.1f, 10.0f);
        float J = s0 * s1 * s2;
        float vj = lam_h * (J - 1.0f) * J;
        tau[0] = 2.0f * mu_h * (s0 - 1.0f) * s0 + vj;
        tau[1] = 2.0f * mu_h * (s1 - 1.0f) * s1 + vj;
        tau[2] = 2.0f * mu_h * (s2 - 1.0f) * s2 + vj;
    } else {
        float tr = d.s[0] + d.s[1] + d.s[2] - 3.0f;
#pragma unroll
        for (int i = 0; i < 3; ++i) tau[i] = (2.0f * mu * (d.s[i] - 1.0f) + lam * tr) * d.s[i];
    }
    float S[9];
    udut(d.U, tau, S);
    const float k = -dt * vol * 4.0f * sc.inv_dx * sc.inv_dx;
#pragma unroll
    for (int i = 0; i < 9; ++i) A[i] = m * C[i] + k * S[i];
}

// LDS for the scatter inputs of a thread's earlier particles of a chunk.
template <int N>
struct StashSpace {
    ScatterStash s[N - 1];
    __device__ __forceinline__ ScatterStash* ptr() { return s; }
};
template <>
struct StashSpace<1> {
    __device__ __forceinline__ ScatterStash* ptr() { return nullptr; }
};

// Three waves per SIMD (168 VGPRs) with three blocks per CU (LDS_CELLS):
// the pass is latency-bound, and this beats the unconstrained 2 waves/SIMD.
// SPARSE: the grid is a tile pool (one shader-model scene; a.tile_slot set).
// PPT: particles per thread (shader model, sorted chunks of up to 256 PPT
// particles): a thread takes positions t, t + 256, ... of the chunk in turn,
// and one block scatter reduces all of them, so the chunk's box, its partial
// and the grid update's work are shared by PPT times the particles.
template <int MODE, int MODEL, bool SPARSE, int PPT>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(3, 3))) void k_particles(StepArgs a) {
    // The differentiable model scatters in int64: its reverse pass divides by
    // grid masses, so edge cells need each contribution kept to f32 precision.
    constexpr bool WIDE = MODEL == MODEL_CPUDIFF;
    static_assert(PPT == 1 || MODEL == MODEL_SHADER, "several particles per thread: shader model only");
    __shared__ ScatterLdsT<WIDE> L;
    __shared__ StashSpace<MODE == MODE_G2P ? 1 : PPT> Lst;
    if (threadIdx.x == 0) L.box[15] = a.status[ST_FAULT] != 0u ? 1 : 0;
    if (SPARSE && threadIdx.x < 64) L.tmask[threadIdx.x] = 0u;
    // the pool's count for the compaction that follows a scattering pass
    if (SPARSE && MODE != MODE_G2P && blockIdx.x == 0 && threadIdx.x == 0) a.status[ST_POOL] = 0u;
    __syncthreads();
    if (L.box[15]) return;  // block-uniform: a latched fault stops the pass
    if (MODE != MODE_P2G && blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&a.status[ST_GATHERS], 1u);
    const uint32_t cap = a.cap;
    const float* ps = a.ps;
    float* po = a.ps_out;  // the updated x, v, C, F, jp (may alias ps)
    const float dt = a.dt;
    const uint32_t nch = a.n_chunks_dev ? *a.n_chunks_dev : a.n_chunks;
    for (ChunkWalk w = chunk_walk(nch); w.ci < w.end; w.ci += w.step) {
        const uint32_t ci = w.ci;
        const Chunk ch = const_load(a.chunks + ci);
        const SceneDev sc = const_load(a.scenes + ch.scene);
        // Gather staging: the chunk's P2G box of the previous pass holds every
        // stencil this gather reads (same particles, same positions), so the
        // block loads that box of grid velocities into LDS once and the 27
        // node reads of each particle come from LDS.  Particles outside the
        // box (escaped ones) read global memory.
        int4 gbox = make_int4(0, 0, 0, 0), gdim = make_int4(0, 0, 0, 0);
        const bool staged = MODE != MODE_P2G && stage_gather_box<WIDE, SPARSE>(a, sc, ci, L, gbox, gdim);
        WaveBounds pre;  // the wave's box and bounds over its earlier particles
        Scatter sp;
#pragma unroll 1
        for (int pq = 0; pq < PPT; ++pq) {
        const uint32_t slot = ch.start + threadIdx.x + uint32_t(pq) * BLOCK;
        const uint32_t boff = 4u * slot;
        const bool active = threadIdx.x + uint32_t(pq) * BLOCK < ch.count;
        float xs[3] = {0.f, 0.f, 0.f};  // the scattered position
        // every field written here, so nothing of the previous particle stays live
        sp.on = false;
        sp.esc = false;
        sp.slot = slot;
        sp.m = 0.f;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            sp.b[k] = 0;
            sp.fx[k] = 0.f;
            sp.mv[k] = 0.f;
        }
#pragma unroll
        for (int k = 0; k < 9; ++k) sp.A[k] = 0.f;
        if (active) {
            float x[3], F[9];
#pragma unroll
            for (int k = 0; k < 3; ++k) x[k] = plane_ld(ps, cap, CX + k, boff);
#pragma unroll
            for (int k = 0; k < 9; ++k) F[k] = plane_ld(ps, cap, CF + k, boff);
            float jp = plane_ld(ps, cap, CJP, boff);
            const float m = plane_ld(ps, cap, CMASS, boff);
            const float vol = plane_ld(ps, cap, CVOL, boff);
            const uint32_t matid = __float_as_uint(plane_ld(ps, cap, CMAT, boff));
            const float* mrow = mat_row(a, sc, matid);
            float mu = sc.mu, lam = sc.lam;
            if (a.has_E) {
                float E = plane_ld(ps, cap, CE, boff);
                mu = E / (2.0f * (1.0f + sc.poisson));
                lam = E * sc.poisson / ((1.0f + sc.poisson) * (1.0f - 2.0f * sc.poisson));
            }
            bool ok = true;
            float v[3], C[9];
            // the slot's sorted tile key, for the scatter's escape test; read
            // before this particle's state stores, which the compiler cannot
            // move it past
            uint32_t skey = 0u;
            if (MODE == MODE_P2G) {
                if (a.use_lds) skey = a.sorted_keys[slot];
#pragma unroll
                for (int k = 0; k < 3; ++k) v[k] = plane_ld(ps, cap, CV + k, boff);
#pragma unroll
                for (int k = 0; k < 9; ++k) C[k] = plane_ld(ps, cap, CC + k, boff);
                if (MODEL == MODEL_SHADER) {
                    float fa = finite_acc(0.0f, jp);
#pragma unroll
                    for (int k = 0; k < 3; ++k) fa = finite_acc(finite_acc(fa, x[k]), v[k]);
#pragma unroll
                    for (int k = 0; k < 9; ++k) fa = finite_acc(finite_acc(fa, C[k]), F[k]);
                    if (!finite_acc_ok(fa)) {
                        latch(a.status, FAULT_NUMERICAL);
                        ok = false;
                    }
                }
                if (ok) {
                    Svd32 d;
                    svd3<MODEL>(F, d);
                    affine_from_svd<MODEL>(sc, mrow, d, mu, lam, jp, dt, vol, m, C, sp.A);
                    if (a.aff_out)
#pragma unroll
                        for (int k = 0; k < 9; ++k) plane_st(a.aff_out, cap, k, boff, sp.A[k]);
                }
            } else {
                // ---- G2P (mpm.wgsl:1241-1353 / mpm_cpu_diff.rs:544-580) ----
                float xp[3], fx[3], w[3][3];
                int b[3];
                float fa = finite_acc(0.0f, jp);
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    xp[k] = (x[k] - sc.origin[k]) * sc.inv_dx;
                    fa = finite_acc(finite_acc(fa, x[k]), xp[k]);
                }
#pragma unroll
                for (int k = 0; k < 9; ++k) fa = finite_acc(fa, F[k]);
                if (MODEL == MODEL_SHADER && !finite_acc_ok(fa)) {
                    latch(a.status, FAULT_NUMERICAL);
                    ok = false;
                }
                if (ok) {
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        float bf = floorf(xp[k] - 0.5f);
                        b[k] = int(bf) - (MODEL == MODEL_SHADER ? sc.window[k] : 0);
                        fx[k] = xp[k] - bf;
                        quad_weights(fx[k], w[k]);
                    }
                    // v = sum w v_i and, with d = ((i, j, k) - fx) dx,
                    // C = 4/dx^2 sum w v_i d^T = 4/dx (M - v fx^T),
                    // M = sum w v_i (i, j, k)^T, accumulated per x-row.
                    float vn[3] = {0.f, 0.f, 0.f};
                    float M[9];
#pragma unroll
                    for (int k = 0; k < 9; ++k) M[k] = 0.f;
                    // fetch(i, j, k, g): node (b + (i, j, k)), false when outside the grid
                    // Row sums over i weighted by w0 (and by i w0), then one
                    // multiply by w1 w2 per row: 3-6 FMAs per node.
                    const float wi1 = w[0][1], wi2 = 2.0f * w[0][2];
                    auto gather = [&](auto fetch) {
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
#pragma unroll
                            for (int j = 0; j < 3; ++j) {
                                const float wjk = w[1][j] * w[2][k];
                                float rs[3] = {0.f, 0.f, 0.f}, ri[3] = {0.f, 0.f, 0.f};
#pragma unroll
                                for (int i = 0; i < 3; ++i) {
                                    float4 g;
                                    if (!fetch(i, j, k, g)) continue;
                                    rs[0] += w[0][i] * g.x;
                                    rs[1] += w[0][i] * g.y;
                                    rs[2] += w[0][i] * g.z;
                                    if (i > 0) {
                                        const float wi = i == 1 ? wi1 : wi2;
                                        ri[0] += wi * g.x;
                                        ri[1] += wi * g.y;
                                        ri[2] += wi * g.z;
                                    }
                                }
                                // j and k are unrolled constants: rows with j = 0 or
                                // k = 0 add nothing to those moments
                                const float wj = float(j) * wjk, wk = float(k) * wjk;
#pragma unroll
                                for (int r = 0; r < 3; ++r) {
                                    vn[r] += wjk * rs[r];
                                    M[3 * r] += wjk * ri[r];
                                    if (j > 0) M[3 * r + 1] += wj * rs[r];
                                    if (k > 0) M[3 * r + 2] += wk * rs[r];
                                }
                            }
                        }
                    };
                    const bool in_box = staged && b[0] >= gbox.x && b[1] >= gbox.y && b[2] >= gbox.z &&
                                        b[0] + 2 < gbox.x + gdim.x && b[1] + 2 < gbox.y + gdim.y &&
                                        b[2] + 2 < gbox.z + gdim.z;
                    if (in_box) {
                        const float4* stage = reinterpret_cast<const float4*>(&L.acc[0][0]);
                        const int li0 = (b[0] - gbox.x) + gdim.x * ((b[1] - gbox.y) + gdim.y * (b[2] - gbox.z));
                        gather([&](int i, int j, int k, float4& g) {
                            g = stage[li0 + i + gdim.x * (j + gdim.y * k)];
                            return true;
                        });
                    } else {
                        const int G = int(sc.G);
                        gather([&](int i, int j, int k, float4& g) {
                            const int ix = b[0] + i, iy = b[1] + j, iz = b[2] + k;
                            if (ix < 0 || ix >= G || iy < 0 || iy >= G || iz < 0 || iz >= G) return false;
                            uint32_t c;
                            if (!cell_storage(sc, SPARSE ? a.tile_slot : nullptr, ix, iy, iz, c)) return false;
                            g = a.gv[c];
                            return true;
                        });
                    }
                    const float dx = sc.dx, s4dx = 4.0f * sc.inv_dx;
                    float Cn[9];
#pragma unroll
                    for (int r = 0; r < 3; ++r)
#pragma unroll
                        for (int c = 0; c < 3; ++c) Cn[3 * r + c] = s4dx * (M[3 * r + c] - vn[r] * fx[c]);
                    const int rheo = int(mrow[0] + 0.5f);
                    if (MODEL == MODEL_SHADER && rheo == RHEO_VISCOUS) {
                        float vd = __expf(-fmaxf(mrow[5], 0.0f) * dt);
                        float ad = __expf(-fmaxf(mrow[6], 0.0f) * dt);
#pragma unroll
                        for (int k = 0; k < 3; ++k) vn[k] *= vd;
#pragma unroll
                        for (int k = 0; k < 9; ++k) Cn[k] *= ad;
                    }
                    float nx[3];
                    float fa2 = 0.0f;
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        nx[k] = x[k] + dt * vn[k];
                        fa2 = finite_acc(finite_acc(fa2, nx[k]), vn[k]);
                    }
#pragma unroll
                    for (int k = 0; k < 9; ++k) fa2 = finite_acc(fa2, Cn[k]);
                    if (!finite_acc_ok(fa2)) {
                        latch(a.status, FAULT_NUMERICAL);
                        ok = false;
                    }
                    if (ok && MODEL == MODEL_SHADER) {
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            float lo = sc.origin[k] + float(sc.window[k] + 2) * dx;
                            float hi = sc.origin[k] + float(sc.window[k] + int(sc.G) - 3) * dx;
                            if (nx[k] < lo || nx[k] > hi) vn[k] = 0.0f;
                            nx[k] = fminf(fmaxf(nx[k], lo), hi);
                        }
                    }
                    float Fn[9];
                    if (ok) {
#pragma unroll
                        for (int i = 0; i < 3; ++i)
#pragma unroll
                            for (int j = 0; j < 3; ++j)
                                Fn[3 * i + j] = F[3 * i + j] + dt * (Cn[3 * i] * F[j] + Cn[3 * i + 1] * F[3 + j] +
                                                                     Cn[3 * i + 2] * F[6 + j]);
                        float fa3 = 0.0f;
#pragma unroll
                        for (int k = 0; k < 9; ++k) fa3 = finite_acc(fa3, Fn[k]);
                        if (!finite_acc_ok(fa3)) ok = false;
                        if (!ok) latch(a.status, FAULT_NUMERICAL);
                    }
                    if (ok) {
                        // ---- plasticity (mpm.wgsl:1355-1479) + stress from the same SVD ----
                        Svd32 d;
                        bool have_svd = false;
                        bool plast_ok = true;
                        float jp_new = jp;
                        if (MODEL == MODEL_SHADER) {
                            if (rheo == RHEO_FLUID) {
                                float J = Fn[0] * (Fn[4] * Fn[8] - Fn[5] * Fn[7]) -
                                          Fn[1] * (Fn[3] * Fn[8] - Fn[5] * Fn[6]) +
                                          Fn[2] * (Fn[3] * Fn[7] - Fn[4] * Fn[6]);
                                float s = clampf(cbrtf(J), 0.05f, 20.0f);
                                if (!finitef(s)) {
                                    plast_ok = false;
                                } else {
#pragma unroll
                                    for (int k = 0; k < 9; ++k) Fn[k] = (k % 4 == 0) ? s : 0.0f;
                                    jp_new = 0.0f;
                                    d.s[0] = d.s[1] = d.s[2] = s;
#pragma unroll
                                    for (int k = 0; k < 9; ++k) d.U[k] = d.V[k] = (k % 4 == 0) ? 1.0f : 0.0f;
                                    have_svd = true;
                                }
                            } else {
                                svd3<MODEL_SHADER>(Fn, d);
                                float ns[3] = {d.s[0], d.s[1], d.s[2]};
                                float dq = 0.0f;
                                bool jp_replace = false;
                                bool fin3 = finitef(ns[0]) && finitef(ns[1]) && finitef(ns[2]);
                                if (!fin3) plast_ok = false;
                                if (plast_ok && rheo == RHEO_SNOW) {
                                    const float tc = mrow[2], tsv = mrow[3];
#pragma unroll
                                    for (int k = 0; k < 3; ++k) ns[k] = clampf(d.s[k], 1.0f - tc, 1.0f + tsv);
                                    float det_old = fmaxf(d.s[0] * d.s[1] * d.s[2], 1.0e-6f);
                                    float det_new = fmaxf(ns[0] * ns[1] * ns[2], 1.0e-6f);
                                    jp_replace = true;
                                    jp_new = jp + (__logf(det_old) - __logf(det_new));
                                    if (!finitef(jp_new)) plast_ok = false;
                                    jp_new = clampf(jp_new, -5.0f, 5.0f);
                                } else if (plast_ok && rheo == RHEO_VISCOUS) {
                                    jp_replace = true;
                                    jp_new = 0.0f;
                                } else if (plast_ok) {
                                    // sand (Drucker-Prager), mpm.wgsl:1421-1457
                                    const float e0 = __logf(fmaxf(d.s[0], 1.0e-6f)),
                                                e1 = __logf(fmaxf(d.s[1], 1.0e-6f)),
                                                e2 = __logf(fmaxf(d.s[2], 1.0e-6f));
                                    float tre = e0 + e1 + e2, mean = tre / 3.0f;
                                    float d0 = e0 - mean, d1 = e1 - mean, d2 = e2 - mean;
                                    float dn = sqrtf(d0 * d0 + d1 * d1 + d2 * d2);
                                    float kappa = (3.0f * lam + 2.0f * mu) / (2.0f * mu);
                                    if (tre > 0.0f) {
                                        ns[0] = ns[1] = ns[2] = 1.0f;
                                        dq = sqrtf(e0 * e0 + e1 * e1 + e2 * e2);
                                    } else if (dn != 0.0f) {
                                        float fy = dn + kappa * tre * mrow[1];
                                        if (fy > 0.0f) {
                                            float rc = fmaxf(0.0f, -mrow[1] * kappa * tre);
                                            float sc2 = rc / dn;
                                            ns[0] = __expf(d0 * sc2 + mean);
                                            ns[1] = __expf(d1 * sc2 + mean);
                                            ns[2] = __expf(d2 * sc2 + mean);
                                            dq = fy;
                                        }
                                    }
                                }
                                if (plast_ok && (!finitef(ns[0]) || !finitef(ns[1]) || !finitef(ns[2]) ||
                                                 !finitef(dq) || !finitef(jp + dq)))
                                    plast_ok = false;
                                if (plast_ok) {
                                    float ss[3];
                                    bool same = true;
#pragma unroll
                                    for (int k = 0; k < 3; ++k) {
                                        ss[k] = clampf(ns[k], 0.05f, 20.0f);
                                        same = same && (ss[k] == d.s[k]);
                                    }
                                    if (!same) {
                                        udvt(d.U, ss, d.V, Fn);
                                        d.s[0] = ss[0];
                                        d.s[1] = ss[1];
                                        d.s[2] = ss[2];
                                    }
                                    jp_new = jp_replace ? jp_new : clampf(jp + dq, 0.0f, 5.0f);
                                    have_svd = true;
                                }
                            }
                            if (!plast_ok) latch(a.status, FAULT_NUMERICAL);
                        }
                        if (MODE != MODE_G2P && a.use_lds) skey = a.sorted_keys[slot];
                        // ---- write the particle state ----
#pragma unroll
                        for (int k = 0; k < 3; ++k) plane_st(po, cap, CX + k, boff, nx[k]);
                        if (a.write_vc || MODE == MODE_G2P) {
#pragma unroll
                            for (int k = 0; k < 3; ++k) plane_st(po, cap, CV + k, boff, vn[k]);
#pragma unroll
                            for (int k = 0; k < 9; ++k) plane_st(po, cap, CC + k, boff, Cn[k]);
                        }
#pragma unroll
                        for (int k = 0; k < 9; ++k) plane_st(po, cap, CF + k, boff, Fn[k]);
                        if (MODEL == MODEL_SHADER && plast_ok) plane_st(po, cap, CJP, boff, jp_new);
                        if (MODE == MODE_G2P2G && plast_ok) {
                            if (MODEL == MODEL_CPUDIFF) svd3<MODEL_CPUDIFF>(Fn, d);
                            (void)have_svd;
                            affine_from_svd<MODEL>(sc, mrow, d, mu, lam, jp_new, dt, vol, m, Cn, sp.A);
                            if (a.aff_out)
#pragma unroll
                                for (int k = 0; k < 9; ++k) plane_st(a.aff_out, cap, k, boff, sp.A[k]);
#pragma unroll
                            for (int k = 0; k < 3; ++k) {
                                x[k] = nx[k];
                                v[k] = vn[k];
                            }
                        } else {
                            ok = false;
                        }
                    }
                }
            }
            if (ok && MODE != MODE_G2P) {
                stencil_of<MODEL>(sc, x, sp.b, sp.fx);
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    sp.mv[k] = m * v[k];
                    xs[k] = x[k];
                }
                sp.m = m;
                sp.on = true;
                sp.esc = !a.use_lds;
                if (a.use_lds && stencil_escapes(sc, ch, skey, sp.b)) sp.esc = true;
            }
        }
        // the earlier particles wait in LDS; the last one scatters them all
        if (MODE != MODE_G2P && PPT > 1 && pq < PPT - 1) {
            Lst.ptr()[pq].put(sp, xs);
            wave_bounds_add(sp, sc.dx, pre);
        }
        }
        if (MODE != MODE_G2P) block_scatter<true, WIDE, SPARSE, PPT>(a, sc, sp, ci, L, Lst.ptr(), &pre);
        else if (staged) __syncthreads();  // the next chunk's staging overwrites the box
    }
}

hipError_t launch_particle_pass(int mode, int model, const StepArgs& a, int ppt, int blocks,
                                hipStream_t s) {
    if (ppt < 1 || ppt > MAX_PPT || (ppt > 1 && model != MODEL_SHADER)) return hipErrorInvalidValue;
    if (a.n_chunks == 0) return hipSuccess;
    if (blocks <= 0 || uint32_t(blocks) > a.n_chunks) blocks = int(a.n_chunks);
    if (blocks > int(NUM_XCD)) blocks &= ~int(NUM_XCD - 1);  // XCD-aware chunk walk
    blocks = std::max(blocks, 1);
    dim3 g(blocks), b(BLOCK);
#define MPM_LAUNCH(M, D, S) hipLaunchKernelGGL((k_particles<M, D, S, 1>), g, b, 0, s, a)
#define MPM_LAUNCH2(M, S) hipLaunchKernelGGL((k_particles<M, MODEL_SHADER, S, 2>), g, b, 0, s, a)
    if (ppt == 2) {
        if (mode == MODE_P2G) {
            if (a.tile_slot) MPM_LAUNCH2(MODE_P2G, true);
            else MPM_LAUNCH2(MODE_P2G, false);
        } else if (mode == MODE_G2P) {
            if (a.tile_slot) MPM_LAUNCH2(MODE_G2P, true);
            else MPM_LAUNCH2(MODE_G2P, false);
        } else {
            if (a.tile_slot) MPM_LAUNCH2(MODE_G2P2G, true);
            else MPM_LAUNCH2(MODE_G2P2G, false);
        }
    } else if (model == MODEL_SHADER && a.tile_slot) {
        if (mode == MODE_P2G) MPM_LAUNCH(MODE_P2G, MODEL_SHADER, true);
        else if (mode == MODE_G2P) MPM_LAUNCH(MODE_G2P, MODEL_SHADER, true);
        else MPM_LAUNCH(MODE_G2P2G, MODEL_SHADER, true);
    } else if (model == MODEL_SHADER) {
        if (mode == MODE_P2G) MPM_LAUNCH(MODE_P2G, MODEL_SHADER, false);
        else if (mode == MODE_G2P) MPM_LAUNCH(MODE_G2P, MODEL_SHADER, false);
        else MPM_LAUNCH(MODE_G2P2G, MODEL_SHADER, false);
    } else {
        if (a.tile_slot) return hipErrorInvalidValue;  // pools hold shader-model scenes
        if (mode == MODE_P2G) MPM_LAUNCH(MODE_P2G, MODEL_CPUDIFF, false);
        else if (mode == MODE_G2P) MPM_LAUNCH(MODE_G2P, MODEL_CPUDIFF, false);
        else MPM_LAUNCH(MODE_G2P2G, MODEL_CPUDIFF, false);
    }
#undef MPM_LAUNCH
#undef MPM_LAUNCH2
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Grid update over the active tiles (mpm.wgsl:1010-1058; CPUDIFF model:
// mpm_cpu_diff.rs:513-542), fused with the reduction of the P2G partials:
// one wave per tile, one lane per cell.  The tiles are the static list of the
// last sort followed by the dynamic list of tiles reached by global atomics.
// The chunks that may hold partials for tile T are those of the particles
// sorted into T's 3x3x3 neighbourhood: nine x-rows of consecutive tile keys,
// i.e. nine ascending slot ranges read from the tile lower-bound table.
__device__ __forceinline__ void cell_update(const SceneDev& sc, float4 q, int ix, int iy, int iz, float dt,
                                            float4& out) {
    const float m = q.x;
    out = make_float4(0.f, 0.f, 0.f, m);
    const int n_ = int(sc.G);
    if (sc.model == MODEL_SHADER) {
        if (m > 1.0e-9f && m == m) {
            float vx = q.y / m, vy = q.z / m, vz = q.w / m;
            vy = vy + dt * sc.gravity_y;
            const float bf = sc.boundary_friction;
            const int pad = 2;
            if (ix < pad) { vx = fmaxf(vx, 0.f); vy *= bf; vz *= bf; }
            if (ix >= n_ - pad) { vx = fminf(vx, 0.f); vy *= bf; vz *= bf; }
            if (iy < pad) { vy = fmaxf(vy, 0.f); vx *= bf; vz *= bf; }
            if (iy >= n_ - pad) { vy = fminf(vy, 0.f); vx *= bf; vz *= bf; }
            if (iz < pad) { vz = fmaxf(vz, 0.f); vx *= bf; vy *= bf; }
            if (iz >= n_ - pad) { vz = fminf(vz, 0.f); vx *= bf; vy *= bf; }
            out = make_float4(vx, vy, vz, m);
        }
    } else {
        if (m > 0.0f) {
            float vx = q.y / m, vy = q.z / m, vz = q.w / m;
            vy += sc.gravity_y * dt;
            if (below_floor(sc, iy)) {
                if (vy < 0.f) vy = 0.f;
                const float damp = 1.0f - sc.floor_friction;
                vx *= damp;
                vz *= damp;
            }
            out = make_float4(vx, vy, vz, m);
        }
    }
}

// RIGID: bodies are present (the imprint code stays out of the plain kernel).
// SPLIT = false: one wave per tile sums its candidate chunks' partials in
// ascending order (scenes with many more active tiles than blocks).
// SPLIT = true: the block's four waves sum four ranges of the candidate list
// and wave 0 adds the range sums in order, so the latency of the ordered
// partial loads is shared four ways (small scenes: a few hundred tiles, each
// overlapped by tens of chunks).  The host picks the shape from the particle
// count and the launch size only, so a run repeats bitwise; the two shapes
// agree to f32 rounding.
constexpr int GRID_RANGES = 4;
// One wave per tile runs at eight waves per SIMD with four partial loads in
// flight (51 VGPRs, the tile's record and scene in scalar registers): with
// ten thousand tiles or more, more tiles in flight beat deeper load batches.
// The split shape keeps eight loads in flight (dense small scenes have ~100
// overlapping chunks per tile).
template <bool RIGID, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RIGID ? 4 : (SPLIT ? 5 : 8)))) void k_grid_update(
    const SceneDev* __restrict__ scenes, GridDev g,
                                                     const uint32_t* __restrict__ dlist,
                                                     const uint32_t* __restrict__ dcount,
                                                     uint32_t* __restrict__ next_count, float dt,
                                                     int zero_after, int use_partials, float4* keep, RigidDev rg) {
    __shared__ float4 wsum[SPLIT ? GRID_RANGES - 1 : 1][64];
    const TileWalk walk(g, dcount);
    const int lane = threadIdx.x & 63, wave = wave_id();
    const uint32_t first = SPLIT ? blockIdx.x : blockIdx.x * 4 + uint32_t(wave);
    const uint32_t stride = SPLIT ? gridDim.x : gridDim.x * 4;
    // A static tile's record holds its id, scene and candidate ranges; the
    // next tile's record is requested before this tile's stores (which the
    // compiler cannot move it past), so a wave that takes several tiles
    // finds it loaded.
    TileRec cur, nxt;
    if (first < walk.n) load_tile_rec(g, walk.ns, first, cur);
    for (uint32_t i = first; i < walk.n; i += stride) {
        nxt.valid = false;
        if (i + stride < walk.n) load_tile_rec(g, walk.ns, i + stride, nxt);
        uint32_t t, st, scene;
        if (cur.valid) {
            t = cur.t;
            st = t;
            scene = cur.scene;
        } else {
            walk.at(g, dlist, i, t, st);
            scene = g.tile_scene[t];
        }
        const SceneDev sc = const_load(scenes + scene);
        int tx, ty, tz, ix, iy, iz;
        tile_cell(sc, t, lane, tx, ty, tz, ix, iy, iz);
        const uint32_t c = (st << 6) | uint32_t(lane);
        const uint32_t flag = g.tile_flag[t];
        // range 0 starts from the atomic channel
        float4 q = (flag & FLAG_GMP) && (!SPLIT || wave == 0) ? g.gmp[c] : make_float4(0.f, 0.f, 0.f, 0.f);
        if (use_partials) {
            add_partials<(SPLIT || RIGID) ? 8 : 4>(g, sc, tx, ty, tz, ix, iy, iz, q, SPLIT ? wave : 0,
                                                   SPLIT ? GRID_RANGES : 1, cur.valid, cur.rng);
            if (SPLIT) {
                if (wave > 0) wsum[wave - 1][lane] = q;
                __syncthreads();
                if (wave == 0) {
#pragma unroll
                    for (int r = 0; r < GRID_RANGES - 1; ++r) {
                        const float4 v = wsum[r][lane];
                        q.x += v.x;
                        q.y += v.y;
                        q.z += v.z;
                        q.w += v.w;
                    }
                }
            }
        }
        if (!SPLIT || wave == 0) {
            float4 out;
            int owner = -1;
            if (RIGID && rg.count) {
                // rigid_imprint (mpm.wgsl:937-1006) between the P2G and the update:
                // a stamped cell keeps the body's velocity (grid_update :1034-1038)
                float3 force, torque;
                owner = in_grid(sc, ix, iy, iz) ? rigid_imprint(rg, sc, ix, iy, iz, dt, q, force, torque) : -1;
                if (rg.wrench) rigid_wrench_add(rg, owner, force, torque);
            }
            if (owner >= 0) {
                out = make_float4(q.y / q.x, q.z / q.x, q.w / q.x, q.x);
            } else {
                cell_update(sc, q, ix, iy, iz, dt, out);
            }
            g.gv[c] = out;
            if (keep) keep[c] = q;  // the P2G total, for the reverse pass
            if (zero_after) {
                if (flag & FLAG_GMP) g.gmp[c] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (lane == 0) g.tile_flag[t] = flag & (zero_after == 1 ? FLAG_STATIC : FLAG_STATIC | FLAG_DYN);
            } else {
                g.gmp[c] = q;  // the last P2G stays readable (read_grid_mass_momentum)
                if (lane == 0) g.tile_flag[t] = flag | FLAG_GMP;
            }
        }
        if (SPLIT && use_partials) __syncthreads();  // wsum is reused by the next tile
        cur = nxt;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (next_count) *next_count = 0u;
        if (g.defer_count) *g.defer_count = 0u;  // the deferred scatters are done
    }
}

hipError_t launch_grid_update(const SceneDev* scenes, const GridDev& g, const uint32_t* dlist,
                              const uint32_t* dcount, uint32_t* next_count, float dt,
                              int zero_after, int use_partials, int blocks, hipStream_t s, float4* keep,
                              const RigidDev* rigid, int split) {
    const RigidDev rg = rigid ? *rigid : RigidDev{nullptr, nullptr, 0u, 0u};
#define MPM_GRID(R, S)                                                                                          \
    hipLaunchKernelGGL((k_grid_update<R, S>), dim3(blocks), dim3(256), 0, s, scenes, g, dlist, dcount, next_count, \
                       dt, zero_after, use_partials, keep, rg)
    if (rg.count) {
        if (split) MPM_GRID(true, true);
        else MPM_GRID(true, false);
    } else {
        if (split) MPM_GRID(false, true);
        else MPM_GRID(false, false);
    }
#undef MPM_GRID
    return hipGetLastError();
}

// Shell force of legacy rigid spheres (mpm_rigid_force_integrate,
// mpm.wgsl:1174-1226) after the grid update and the implicit sweeps: every
// unstamped cell with sand mass within one cell of a sphere's surface (full
// weight inside, tapering to zero one cell out) pushes on the sphere with
// -(m w / dt) (v_sphere - v_cell).  One wave per active tile.
__global__ __launch_bounds__(256) void k_rigid_shell(const SceneDev* __restrict__ scenes, GridDev g,
                                                     const uint32_t* __restrict__ dlist,
                                                     const uint32_t* __restrict__ dcount, float dt, RigidDev rg) {
    const TileWalk walk(g, dcount);
    const int lane = threadIdx.x & 63;
    for (uint32_t i = blockIdx.x * 4 + uint32_t(wave_id()); i < walk.n; i += gridDim.x * 4) {
        uint32_t t, st;
        walk.at(g, dlist, i, t, st);
        const SceneDev sc = scenes[g.tile_scene[t]];
        int tx, ty, tz, ix, iy, iz;
        tile_cell(sc, t, lane, tx, ty, tz, ix, iy, iz);
        const float4 cv = g.gv[(st << 6) | uint32_t(lane)];
        const bool live = in_grid(sc, ix, iy, iz) && cv.w > 1.0e-9f && cv.w == cv.w &&
                          !rigid_masked_legacy(rg, sc, ix, iy, iz);
        const float3 node = node_position(sc, ix, iy, iz);
        for (uint32_t r = 0; r < rg.count; ++r) {
            const float4* b = rg.body + RIGID_ROWS * r;
            const float3 arm = make_float3(node.x - b[0].x, node.y - b[0].y, node.z - b[0].z);
            const float d = sqrtf(arm.x * arm.x + arm.y * arm.y + arm.z * arm.z);
            const bool near = live && b[4].w == 0.0f && !(d > b[0].w + sc.dx);
            float3 force = make_float3(0.f, 0.f, 0.f), torque = force;
            if (near) {
                float w = 1.0f;
                if (d > b[0].w) w = fmaxf(0.0f, 1.0f - (d - b[0].w) / sc.dx);
                const float k = -(cv.w * w / fmaxf(dt, 1.0e-6f));
                force = make_float3(k * (b[1].x - cv.x), k * (b[1].y - cv.y), k * (b[1].z - cv.z));
                torque = cross3(arm, force);
            }
            if (__ballot(near)) rigid_wrench_add(rg, near ? int(r) : -1, force, torque);
        }
    }
}

hipError_t launch_rigid_shell(const SceneDev* scenes, const GridDev& g, const uint32_t* dlist,
                              const uint32_t* dcount, float dt, const RigidDev& rg, int blocks, hipStream_t s) {
    hipLaunchKernelGGL(k_rigid_shell, dim3(blocks), dim3(256), 0, s, scenes, g, dlist, dcount, dt, rg);
    return hipGetLastError();
}

__global__ void k_zero_f64(double* p, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0.0;
}

hipError_t launch_zero_f64(double* p, uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_zero_f64, dim3(1), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Semi-implicit Jacobi sweeps (mpm_implicit_apply, mpm.wgsl:1060-1153) over the
// active tiles:
//   v' = (m v + a v_avg) / (m + a),  a = dt^2 m (E / 1500) / dx^2,
// v_avg = mean velocity of the face neighbours with m > 1e-9 (v if none);
// empty cells are copied.  A neighbour in a tile that is not on this
// substep's lists (neither FLAG_STATIC nor FLAG_DYN) holds no P2G mass, as
// in the reference's sparse grid, whatever its stale contents.
// K sweeps per launch, one block per tile: the block loads the tile and K
// cells around it into LDS and sweeps a region that shrinks by one cell per
// sweep, so the K sweeps of a tile need nothing of its neighbours' blocks.
// The halo is computed again by every block that needs it (K = 3: 792 cell
// updates for 192), which costs less than the launches it saves up to some
// 3,000 tiles: 32,768 sand particles, three sweeps 9.7 us in a trace against
// 19.5 us as one launch each and 3.9 us for the copy that made an odd count
// end in gv.  A frame of 8 substeps with three against one sweep per launch:
// 8,000 particles 273 / 361 us, 100,000 376 / 409.
// `tickets` (not null in the launch that ends the substep's sweeps): where the
// dynamic list holds tiles, the last block to finish takes FLAG_DYN off them,
// which every block has read by then.
// A cell of mass m > 1e-9 and the sum of its cnt neighbours' velocities.
__device__ __forceinline__ float4 implicit_cell(const SceneDev& sc, const float4& me, float ax, float ay, float az,
                                                float cnt, float dt) {
    const float m = me.w;
    if (cnt > 0.f) {
        ax = ax / cnt;
        ay = ay / cnt;
        az = az / cnt;
    } else {
        ax = me.x;
        ay = me.y;
        az = me.z;
    }
    const float alpha = dt * dt * m * (sc.youngs / 1500.0f) * sc.inv_dx * sc.inv_dx;
    const float den = m + alpha;
    const float vx = (m * me.x + alpha * ax) / den, vy = (m * me.y + alpha * ay) / den,
                vz = (m * me.z + alpha * az) / den;
    return vx == vx && vy == vy && vz == vz ? make_float4(vx, vy, vz, m) : me;
}

template <int K>
__global__ __launch_bounds__(256) void k_implicit_sweeps(const SceneDev* __restrict__ scenes, GridDev g,
                                                         const float4* __restrict__ src, float4* __restrict__ dst,
                                                         const uint32_t* __restrict__ dlist,
                                                         const uint32_t* __restrict__ dcount, float dt, RigidDev rg,
                                                         uint32_t* tickets) {
    constexpr int R = 4 + 2 * K, CELLS = R * R * R, PER = (CELLS + 255) / 256;
    // velocity and mass; the mass is 0 where the cell is no neighbour (empty,
    // outside the grid, off the lists), negated where it keeps its velocity
    __shared__ float4 buf[2][CELLS];
    __shared__ uint32_t s_last;
    const TileWalk walk(g, dcount);
    const int tid = threadIdx.x;
    for (uint32_t i = blockIdx.x; i < walk.n; i += gridDim.x) {
        uint32_t t, st;
        walk.at(g, dlist, i, t, st);
        const SceneDev sc = scenes[g.tile_scene[t]];
        int tx, ty, tz, ix0, iy0, iz0;
        tile_cell(sc, t, 0, tx, ty, tz, ix0, iy0, iz0);
        const int lo[3] = {ix0 - K, iy0 - K, iz0 - K}, hi[3] = {ix0 + 3 + K, iy0 + 3 + K, iz0 + 3 + K};
        const uint64_t near = rigid_near_legacy(rg, sc, lo, hi);
        float4 v[PER];
        bool on[PER];
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int c = tid + 256 * u;
            const int lx = c % R, ly = (c / R) % R, lz = c / (R * R);
            const int ix = ix0 + lx - K, iy = iy0 + ly - K, iz = iz0 + lz - K;
            v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            on[u] = c < CELLS && in_grid(sc, ix, iy, iz);
            if (on[u]) {
                uint32_t nc;
                if (g.tile_slot) {
                    on[u] = cell_storage(sc, g.tile_slot, ix, iy, iz, nc);  // no slot: no P2G mass
                } else {
                    nc = cell_index(sc, ix, iy, iz);
                    on[u] = (g.tile_flag[nc >> 6] & (FLAG_STATIC | FLAG_DYN)) != 0u;
                }
                if (!g.tile_slot || on[u]) v[u] = src[nc];
                // empty cells and negative masses are no neighbours; cells
                // stamped by a legacy sphere keep their velocity
                if (!(v[u].w > 1.0e-9f)) v[u].w = 0.f;
                else if (rigid_masked_near(rg, near, sc, ix, iy, iz)) v[u].w = -v[u].w;
            }
        }
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int c = tid + 256 * u;
            if (c >= CELLS) continue;
            if (!on[u]) v[u].w = 0.f;
            buf[0][c] = v[u];
        }
        __syncthreads();
#pragma unroll
        for (int s = 1; s <= K; ++s) {
            const float4* a = buf[(s - 1) & 1];
            float4* b = buf[s & 1];
            const int first = s, side = R - 2 * s;  // cells [first, first + side) on each axis
            for (int c = tid; c < side * side * side; c += 256) {
                const int lx = first + c % side, ly = first + (c / side) % side, lz = first + c / (side * side);
                const int at = lx + R * (ly + R * lz);
                const float4 me = a[at];
                const float m = me.w;
                float4 out = me;
                if (m > 0.f) {
                    const int off[6] = {1, -1, R, -R, R * R, -R * R};
                    float ax = 0.f, ay = 0.f, az = 0.f, cnt = 0.f;
#pragma unroll
                    for (int k = 0; k < 6; ++k) {
                        const float4 nb = a[at + off[k]];
                        if (nb.w == 0.f) continue;
                        ax += nb.x;
                        ay += nb.y;
                        az += nb.z;
                        cnt += 1.0f;
                    }
                    out = implicit_cell(sc, me, ax, ay, az, cnt, dt);
                }
                b[at] = out;
            }
            __syncthreads();
        }
        if (tid < 64) {
            const int at = K + (tid & 3) + R * (K + ((tid >> 2) & 3) + R * (K + (tid >> 4)));
            const uint32_t c = (st << 6) | uint32_t(tid);
            const float4 out = buf[K & 1][at];
            const float4 own = src[c];  // empty cells are copied, every cell keeps its mass
            dst[c] = out.w != 0.f ? make_float4(out.x, out.y, out.z, own.w) : own;
        }
        __syncthreads();
    }
    // only flag reads are ordered by the tickets, and a block's are done here
    const uint32_t nd = tickets ? *dcount : 0u;
    if (nd == 0u || blockIdx.x >= walk.n) return;
    if (tid == 0) s_last = last_block(tickets, min(gridDim.x, walk.n)) ? 1u : 0u;
    __syncthreads();
    if (!s_last) return;
    for (uint32_t i = tid; i < nd; i += 256u) g.tile_flag[dlist[i]] &= ~FLAG_DYN;
}

// One sweep per launch, a wave per tile and a lane per cell: half the cell
// updates of K = 2, a quarter of K = 3.  A chain of dependent loads per wave,
// so it needs its 8,192 waves in flight at once: with the tickets in it, 96
// scalar registers, seven blocks fitted on a CU and 32,768 tiles took 50
// instead of 32 us.
__global__ __launch_bounds__(256) void k_implicit_sweep(const SceneDev* __restrict__ scenes, GridDev g,
                                                        const float4* __restrict__ src, float4* __restrict__ dst,
                                                        const uint32_t* __restrict__ dlist,
                                                        const uint32_t* __restrict__ dcount, float dt, RigidDev rg) {
    const TileWalk walk(g, dcount);
    const int lane = threadIdx.x & 63;
    for (uint32_t i = blockIdx.x * 4 + uint32_t(wave_id()); i < walk.n; i += gridDim.x * 4) {
        uint32_t t, st;
        walk.at(g, dlist, i, t, st);
        const SceneDev sc = scenes[g.tile_scene[t]];
        int tx, ty, tz, ix, iy, iz;
        tile_cell(sc, t, lane, tx, ty, tz, ix, iy, iz);
        const uint32_t c = (st << 6) | uint32_t(lane);
        const float4 me = src[c];
        // empty cells and cells stamped by a legacy sphere keep their velocity
        if (!(me.w > 1.0e-9f) || rigid_masked_legacy(rg, sc, ix, iy, iz)) {
            dst[c] = me;
            continue;
        }
        const int off[6][3] = {{1, 0, 0}, {-1, 0, 0}, {0, 1, 0}, {0, -1, 0}, {0, 0, 1}, {0, 0, -1}};
        float ax = 0.f, ay = 0.f, az = 0.f, cnt = 0.f;
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const int jx = ix + off[k][0], jy = iy + off[k][1], jz = iz + off[k][2];
            if (!in_grid(sc, jx, jy, jz)) continue;
            uint32_t nc;
            if (g.tile_slot) {
                if (!cell_storage(sc, g.tile_slot, jx, jy, jz, nc)) continue;  // no slot: no P2G mass
            } else {
                nc = cell_index(sc, jx, jy, jz);
                if ((g.tile_flag[nc >> 6] & (FLAG_STATIC | FLAG_DYN)) == 0u) continue;
            }
            const float4 nb = src[nc];
            if (!(nb.w > 1.0e-9f)) continue;
            ax += nb.x;
            ay += nb.y;
            az += nb.z;
            cnt += 1.0f;
        }
        dst[c] = implicit_cell(sc, me, ax, ay, az, cnt, dt);
    }
}

// Takes FLAG_DYN off the listed tiles.
__global__ __launch_bounds__(256) void k_end_dynamic(GridDev g, const uint32_t* __restrict__ dlist,
                                                     const uint32_t* __restrict__ dcount) {
    const uint32_t nd = *dcount;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nd; i += gridDim.x * blockDim.x)
        g.tile_flag[dlist[i]] &= ~FLAG_DYN;
}

constexpr uint32_t SWEEPS_PER_LAUNCH = 3;

float4* implicit_first(float4* gv, float4* scratch, uint32_t iters, bool many) {
    const uint32_t launches = many ? iters : (iters + SWEEPS_PER_LAUNCH - 1) / SWEEPS_PER_LAUNCH;
    return launches % 2 ? scratch : gv;
}

hipError_t launch_implicit_sweeps(const SceneDev* scenes, const GridDev& g, float4* scratch, uint32_t iters, bool many,
                                  const uint32_t* dlist, const uint32_t* dcount, float dt, int blocks, uint32_t* tickets,
                                  bool end, bool listed, hipStream_t s, const RigidDev* rigid) {
    const RigidDev rg = rigid ? *rigid : RigidDev{nullptr, nullptr, 0u, 0u};
    // one block takes the few marks of escaped particles off by the way
    const bool ticket = end && !many && !listed;
    float4* a = implicit_first(g.gv, scratch, iters, many);
    while (iters > 0) {
        float4* b = a == scratch ? g.gv : scratch;
        const uint32_t k = many ? 1u : std::min(iters, SWEEPS_PER_LAUNCH);
        iters -= k;
        uint32_t* tk = iters == 0 && ticket ? tickets : nullptr;
#define MPM_SWEEPS(K) \
    hipLaunchKernelGGL(k_implicit_sweeps<K>, dim3(blocks), dim3(256), 0, s, scenes, g, a, b, dlist, dcount, dt, rg, tk)
        if (many)
            hipLaunchKernelGGL(k_implicit_sweep, dim3(blocks), dim3(256), 0, s, scenes, g, a, b, dlist, dcount, dt, rg);
        else if (k == 3) MPM_SWEEPS(3);
        else if (k == 2) MPM_SWEEPS(2);
        else MPM_SWEEPS(1);
#undef MPM_SWEEPS
        a = b;
    }
    if (end && !ticket) hipLaunchKernelGGL(k_end_dynamic, dim3(256), dim3(256), 0, s, g, dlist, dcount);
    return hipGetLastError();
}

// Zero the accumulation grid of the static and dynamic lists; keep only the
// static bit.
// `also` (may be null) is a second per-cell buffer cleared on the same tiles.
// The dynamic list's count is cleared by the last of the blocks that have a
// tile, once all of them have read it; with no dynamic tile, the usual case,
// nobody takes a ticket.  A launch of its own for that one word cost 4.7 us of
// each frame, and of each reversed substep with escaped particles; the tickets
// cost 2,048 blocks about 1 us (clear of 30,000 dynamic tiles 9 us, 8.4 before
// that launch).
__global__ __launch_bounds__(256) void k_clear_tiles(GridDev g, const uint32_t* __restrict__ dlist, uint32_t* dcount,
                                                     uint32_t* tickets, float4* also) {
    const TileWalk walk(g, dcount);
    const uint32_t nd = *dcount;
    const int lane = threadIdx.x & 63;
    for (uint32_t i = blockIdx.x * 4 + uint32_t(wave_id()); i < walk.n; i += gridDim.x * 4) {
        uint32_t t, st;
        walk.at(g, dlist, i, t, st);
        g.gmp[(st << 6) | uint32_t(lane)] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (also) also[(st << 6) | uint32_t(lane)] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (lane == 0) g.tile_flag[t] &= FLAG_STATIC;
    }
    // a block without a tile may read the count before or after: it is done
    const uint32_t busy = max(min(gridDim.x, (walk.n + 3u) / 4u), 1u);
    if (blockIdx.x >= busy || nd == 0u) return;
    __syncthreads();  // the block's four waves have read the count
    if (threadIdx.x == 0 && last_block(tickets, busy)) *dcount = 0u;
}

__global__ void k_set_u32(uint32_t* p, uint32_t v) { *p = v; }

hipError_t launch_set_u32(uint32_t* p, uint32_t v, hipStream_t s) {
    hipLaunchKernelGGL(k_set_u32, dim3(1), dim3(1), 0, s, p, v);
    return hipGetLastError();
}

// Status bookkeeping of the differentiable path without host round trips:
// the escape and fallback counters into dst[0..2).
__global__ void k_snap_counters(const uint32_t* status, uint32_t* dst) {
    dst[0] = status[ST_ESCAPES];
    dst[1] = status[ST_FALLBACK];
}

hipError_t launch_snap_counters(const uint32_t* status, uint32_t* dst, hipStream_t s) {
    hipLaunchKernelGGL(k_snap_counters, dim3(1), dim3(1), 0, s, status, dst);
    return hipGetLastError();
}

// Sum of the per-chunk (dJ/dmu, dJ/dlambda) pairs v[2i], v[2i+1], i < *count
// (clamped to cap), in a fixed order: thread t adds entries t, t+256, ...
// in sequence, then a fixed tree combines the 256 partials.  One block.
__global__ __launch_bounds__(256) void k_sum_pairs(const double* __restrict__ v, const uint32_t* count, uint32_t cap,
                                                   double* __restrict__ out) {
    __shared__ double sm[2][256];
    const uint32_t n = min(*count, cap);
    double a = 0.0, b = 0.0;
    for (uint32_t i = threadIdx.x; i < n; i += 256) {
        a += v[2 * (size_t)i];
        b += v[2 * (size_t)i + 1];
    }
    sm[0][threadIdx.x] = a;
    sm[1][threadIdx.x] = b;
    __syncthreads();
    for (uint32_t h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) {
            sm[0][threadIdx.x] += sm[0][threadIdx.x + h];
            sm[1][threadIdx.x] += sm[1][threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = sm[0][0];
        out[1] = sm[1][0];
    }
}

hipError_t launch_sum_pairs(const double* v, const uint32_t* count, uint32_t cap, double* out, hipStream_t s) {
    hipLaunchKernelGGL(k_sum_pairs, dim3(1), dim3(256), 0, s, v, count, cap, out);
    return hipGetLastError();
}

hipError_t launch_clear_tiles(const GridDev& g, const uint32_t* dlist, uint32_t* dcount, uint32_t* tickets, int blocks,
                              hipStream_t s, float4* also) {
    hipLaunchKernelGGL(k_clear_tiles, dim3(blocks), dim3(256), 0, s, g, dlist, dcount, tickets, also);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Tile keys, written at the particle's original id so that a stable sort over
// ids 0..n-1 reproduces the reference order, or (the layout sort) at the
// particle's slot, so ties keep the current slot order and the reorder gather
// reads nearly sequential memory.
__global__ __launch_bounds__(256) void k_tile_keys(StepArgs a, uint32_t* __restrict__ keys_out, int by_slot) {
    for (uint32_t ci = blockIdx.x; ci < a.n_chunks; ci += gridDim.x) {
        const Chunk ch = a.chunks[ci];
        if (threadIdx.x >= ch.count) continue;
        const uint32_t slot = ch.start + threadIdx.x;
        const uint32_t at = by_slot ? slot : __float_as_uint(a.ps[(size_t)CID * a.cap + slot]);
        keys_out[at] = tile_key(a.scenes[ch.scene], a.ps, a.cap, slot);
    }
}

hipError_t launch_tile_keys(const StepArgs& a, uint32_t* keys_out, int by_slot, hipStream_t s) {
    if (a.n_chunks == 0) return hipSuccess;
    unsigned blocks = a.n_chunks < 65535u ? a.n_chunks : 65535u;
    hipLaunchKernelGGL(k_tile_keys, dim3(blocks), dim3(256), 0, s, a, keys_out, by_slot);
    return hipGetLastError();
}

// src_slot[j] = slot_of_id[sorted_ids[j]]; then every plane is gathered with
// one (plane, slot) pair per thread so reads and writes stay coalesced.
__global__ void k_reorder_index(const uint32_t* __restrict__ sorted_ids, const uint32_t* __restrict__ slot_of_id,
                                uint32_t* __restrict__ src_slot, uint32_t n) {
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x)
        src_slot[j] = slot_of_id[sorted_ids[j]];
}

hipError_t launch_reorder_index(const uint32_t* sorted_ids, const uint32_t* slot_of_id,
                                uint32_t* src_slot, uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    unsigned blocks = std::min<unsigned>((n + 255) / 256, 8192u);
    hipLaunchKernelGGL(k_reorder_index, dim3(blocks), dim3(256), 0, s, sorted_ids, slot_of_id, src_slot, n);
    return hipGetLastError();
}

// One (static tile, tile row) pair per j: the row's candidate chunk range, as
// add_partials would find it from the tile bounds and the chunk of each slot.
__device__ __forceinline__ void static_record(const RecordArgs& q, uint32_t j) {
    const uint32_t i = j / 9u, r = j % 9u;
    const uint32_t t = q.slist[i], scene = q.tile_scene[t];
    const SceneDev& sc = q.scenes[scene];
    const uint32_t tl = t - sc.tile_base;
    const int W = int(sc.W);
    const int tx = int(tl % sc.W), ty = int((tl / sc.W) % sc.W), tz = int(tl / (sc.W * sc.W));
    const int xa = max(tx - 1, 0), xb = min(tx + 1, W - 1);
    const int nz = tz + int(r) / 3 - 1, ny = ty + int(r) % 3 - 1;
    int c0 = 0, c1 = -1;
    if (nz >= 0 && nz < W && ny >= 0 && ny < W) {
        const uint32_t row = sc.tile_base + uint32_t(W * (ny + W * nz));
        const uint32_t s0 = q.tile_lb[row + xa], s1 = q.tile_lb[row + xb + 1];
        if (s0 < s1) {
            c0 = int(q.chunk_of_slot[s0]);
            c1 = min(int(q.chunk_of_slot[s1 - 1]), int(q.part_capacity) - 1);
        }
    }
    int* rec = q.srec + (size_t)i * SREC_WORDS;
    if (r == 0) {
        rec[0] = int(t);
        rec[1] = int(scene);
    }
    rec[2 + 2 * r] = c0;
    rec[3 + 2 * r] = c1;
}

// One slot per thread through all planes: the index is read once and every
// thread keeps a plane group's loads in flight together.  The first
// `rec_blocks` blocks write the static tiles' records, which need nothing of
// the gather, so they cost no launch of their own.
__global__ __launch_bounds__(256) void k_reorder(const float* __restrict__ src, float* __restrict__ dst,
                                                 uint32_t cap, const uint32_t* __restrict__ src_slot, uint32_t n,
                                                 uint32_t* __restrict__ slot_of_id, RecordArgs rec,
                                                 uint32_t rec_blocks) {
    constexpr int GROUP = 10;
    static_assert(NCOMP % GROUP == 0 && CID == NCOMP - 1, "plane groups; the id is the last plane");
    if (blockIdx.x < rec_blocks) {
        const uint32_t m = min(*rec.scount, rec.max_static) * 9u;
        for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < m; j += rec_blocks * blockDim.x)
            static_record(rec, j);
        return;
    }
    const uint32_t stride = (gridDim.x - rec_blocks) * blockDim.x;
    for (uint32_t j = (blockIdx.x - rec_blocks) * blockDim.x + threadIdx.x; j < n; j += stride) {
        const size_t from = src_slot[j];
        for (int c0 = 0; c0 < NCOMP; c0 += GROUP) {
            float v[GROUP];
#pragma unroll
            for (int c = 0; c < GROUP; ++c) v[c] = src[(size_t)(c0 + c) * cap + from];
#pragma unroll
            for (int c = 0; c < GROUP; ++c) dst[(size_t)(c0 + c) * cap + j] = v[c];
            if (slot_of_id && c0 + GROUP == NCOMP) slot_of_id[__float_as_uint(v[GROUP - 1])] = j;
        }
    }
}

hipError_t launch_reorder(const float* src, float* dst, uint32_t cap, const uint32_t* src_slot, uint32_t n,
                          uint32_t* slot_of_id, const RecordArgs& rec, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const unsigned blocks = std::min<unsigned>((n + 255) / 256, 16384u);
    // nine threads per static tile, whose count is on the device: at most 27
    // tiles a particle; blocks without a tile end at once
    const unsigned rec_blocks = rec.srec ? std::min<unsigned>({rec.max_static / 28u + 1u, n, 1024u}) : 0u;
    hipLaunchKernelGGL(k_reorder, dim3(blocks + rec_blocks), dim3(256), 0, s, src, dst, cap, src_slot, n, slot_of_id,
                       rec, rec_blocks);
    return hipGetLastError();
}

// Spreads the particles of each chunk of the sorted layout over cells: the
// chunk's particles are ranked among those with the same stencil base cell
// (ties by slot) and laid out rank-major, base cells ascending within a rank.
// The sort alone leaves a chunk's particles in arbitrary order inside their
// tiles, so the 64 lanes of a wave fall on ~125 base cells at random and the
// scatter's LDS integer adds to one word from several lanes serialise; in
// rank-major order a wave's lanes mostly hold distinct, neighbouring bases.
// Only the order inside a chunk changes: the chunk list and its partial
// boxes stay valid, and the fixed-point scatter sums do not depend on order.
// src_in/src_out: previous slot of each sorted slot, before and after; the
// sorted tile keys are permuted with them (in place), so each slot keeps the
// key of its own particle for the scatter's escape test.
//
// A chunk lies in one tile row and spans at most eight tiles, so its base
// cells fit SPREAD_X x 5 x 5 cells around its first tile (a particle off the
// grid is clamped to that box; only the order depends on it).
constexpr uint32_t SPREAD_X = 40;     // 8 tiles of 4 cells, one cell before them, rounded up
constexpr uint32_t SPREAD_CELLS = 1024;
static_assert(SPREAD_X * 25 <= SPREAD_CELLS, "base cells of a chunk");

// The partner's word at lane ^ J.
template <uint32_t J>
__device__ __forceinline__ uint32_t lane_xor(uint32_t x) {
    if constexpr (J == 1) return (uint32_t)__builtin_amdgcn_update_dpp(0, int(x), 0xB1, 0xF, 0xF, true);
    else if constexpr (J == 2) return (uint32_t)__builtin_amdgcn_update_dpp(0, int(x), 0x4E, 0xF, 0xF, true);
    else if constexpr (J < 32) return (uint32_t)__builtin_amdgcn_ds_swizzle(int(x), int((J << 10) | 0x1F));
    else return (uint32_t)__shfl_xor((int)x, 32, 64);
}

// Ascending bitonic sort of one word per thread of an N-thread block: the
// word at sorted position t.  Partners closer than a wave are exchanged in
// registers; the steps across waves go through v (LDS, N words).  Every
// thread calls it; v is free again on return.
template <uint32_t N, uint32_t K = 2, uint32_t J = 1>
__device__ __forceinline__ uint32_t block_sort(uint32_t x, uint32_t* v, uint32_t t) {
    uint32_t other;
    if constexpr (J >= 64u) {
        __syncthreads();
        v[t] = x;
        __syncthreads();
        other = v[t ^ J];
    } else {
        other = lane_xor<J>(x);
    }
    // the lower index of a pair keeps the minimum in an ascending run
    const bool keep_min = (t < (t ^ J)) == ((t & K) == 0u);
    x = keep_min ? min(x, other) : max(x, other);
    if constexpr (J > 1u) {
        return block_sort<N, K, J / 2>(x, v, t);
    } else if constexpr (K < N) {
        return block_sort<N, K * 2, K>(x, v, t);
    } else {
        __syncthreads();  // the last cross-wave reads of v are done
        return x;
    }
}

// One thread per particle of a chunk of up to N particles (N = 256 x the
// particles per thread of the pass): a thread of the pass takes positions t,
// t + 256, ..., so each of its passes over the block is rank-major too.
// Ranks come from ballots over the base cell's ten bits and a byte counter per
// wave and cell; one 32-bit bitonic sort of (rank, cell, slot) places the
// particles.  Bound by the latency of its steps: 34 us for 2 M particles in
// 4,100 chunks, 76 us with two 64-bit sorts.
template <uint32_t N>
__global__ __launch_bounds__(N) void k_chunk_spread(const SceneDev* __restrict__ scenes,
                                                    const Chunk* __restrict__ chunks,
                                                    const uint32_t* __restrict__ n_chunks,
                                                    const float* __restrict__ ps, uint32_t cap,
                                                    const uint32_t* __restrict__ src_in,
                                                    uint32_t* __restrict__ src_out, uint32_t* __restrict__ keys,
                                                    uint32_t* __restrict__ chunk_of_slot) {
    constexpr uint32_t NW = N / 64;
    __shared__ uint32_t order[N];
    __shared__ uint32_t srcs[N];
    __shared__ uint32_t tiles[N];
    __shared__ uint32_t cnt_words[NW * SPREAD_CELLS / 4];
    uint8_t* cnt = reinterpret_cast<uint8_t*>(cnt_words);  // [wave][cell]: the wave's particles (at most 64)
    const uint32_t nch = *n_chunks;
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    for (uint32_t ci = blockIdx.x; ci < nch; ci += gridDim.x) {
        const Chunk ch = chunks[ci];
        const uint32_t cnt_ch = min(ch.count, N);
        const SceneDev& sc = scenes[ch.scene];
        const uint32_t ty = ch.pad & 0x7fffu, tz = (ch.pad >> 15) & 0xffffu;
        const uint32_t tx = keys[ch.start] - (sc.tile_base + sc.W * (ty + sc.W * tz));  // first tile
        for (uint32_t i = t; i < NW * SPREAD_CELLS / 4; i += N) cnt_words[i] = 0u;
        const bool live = t < cnt_ch;
        uint32_t src = 0u, tile = 0u, cell = 0u;
        if (live) {
            src = src_in[ch.start + t];
            tile = keys[ch.start + t];
            const int first[3] = {int(4u * tx), int(4u * ty), int(4u * tz)};
            const int most[3] = {int(SPREAD_X) - 1, 4, 4};
            int c[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const float xp = (ps[(size_t)(CX + d) * cap + src] - sc.origin[d]) * sc.inv_dx;
                const int b = int(floorf(xp - 0.5f)) - sc.window[d];
                c[d] = min(max(b - first[d] + 1, 0), most[d]);
            }
            cell = uint32_t(c[0]) + SPREAD_X * uint32_t(c[1] + 5 * c[2]);
        }
        uint64_t same = __ballot(live);
#pragma unroll
        for (int bit = 0; bit < 10; ++bit) {
            const bool on = (cell >> bit) & 1u;
            const uint64_t m = __ballot(on);
            same &= on ? m : ~m;
        }
        uint32_t rank = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
        __syncthreads();
        if (live && rank == 0u) cnt[wave * SPREAD_CELLS + cell] = uint8_t(__popcll(same));
        srcs[t] = src;
        tiles[t] = tile;
        __syncthreads();
#pragma unroll
        for (uint32_t w = 0; w + 1 < NW; ++w)
            if (w < wave) rank += cnt[w * SPREAD_CELLS + cell];
        const uint32_t f = block_sort<N>(live ? (rank << 19) | (cell << 9) | t : ~0u, order, t);
        const uint32_t from = f & 511u;
        if (live) {
            src_out[ch.start + t] = srcs[from];
            keys[ch.start + t] = tiles[from];
            chunk_of_slot[ch.start + t] = ci;
        }
        __syncthreads();
    }
}

hipError_t launch_chunk_spread(const SceneDev* scenes, const Chunk* chunks, const uint32_t* n_chunks,
                               uint32_t max_chunks, const float* ps, uint32_t cap, const uint32_t* src_in,
                               uint32_t* src_out, uint32_t* keys, uint32_t* chunk_of_slot, uint32_t chunk_cap,
                               hipStream_t s) {
    if (max_chunks == 0) return hipSuccess;
    const unsigned blocks = std::min<unsigned>(max_chunks, 8192u);
    if (chunk_cap <= CHUNK_PARTICLES)
        hipLaunchKernelGGL(k_chunk_spread<CHUNK_PARTICLES>, dim3(blocks), dim3(CHUNK_PARTICLES), 0, s, scenes,
                           chunks, n_chunks, ps, cap, src_in, src_out, keys, chunk_of_slot);
    else if (chunk_cap <= CHUNK_PARTICLES * MAX_PPT)
        hipLaunchKernelGGL(k_chunk_spread<CHUNK_PARTICLES * MAX_PPT>, dim3(blocks), dim3(CHUNK_PARTICLES * MAX_PPT),
                           0, s, scenes, chunks, n_chunks, ps, cap, src_in, src_out, keys, chunk_of_slot);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_chunk_slots(const Chunk* __restrict__ chunks,
                                                     const uint32_t* __restrict__ n_chunks,
                                                     uint32_t* __restrict__ chunk_of_slot) {
    const uint32_t nch = *n_chunks;
    for (uint32_t ci = blockIdx.x; ci < nch; ci += gridDim.x) {
        const Chunk ch = chunks[ci];
        for (uint32_t i = threadIdx.x; i < ch.count; i += blockDim.x) chunk_of_slot[ch.start + i] = ci;
    }
}

hipError_t launch_chunk_slots(const Chunk* chunks, const uint32_t* n_chunks, uint32_t max_chunks,
                              uint32_t* chunk_of_slot, hipStream_t s) {
    if (max_chunks == 0) return hipSuccess;
    hipLaunchKernelGGL(k_chunk_slots, dim3(std::min<unsigned>(max_chunks, 8192u)), dim3(256), 0, s, chunks, n_chunks,
                       chunk_of_slot);
    return hipGetLastError();
}

// One thread per particle, a block per chunk of the unsorted list (one scene).
// Bound by the 124 bytes it writes per particle: the planes of 1.78 M
// particles in 52 us, where 30 planes built on the host and copied one by
// one took 10 ms.
__global__ __launch_bounds__(256) void k_init_particles(const SceneDev* __restrict__ scenes,
                                                        const Chunk* __restrict__ chunks, uint32_t n_chunks,
                                                        const float* __restrict__ pos, const float* __restrict__ vel,
                                                        float* __restrict__ ps, uint32_t cap,
                                                        uint32_t* __restrict__ slot_of_id) {
    for (uint32_t ci = blockIdx.x; ci < n_chunks; ci += gridDim.x) {
        const Chunk ch = chunks[ci];
        if (threadIdx.x >= ch.count) continue;
        const SceneDev& sc = scenes[ch.scene];
        const uint32_t j = ch.start + threadIdx.x;
        auto put = [&](int c, float v) { ps[(size_t)c * cap + j] = v; };
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            put(CX + k, pos[3 * (size_t)j + k]);
            put(CV + k, vel ? vel[3 * (size_t)j + k] : 0.0f);
        }
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            put(CC + k, 0.0f);
            put(CF + k, k % 4 == 0 ? 1.0f : 0.0f);
        }
        put(CJP, 0.0f);
        put(CMASS, sc.pmass);
        put(CVOL, sc.pvol);
        put(CE, sc.youngs);
        put(CMAT, 0.0f);  // material row 0
        put(CID, __uint_as_float(j));
        slot_of_id[j] = j;
    }
}

hipError_t launch_init_particles(const SceneDev* scenes, const Chunk* chunks, uint32_t n_chunks, const float* pos,
                                 const float* vel, float* ps, uint32_t cap, uint32_t* slot_of_id, hipStream_t s) {
    if (n_chunks == 0) return hipSuccess;
    hipLaunchKernelGGL(k_init_particles, dim3(std::min(n_chunks, 65535u)), dim3(256), 0, s, scenes, chunks, n_chunks,
                       pos, vel, ps, cap, slot_of_id);
    return hipGetLastError();
}

__global__ void k_index_slots(const float* __restrict__ ps, uint32_t cap, uint32_t* __restrict__ slot_of_id,
                              uint32_t n) {
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x)
        slot_of_id[__float_as_uint(ps[(size_t)CID * cap + j])] = j;
}

hipError_t launch_index_slots(const float* ps, uint32_t cap, uint32_t* slot_of_id, uint32_t n,
                              hipStream_t s) {
    if (n == 0) return hipSuccess;
    unsigned blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_index_slots, dim3(blocks), dim3(256), 0, s, ps, cap, slot_of_id, n);
    return hipGetLastError();
}

// NC planes <-> an array of NC words per particle in original order.  `ids` is
// the id plane of the same slot order.  One thread per slot: the plane side is
// coalesced and the array side moves NC consecutive words per particle, where
// one thread per id would touch a 64-byte sector of every plane for 4 bytes.
// Bound by the scattered sectors of the array side.  2 M particles in tile
// order: x, v (3 words each) and F (9) take 152 us, by id they took 508 us.
template <int NC>
__global__ __launch_bounds__(256) void k_unpermute(const float* __restrict__ ps, uint32_t cap, int comp0,
                                                   const float* __restrict__ ids, float* __restrict__ out, uint32_t n) {
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
        const uint32_t id = __float_as_uint(ids[j]);
        float v[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) v[c] = ps[(size_t)(comp0 + c) * cap + j];
        __builtin_memcpy(out + (size_t)id * NC, v, sizeof(v));
    }
}

template <int NC>
__global__ __launch_bounds__(256) void k_permute_in(float* __restrict__ ps, uint32_t cap, int comp0,
                                                    const float* __restrict__ ids, const float* __restrict__ in,
                                                    uint32_t n) {
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
        const uint32_t id = __float_as_uint(ids[j]);
        float v[NC];
        __builtin_memcpy(v, in + (size_t)id * NC, sizeof(v));
#pragma unroll
        for (int c = 0; c < NC; ++c) ps[(size_t)(comp0 + c) * cap + j] = v[c];
    }
}

hipError_t launch_unpermute(const float* ps, uint32_t cap, int comp0, int ncomp, const float* ids, float* out,
                            uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const dim3 g(std::min<unsigned>((n + 255) / 256, 8192u)), b(256);
    if (ncomp == 1) hipLaunchKernelGGL(k_unpermute<1>, g, b, 0, s, ps, cap, comp0, ids, out, n);
    else if (ncomp == 3) hipLaunchKernelGGL(k_unpermute<3>, g, b, 0, s, ps, cap, comp0, ids, out, n);
    else if (ncomp == 9) hipLaunchKernelGGL(k_unpermute<9>, g, b, 0, s, ps, cap, comp0, ids, out, n);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_permute_in(float* ps, uint32_t cap, int comp0, int ncomp, const float* ids, const float* in,
                             uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const dim3 g(std::min<unsigned>((n + 255) / 256, 8192u)), b(256);
    if (ncomp == 1) hipLaunchKernelGGL(k_permute_in<1>, g, b, 0, s, ps, cap, comp0, ids, in, n);
    else if (ncomp == 3) hipLaunchKernelGGL(k_permute_in<3>, g, b, 0, s, ps, cap, comp0, ids, in, n);
    else if (ncomp == 9) hipLaunchKernelGGL(k_permute_in<9>, g, b, 0, s, ps, cap, comp0, ids, in, n);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// ---- soil checkpoint streams (mpm_checkpoint.rs:78-83, :352-369) ----------
// The archive holds n particles as nine streams, stream-major, 40 words per
// particle: position+w (4), velocity+w (4), C (12), F (12), volume, mass,
// log-Jp, material id, tire compaction (4).  C and F are three 16-byte
// columns, word 4j+i = M_ij, word 4j+3 a pad.  The planes hold M row-major
// (plane 3i+j).  `aux` keeps, by particle id, the words the planes do not:
// position w [n], velocity w [n], C pads [3n], F pads [3n], tire [4n]; a null
// aux reads as zeros.  Every stream offset is a multiple of 4 words from a
// 256-byte-aligned base, so the 4-word groups move as 16-byte accesses.
__global__ void k_ckpt_pack(const float* __restrict__ ps, uint32_t cap, const uint32_t* __restrict__ slot_of_id,
                            const uint32_t* __restrict__ aux, int zero_w, uint32_t n, uint32_t* __restrict__ out) {
    const size_t N = n;
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
        const size_t s = slot_of_id[p];
        auto P = [&](int c) { return __float_as_uint(ps[(size_t)c * cap + s]); };
        auto A = [&](size_t i) { return aux ? aux[i] : 0u; };
        // a step stores w = 0 (mpm.wgsl:1349-1350)
        reinterpret_cast<uint4*>(out)[p] = make_uint4(P(CX), P(CX + 1), P(CX + 2), zero_w ? 0u : A(p));
        reinterpret_cast<uint4*>(out + 4 * N)[p] = make_uint4(P(CV), P(CV + 1), P(CV + 2), zero_w ? 0u : A(N + p));
        for (int j = 0; j < 3; ++j) {
            reinterpret_cast<uint4*>(out + 8 * N)[3 * p + j] =
                make_uint4(P(CC + j), P(CC + 3 + j), P(CC + 6 + j), A(2 * N + 3 * p + j));
            reinterpret_cast<uint4*>(out + 20 * N)[3 * p + j] =
                make_uint4(P(CF + j), P(CF + 3 + j), P(CF + 6 + j), A(5 * N + 3 * p + j));
        }
        out[32 * N + p] = P(CVOL);
        out[33 * N + p] = P(CMASS);
        out[34 * N + p] = P(CJP);
        out[35 * N + p] = P(CMAT);
        const size_t t = 8 * N + 4 * (size_t)p;
        reinterpret_cast<uint4*>(out + 36 * N)[p] = make_uint4(A(t), A(t + 1), A(t + 2), A(t + 3));
    }
}

// Inverse of k_ckpt_pack into slot = id order; E is the scene's, the id plane
// the identity.  `aux` (12n words) receives the words the planes do not hold.
__global__ void k_ckpt_unpack(const uint32_t* __restrict__ in, uint32_t n, float* __restrict__ ps, uint32_t cap,
                              float youngs, uint32_t* __restrict__ aux) {
    const size_t N = n;
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
        auto put = [&](int c, uint32_t w) { ps[(size_t)c * cap + p] = __uint_as_float(w); };
        const uint4 x = reinterpret_cast<const uint4*>(in)[p];
        const uint4 v = reinterpret_cast<const uint4*>(in + 4 * N)[p];
        put(CX, x.x), put(CX + 1, x.y), put(CX + 2, x.z);
        put(CV, v.x), put(CV + 1, v.y), put(CV + 2, v.z);
        aux[p] = x.w;
        aux[N + p] = v.w;
        for (int j = 0; j < 3; ++j) {
            const uint4 c = reinterpret_cast<const uint4*>(in + 8 * N)[3 * p + j];
            const uint4 f = reinterpret_cast<const uint4*>(in + 20 * N)[3 * p + j];
            put(CC + j, c.x), put(CC + 3 + j, c.y), put(CC + 6 + j, c.z);
            put(CF + j, f.x), put(CF + 3 + j, f.y), put(CF + 6 + j, f.z);
            aux[2 * N + 3 * p + j] = c.w;
            aux[5 * N + 3 * p + j] = f.w;
        }
        put(CVOL, in[32 * N + p]);
        put(CMASS, in[33 * N + p]);
        put(CJP, in[34 * N + p]);
        put(CMAT, in[35 * N + p]);
        const uint4 t = reinterpret_cast<const uint4*>(in + 36 * N)[p];
        const size_t a = 8 * N + 4 * (size_t)p;
        aux[a] = t.x, aux[a + 1] = t.y, aux[a + 2] = t.z, aux[a + 3] = t.w;
        ps[(size_t)CE * cap + p] = youngs;
        put(CID, p);
    }
}

hipError_t launch_ckpt_pack(const float* ps, uint32_t cap, const uint32_t* slot_of_id, const uint32_t* aux,
                            int zero_w, uint32_t n, uint32_t* out, hipStream_t s) {
    if (n == 0) return hipSuccess;
    unsigned blocks = std::min<unsigned>((n + 255) / 256, 8192);
    hipLaunchKernelGGL(k_ckpt_pack, dim3(blocks), dim3(256), 0, s, ps, cap, slot_of_id, aux, zero_w, n, out);
    return hipGetLastError();
}

hipError_t launch_ckpt_unpack(const uint32_t* in, uint32_t n, float* ps, uint32_t cap, float youngs,
                              uint32_t* aux, hipStream_t s) {
    if (n == 0) return hipSuccess;
    unsigned blocks = std::min<unsigned>((n + 255) / 256, 8192);
    hipLaunchKernelGGL(k_ckpt_unpack, dim3(blocks), dim3(256), 0, s, in, n, ps, cap, youngs, aux);
    return hipGetLastError();
}

__global__ void k_grid_to_dense(const float4* __restrict__ gmp, const SceneDev* __restrict__ scenes,
                                uint32_t scene, uint32_t G, float* __restrict__ mass, float* __restrict__ mom) {
    const SceneDev sc = scenes[scene];
    const size_t total = (size_t)G * G * G;
    for (size_t c = blockIdx.x * (size_t)blockDim.x + threadIdx.x; c < total; c += (size_t)gridDim.x * blockDim.x) {
        int ix = int(c % G), iy = int((c / G) % G), iz = int(c / ((size_t)G * G));
        float4 q = gmp[cell_index(sc, ix, iy, iz)];
        mass[c] = q.x;
        mom[3 * c] = q.y;
        mom[3 * c + 1] = q.z;
        mom[3 * c + 2] = q.w;
    }
}

hipError_t launch_grid_to_dense(const float4* gmp, const SceneDev* scenes, uint32_t scene,
                                uint32_t G, float* mass, float* mom, hipStream_t s) {
    size_t total = (size_t)G * G * G;
    unsigned blocks = (unsigned)((total + 255) / 256);
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_grid_to_dense, dim3(blocks), dim3(256), 0, s, gmp, scenes, scene, G, mass, mom);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Deterministic gather-order P2G (mpm_deterministic_p2g.wgsl:12-150).
// Per particle: affine matrix A (planes 0-8) and m v (planes 9-11).
template <int MODEL>
__global__ __launch_bounds__(256) void k_gather_prepare(StepArgs a, float* __restrict__ aff) {
    const uint32_t cap = a.cap;
    const float* ps = a.ps;
    for (uint32_t ci = blockIdx.x; ci < a.n_chunks; ci += gridDim.x) {
        const Chunk ch = const_load(a.chunks + ci);
        if (threadIdx.x >= ch.count) continue;
        const SceneDev sc = const_load(a.scenes + ch.scene);
        const uint32_t slot = ch.start + threadIdx.x;
        float F[9], C[9];
        for (int k = 0; k < 9; ++k) {
            F[k] = ps[(size_t)(CF + k) * cap + slot];
            C[k] = ps[(size_t)(CC + k) * cap + slot];
        }
        const float m = ps[(size_t)CMASS * cap + slot], vol = ps[(size_t)CVOL * cap + slot];
        const float jp = ps[(size_t)CJP * cap + slot];
        const float* mrow = mat_row(a, sc, __float_as_uint(ps[(size_t)CMAT * cap + slot]));
        float mu = sc.mu, lam = sc.lam;
        if (a.has_E) {
            float E = ps[(size_t)CE * cap + slot];
            mu = E / (2.0f * (1.0f + sc.poisson));
            lam = E * sc.poisson / ((1.0f + sc.poisson) * (1.0f - 2.0f * sc.poisson));
        }
        Svd32 d;
        svd3<MODEL>(F, d);
        float A[9];
        affine_from_svd<MODEL>(sc, mrow, d, mu, lam, jp, a.dt, vol, m, C, A);
        for (int k = 0; k < 9; ++k) aff[(size_t)k * cap + slot] = A[k];
        for (int k = 0; k < 3; ++k) aff[(size_t)(9 + k) * cap + slot] = m * ps[(size_t)(CV + k) * cap + slot];
    }
}

hipError_t launch_gather_prepare(const StepArgs& a, float* affine, int blocks, hipStream_t s) {
    if (a.n_chunks == 0) return hipSuccess;
    if (blocks <= 0 || uint32_t(blocks) > a.n_chunks) blocks = int(a.n_chunks);
    // the model is uniform per context; scenes[0] tells which
    SceneDev h;
    (void)h;
    hipLaunchKernelGGL((k_gather_prepare<MODEL_SHADER>), dim3(blocks), dim3(256), 0, s, a, affine);
    return hipGetLastError();
}

// One block per active tile, or a wave.  For each cell, the particles of the 27 neighbour
// tiles are listed in tile order dx + 3 dy + 9 dz, then in ascending sorted
// slot (mpm_deterministic_p2g.wgsl:100-144), and summed in a fixed order, so
// the result is bitwise repeatable: 16 sums of every 16th particle, then a
// tree, which rounds less than one serial sum (5,003 particles over a few
// tiles: momentum 2.0e-7 off instead of 1.7e-6).  The 27 tiles are nine x-rows
// of consecutive keys, i.e. nine slot ranges of the tile lower-bound table,
// already in that order.
//   1. The block tests the ranges' particles, GATHER_PER per thread at once,
//      and keeps the slots whose stencil reaches the tile (about 1 in 8), in
//      order, in an LDS list.
//   2. In batches of GATHER_RECS the listed particles' weights, node offsets
//      and momentum rows go to LDS, one particle per thread.
//   3. Each of the block's 16 waves takes one x-row of the tile and the records
//      that reach its row, 16 at a time: a lane sums one channel of the row's
//      four cells over every 16th record, and the 16 partial sums are added in
//      a fixed tree at the end.
// One wave per tile that walked every particle of the 27 tiles through
// dependent global loads took 2,352 us on 16,384 sand particles in a 32^3 grid.
// With the records in LDS, reading them is what counts: one wave per z with a
// lane per cell and channel 115 us, a wave per row with 16 lanes per record
// 62 us (36 LDS instructions per 16 records, 12 of them to bring the terms to
// one serial sum); a lane per record and channel reads each record once for
// four cells, 6 LDS instructions per 16 records: 38 us, and 35 with a batch's
// loads issued before the sums of the one before.
// A block fills its CU, so a grid of many thin tiles (20,000 particles over
// 128^3 cells: 32,768 active tiles of 5 candidates) waits for one tile after
// the other, 641 us against 190 with a tile per wave.  Scenes of more than 512
// active tiles and fewer than GATHER_THIN particles a tile therefore give a
// block 16 tiles at once; a wave sums a tile of up to GATHER_WAVE_RECS records
// by itself, row by row and in the same order, and what is left goes to the
// block.  A substep with / without it: 1,000 particles over 64^3 113 / 188 us,
// 3,000 over 40^3 102 / 112, 20,000 over 128^3 361 / 897, 40,000 over 96^3 242 /
// 455, 200,000 over 128^3 461 / 930.  Denser or fewer tiles are faster with the
// block's whole attention: 20,000 particles over 27^3 cells 106 / 128 us,
// 300,000 over 46^3 289 / 322, 16,384 sand particles (a frame of 4) 170 / 176.
// The line lies where a tile's records outgrow its wave: eight particles a tile
// are 27 records.
constexpr int GATHER_THREADS = 1024;
constexpr int GATHER_WAVES = GATHER_THREADS / 64;
constexpr int GATHER_PER = 4;
constexpr int GATHER_FLY = 2;  // records per lane in flight
constexpr int GATHER_STEP = 16 * GATHER_FLY;
constexpr int GATHER_RECS = 512;
constexpr int GATHER_LIST = 8192;
constexpr int GATHER_WAVE_RECS = GATHER_RECS / GATHER_WAVES;
constexpr int GATHER_GRID = 2048;
constexpr int GATHER_BLOCKS = 256;  // one per CU
constexpr uint32_t GATHER_THIN = 8;  // particles per active tile
static_assert(GATHER_WAVE_RECS <= GATHER_STEP && GATHER_RECS + GATHER_STEP >= 8 * GATHER_STEP, "four lists of a step each");

// A particle relative to a tile: the four channels as c + r0 d0 + r1 d1 + r2 d2
// (mass: r = 0), the weight product of the tile's 4 x 4 cell columns in x and y
// (-1: the stencil misses the column), weight and node offset in z, node offset
// in y, and in x the first cell's offset in cells and the fraction.
struct alignas(16) GatherRec {
    float4 row[4];
    float4 wxy[4];
    float2 z[4];
    float4 dy;
    float2 x;
    float pad[6];  // 52 words: 16 records' rows lie in different LDS banks
};

// Stencil base of a position relative to the tile tc (the tile's first cell's
// offset in it) and its fraction.
__device__ __forceinline__ void gather_stencil(const SceneDev& sc, const int* tc, const float* x, int* r, float* fx) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float xp = (x[k] - sc.origin[k]) * sc.inv_dx;
        const float bf = floorf(xp - 0.5f);
        fx[k] = xp - bf;
        r[k] = 4 * tc[k] - (int(bf) - sc.window[k]);
    }
}

// A particle's record; returns its x-rows of the tile (bit y + 4 z).
__device__ __forceinline__ uint32_t gather_record(const SceneDev& sc, const int* tc, const float* px, const float* A,
                                                  float mass, GatherRec& q) {
    int r[3];
    float fx[3];
    gather_stencil(sc, tc, px, r, fx);
    float w[3][4], d[3][4];  // weight (-1: none) and node offset of the tile's cells
    uint32_t in[3] = {0u, 0u, 0u}, rm = 0u;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float wk[3];
        quad_weights(fx[k], wk);
#pragma unroll
        for (int c2 = 0; c2 < 4; ++c2) {
            const int off = r[k] + c2;
            w[k][c2] = off == 0 ? wk[0] : (off == 1 ? wk[1] : (off == 2 ? wk[2] : -1.0f));
            d[k][c2] = (float(off) - fx[k]) * sc.dx;
            if (off >= 0 && off <= 2) in[k] |= 1u << c2;
        }
    }
#pragma unroll
    for (int z = 0; z < 4; ++z)
        if (in[2] & (1u << z)) rm |= in[1] << (4 * z);
#pragma unroll
    for (int y = 0; y < 4; ++y) {
        float v[4];
#pragma unroll
        for (int c2 = 0; c2 < 4; ++c2) v[c2] = w[0][c2] < 0.f || w[1][y] < 0.f ? -1.0f : w[0][c2] * w[1][y];
        q.wxy[y] = make_float4(v[0], v[1], v[2], v[3]);
        q.z[y] = make_float2(w[2][y], d[2][y]);
    }
    q.dy = make_float4(d[1][0], d[1][1], d[1][2], d[1][3]);
    q.x = make_float2(float(r[0]), fx[0]);
    q.row[0] = make_float4(mass, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < 3; ++k) q.row[1 + k] = make_float4(A[9 + k], A[3 * k], A[3 * k + 1], A[3 * k + 2]);
    return rm;
}

// Adds a record to the lane's four cells of the x-row (cy, cz), channel
// lane & 3.
__device__ __forceinline__ void gather_add(const GatherRec& q, int cy, int cz, float dx, float* acc) {
    const float4 r = q.row[threadIdx.x & 3], wv = q.wxy[cy];
    const float2 z = q.z[cz], qx = q.x;
    const float base = r.x + r.z * reinterpret_cast<const float*>(&q.dy)[cy] + r.w * z.y;
    const float w[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
    for (int c2 = 0; c2 < 4; ++c2) {
        const float t = w[c2] * z.x * (base + r.y * ((qx.x + float(c2) - qx.y) * dx));
        acc[c2] += w[c2] < 0.f ? 0.f : t;
    }
}

// The tree over the 16 sums, and the row's cells.
__device__ __forceinline__ void gather_store(const SceneDev& sc, const int* tc, uint32_t t, int cy, int cz, float* acc,
                                             float4* gmp) {
    const int lane = threadIdx.x & 63, ch = lane & 3, grp = lane >> 2;
#pragma unroll
    for (int c2 = 0; c2 < 4; ++c2)
#pragma unroll
        for (int o = 4; o < 64; o *= 2) acc[c2] += __shfl_xor(acc[c2], o, 64);
    if (grp >= 4) return;  // lane's cell of the row
    const int G = int(sc.G);
    const bool valid = 4 * tc[0] + grp < G && 4 * tc[1] + cy < G && 4 * tc[2] + cz < G;
    const uint32_t c = (t << 6) | uint32_t(grp | (cy << 2) | (cz << 4));
    const float v = grp == 0 ? acc[0] : (grp == 1 ? acc[1] : (grp == 2 ? acc[2] : acc[3]));
    reinterpret_cast<float*>(gmp)[4 * (size_t)c + ch] = valid ? v : 0.f;
}

__global__ __launch_bounds__(GATHER_THREADS) void k_gather_p2g(StepArgs a, const uint32_t* __restrict__ tile_scene,
                                                               const uint32_t* __restrict__ lb,
                                                               const float* __restrict__ aff,
                                                               const uint32_t* __restrict__ list,
                                                               const uint32_t* __restrict__ count, uint32_t thin) {
    __shared__ GatherRec rec[GATHER_RECS + 1];  // the last one reaches no cell
    __shared__ uint16_t rows[GATHER_RECS];      // bit y + 4 z: the record reaches that x-row of the tile
    __shared__ uint16_t wlist[GATHER_WAVES][GATHER_RECS + GATHER_STEP];
    __shared__ uint32_t slots[GATHER_LIST];
    __shared__ alignas(16) uint32_t rbeg[GATHER_WAVES][12], roff[GATHER_WAVES][12];  // each wave's tile's ranges
    __shared__ uint32_t wcnt[64];  // [GATHER_PER][GATHER_WAVES]
    __shared__ uint4 whole[GATHER_WAVES];  // a wave's tile that needs the block: id (~0: none), scene, coordinates
    static_assert(GATHER_PER * GATHER_WAVES <= 64, "one lane per count");
    const uint32_t n = *count;
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
    const uint32_t cap = a.cap;
    const uint64_t lt = (1ull << lane) - 1ull;
    if (tid < int(sizeof(GatherRec) / 4))
        reinterpret_cast<float*>(&rec[GATHER_RECS])[tid] = tid >= 16 && tid < 32 ? -1.f : 0.f;
    __syncthreads();
    auto tile = [&](uint32_t t, uint32_t scene, SceneDev& sc, int* tc) __attribute__((always_inline)) {
        sc = const_load(a.scenes + scene);
        const uint32_t tl = t - sc.tile_base;
        tc[0] = int(tl % sc.W);
        tc[1] = int((tl / sc.W) % sc.W);
        tc[2] = int(tl / (sc.W * sc.W));
    };
    // slot of candidate j of a wave's tile, and whether its stencil reaches the tile
    auto candidate = [&](int w, uint32_t j) __attribute__((always_inline)) {
        int r = 0;
#pragma unroll
        for (int q = 1; q < 9; ++q) r += j >= roff[w][q] ? 1 : 0;
        return rbeg[w][r] + (j - roff[w][r]);
    };
    auto reaches = [&](const SceneDev& sc, const int* tc, uint32_t j) __attribute__((always_inline)) {
        const float x[3] = {a.ps[(size_t)CX * cap + j], a.ps[(size_t)(CX + 1) * cap + j],
                            a.ps[(size_t)(CX + 2) * cap + j]};
        int r[3];
        float fx[3];
        gather_stencil(sc, tc, x, r, fx);
        bool hit = true;
#pragma unroll
        for (int k = 0; k < 3; ++k) hit = hit && r[k] >= -3 && r[k] <= 2;
        return hit;
    };
    float px[3], A[12], mass = 0.f;
    auto load = [&](uint32_t j) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 3; ++k) px[k] = a.ps[(size_t)(CX + k) * cap + j];
#pragma unroll
        for (int k = 0; k < 12; ++k) A[k] = aff[(size_t)k * cap + j];
        mass = a.ps[(size_t)CMASS * cap + j];
    };
    // The ranges of the wave's tile; their particles.
    auto ranges = [&](const SceneDev& sc, const int* tc) __attribute__((always_inline)) {
        const int W = int(sc.W);
        uint32_t b = 0u, e = 0u;
        if (lane < 9) {
            const int ny = tc[1] + lane % 3 - 1, nz = tc[2] + lane / 3 - 1;
            if (ny >= 0 && nz >= 0 && ny < W && nz < W) {
                const uint32_t row = sc.tile_base + uint32_t(W * (ny + W * nz));
                b = lb[row + uint32_t(max(tc[0] - 1, 0))];
                e = lb[row + uint32_t(min(tc[0] + 1, W - 1)) + 1u];
            }
        }
        const uint32_t incl = wave_incl_scan(e - b);
        if (lane < 9) {
            rbeg[wave][lane] = b;
            roff[wave][lane + 1] = incl;
        }
        if (lane == 0) roff[wave][0] = 0u;
        __builtin_amdgcn_wave_barrier();
        return (uint32_t)__shfl(int(incl), 63, 64);
    };
    // The wave's tile; false: it needs the block.
    auto by_wave = [&](const SceneDev& sc, const int* tc, uint32_t t, uint32_t total) __attribute__((always_inline)) {
        if (total > uint32_t(GATHER_LIST / GATHER_WAVES)) return false;
        uint32_t* own = slots + wave * (GATHER_LIST / GATHER_WAVES);
        uint32_t held = 0u;
        for (uint32_t c0 = 0; c0 < total && held <= uint32_t(GATHER_WAVE_RECS); c0 += 64u * GATHER_PER) {
            uint32_t slot[GATHER_PER];
            bool hit[GATHER_PER];
#pragma unroll
            for (int u = 0; u < GATHER_PER; ++u) {
                const uint32_t j = c0 + uint32_t(64 * u + lane);
                hit[u] = j < total;
                slot[u] = hit[u] ? candidate(wave, j) : 0u;
            }
#pragma unroll
            for (int u = 0; u < GATHER_PER; ++u) {
                if (hit[u]) hit[u] = reaches(sc, tc, slot[u]);
                const uint64_t m = __ballot(hit[u]);
                if (hit[u]) own[held + uint32_t(__popcll(m & lt))] = slot[u];
                held += uint32_t(__popcll(m));
            }
        }
        if (held > uint32_t(GATHER_WAVE_RECS)) return false;
        if (held == 0u) {
            a.gmp[(size_t)(t << 6) | uint32_t(lane)] = make_float4(0.f, 0.f, 0.f, 0.f);
        } else {
            __builtin_amdgcn_wave_barrier();
            uint32_t rm = 0u;
            if (uint32_t(lane) < held) {
                load(own[lane]);
                rm = gather_record(sc, tc, px, A, mass, rec[wave * GATHER_WAVE_RECS + lane]);
            }
            // four rows in flight; a row's list is one step
#pragma unroll 1
            for (int cz = 0; cz < 4; ++cz) {
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int cy = 0; cy < 4; ++cy) {
                    uint16_t* wl = wlist[wave] + 2 * GATHER_STEP * cy;
                    const bool on = (rm >> (4 * cz + cy)) & 1u;
                    const uint64_t m = __ballot(on);
                    if (on) wl[__popcll(m & lt)] = uint16_t(wave * GATHER_WAVE_RECS + lane);
                    if (lane < GATHER_STEP) wl[__popcll(m) + lane] = uint16_t(GATHER_RECS);
                }
                __builtin_amdgcn_wave_barrier();
                float acc[4][4];
#pragma unroll
                for (int cy = 0; cy < 4; ++cy)
#pragma unroll
                    for (int c2 = 0; c2 < 4; ++c2) acc[cy][c2] = 0.f;
#pragma unroll 1
                for (uint32_t g = 0; g < held; g += 16u)
#pragma unroll
                    for (int cy = 0; cy < 4; ++cy)
                        gather_add(rec[wlist[wave][2 * GATHER_STEP * cy + g + (lane >> 2)]], cy, cz, sc.dx, acc[cy]);
#pragma unroll
                for (int cy = 0; cy < 4; ++cy) gather_store(sc, tc, t, cy, cz, acc[cy], a.gmp);
            }
        }
        if (lane == 0) a.tile_flag[t] |= FLAG_GMP;
        return true;
    };
    // A tile by the whole block, with the ranges that wave w has found.
    auto by_block = [&](const SceneDev& sc, const int* tc, uint32_t t, int w) __attribute__((always_inline)) {
        const int cy = wave & 3, cz = wave >> 2;  // the wave's row
        const uint32_t total = roff[w][9];
        float acc[4] = {0.f, 0.f, 0.f, 0.f};
        uint32_t held = 0u;  // slots in the list (block-uniform)
        for (uint32_t c0 = 0; c0 < total; c0 += GATHER_THREADS * GATHER_PER) {
            uint32_t slot[GATHER_PER];
            bool hit[GATHER_PER];
#pragma unroll
            for (int u = 0; u < GATHER_PER; ++u) {
                const uint32_t j = c0 + uint32_t(u * GATHER_THREADS + tid);
                hit[u] = j < total;
                slot[u] = hit[u] ? candidate(w, j) : 0u;
            }
            uint64_t m[GATHER_PER];
#pragma unroll
            for (int u = 0; u < GATHER_PER; ++u) {
                if (hit[u]) hit[u] = reaches(sc, tc, slot[u]);
                m[u] = __ballot(hit[u]);
                if (lane == 0) wcnt[u * GATHER_WAVES + wave] = uint32_t(__popcll(m[u]));
            }
            __syncthreads();
            // places after the slots held: candidates ascend over (u, wave, lane)
            const uint32_t c = lane < GATHER_PER * GATHER_WAVES ? wcnt[lane] : 0u, incl = wave_incl_scan(c);
#pragma unroll
            for (int u = 0; u < GATHER_PER; ++u) {
                const uint32_t at = held + (uint32_t)__shfl(int(incl - c), u * GATHER_WAVES + wave, 64);
                if (hit[u]) slots[at + uint32_t(__popcll(m[u] & lt))] = slot[u];
            }
            held += (uint32_t)__shfl(int(incl), 63, 64);
            __syncthreads();
            // sum the list when another round might not fit, and at the end
            const bool last = c0 + GATHER_THREADS * GATHER_PER >= total;
            if (!last && held + GATHER_THREADS * GATHER_PER <= GATHER_LIST) continue;
            // a batch's loads are issued before the sums of the batch before it
            if (tid < GATHER_RECS && uint32_t(tid) < held) load(slots[tid]);
            for (uint32_t b0 = 0; b0 < held; b0 += GATHER_RECS) {
                const uint32_t cnt = min(held - b0, uint32_t(GATHER_RECS));
                if (tid < GATHER_RECS)
                    rows[tid] = uint16_t(uint32_t(tid) < cnt ? gather_record(sc, tc, px, A, mass, rec[tid]) : 0u);
                __syncthreads();
                if (tid < GATHER_RECS && b0 + GATHER_RECS + uint32_t(tid) < held)
                    load(slots[b0 + GATHER_RECS + uint32_t(tid)]);
                // the wave's own list: records reaching its row, in order,
                // filled up to a whole step with the record that adds nothing
                uint32_t len = 0u;
                for (uint32_t g = 0; g < cnt; g += 64) {
                    const bool on = (rows[g + uint32_t(lane)] >> wave) & 1u;
                    const uint64_t mm = __ballot(on);
                    if (on) wlist[wave][len + uint32_t(__popcll(mm & lt))] = uint16_t(g + lane);
                    len += uint32_t(__popcll(mm));
                }
                if (lane < GATHER_STEP) wlist[wave][len + uint32_t(lane)] = uint16_t(GATHER_RECS);
                __builtin_amdgcn_wave_barrier();
                for (uint32_t g = 0; g < len; g += GATHER_STEP)
#pragma unroll
                    for (int f = 0; f < GATHER_FLY; ++f)
                        gather_add(rec[wlist[wave][g + uint32_t(16 * f + (lane >> 2))]], cy, cz, sc.dx, acc);
                __syncthreads();
            }
            held = 0u;
        }
        gather_store(sc, tc, t, cy, cz, acc, a.gmp);
        if (tid == 0) a.tile_flag[t] |= FLAG_GMP;
    };
    SceneDev sc;
    int tc[3];
    if (n <= thin && n <= gridDim.x) {  // the whole block takes a tile; each wave finds its ranges
        if (blockIdx.x >= n) return;
        const uint32_t t = list[blockIdx.x];
        tile(t, tile_scene[t], sc, tc);
        ranges(sc, tc);
        by_block(sc, tc, t, wave);
        return;
    }
    // a tile per wave first, on so many blocks that their waves have work
    const uint32_t nb = n > thin ? min(gridDim.x, max(n / uint32_t(GATHER_WAVES), uint32_t(GATHER_BLOCKS))) : gridDim.x;
    if (blockIdx.x >= nb) return;
    uint32_t scene = ~0u;  // whose record sc is
    for (uint32_t i0 = blockIdx.x; i0 < n; i0 += nb * GATHER_WAVES) {
        const uint32_t i = i0 + nb * uint32_t(wave);
        uint4 left = make_uint4(~0u, 0u, 0u, 0u);
        if (i < n) {
            const uint32_t t = list[i];
            scene = tile_scene[t];
            tile(t, scene, sc, tc);
            const uint32_t total = ranges(sc, tc);
            if (n <= thin || !by_wave(sc, tc, t, total))
                left = make_uint4(t, scene, uint32_t(tc[0]) | uint32_t(tc[1]) << 16, uint32_t(tc[2]));
        }
        if (lane == 0) whole[wave] = left;
        __syncthreads();
        const int held = int(min((n - i0 + nb - 1u) / nb, uint32_t(GATHER_WAVES)));  // waves with a tile
        for (int w = 0; w < held; ++w) {
            const uint4 q = whole[w];
            const uint32_t t = uint32_t(__builtin_amdgcn_readfirstlane(int(q.x)));
            if (t == ~0u) continue;
            const uint32_t its = uint32_t(__builtin_amdgcn_readfirstlane(int(q.y)));
            const uint32_t xy = uint32_t(__builtin_amdgcn_readfirstlane(int(q.z)));
            if (its != scene) sc = const_load(a.scenes + its);
            scene = its;
            tc[0] = int(xy & 0xffffu);
            tc[1] = int(xy >> 16);
            tc[2] = __builtin_amdgcn_readfirstlane(int(q.w));
            by_block(sc, tc, t, w);
        }
        __syncthreads();  // the ranges and the marks are the next tiles'
    }
}

hipError_t launch_gather_p2g(const StepArgs& a, const uint32_t* tile_scene, const uint32_t* tile_lb,
                             const float* affine, const uint32_t* slist, const uint32_t* scount,
                             uint32_t total_tiles, uint32_t n, hipStream_t s) {
    const unsigned blocks = std::min(total_tiles, uint32_t(GATHER_GRID));
    hipLaunchKernelGGL(k_gather_p2g, dim3(blocks), dim3(GATHER_THREADS), 0, s, a, tile_scene, tile_lb, affine, slist,
                       scount, std::max(n / GATHER_THIN, 2u * GATHER_BLOCKS));
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Sparse tile pool (MpmSimulation::new_sparse, mpm.rs:848-853; tile marking
// mpm_active_tiles.wgsl:79-130).  Every substep the particles that scatter
// mark the tiles within one cell of their stencils (block_scatter, from its
// LDS box; deferred particles directly), legacy rigid spheres mark the tiles
// their shell can reach, and one pass over the tile table gives the marked
// tiles the pool's slots, in arrival order, and clears the marks.  A demand
// above the capacity latches FAULT_OVERFLOW: every later kernel of the
// substep sees the latch and leaves the particles as they were.
__global__ __launch_bounds__(256) void k_pool_compact(uint32_t* __restrict__ tile_mark, uint32_t total,
                                                      uint32_t* __restrict__ tile_slot,
                                                      uint32_t* __restrict__ slot_tile, uint32_t capacity,
                                                      uint32_t* __restrict__ status) {
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < total; t += gridDim.x * blockDim.x) {
        uint32_t s1 = 0u;
        if (tile_mark[t]) {
            tile_mark[t] = 0u;
            const uint32_t slot = atomicAdd(&status[ST_POOL], 1u);
            if (slot < capacity) {
                s1 = slot + 1u;
                slot_tile[slot] = t;
            } else {
                latch(status, FAULT_OVERFLOW);
            }
        }
        tile_slot[t] = s1;
    }
}

hipError_t launch_pool_compact(uint32_t* tile_mark, uint32_t total_tiles, uint32_t* tile_slot, uint32_t* slot_tile,
                               uint32_t capacity, uint32_t* status, hipStream_t s) {
    const unsigned blocks = std::max(1u, std::min<unsigned>((total_tiles + 255) / 256, 16384u));
    hipLaunchKernelGGL(k_pool_compact, dim3(blocks), dim3(256), 0, s, tile_mark, total_tiles, tile_slot, slot_tile,
                       capacity, status);
    return hipGetLastError();
}

// One block per legacy sphere: the tiles of its cells within radius + 2 cells
// (mark_rigids, mpm_active_tiles.wgsl:108-124).  A sphere whose tile range
// alone exceeds the pool latches the overflow without marking.
__global__ __launch_bounds__(256) void k_mark_spheres(const SceneDev* __restrict__ scenes, RigidDev rg,
                                                      uint32_t* __restrict__ tile_mark, uint32_t capacity,
                                                      uint32_t* __restrict__ status) {
    const float4* b = rg.body + RIGID_ROWS * blockIdx.x;
    if (b[4].w != 0.0f) return;  // prescribed solids mark nothing
    const SceneDev& sc = scenes[0];
    int lo[3], n[3];
    const float c[3] = {b[0].x, b[0].y, b[0].z};
    const float extent = fmaxf(b[0].w, 0.0f) * sc.inv_dx + 2.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float ck = (c[k] - sc.origin[k]) * sc.inv_dx;
        const int l = max(int(floorf(ck - extent)) - sc.window[k], 0);
        const int h = min(int(ceilf(ck + extent)) - sc.window[k], int(sc.G) - 1);
        if (l > h) return;
        lo[k] = l >> 2;
        n[k] = (h >> 2) - lo[k] + 1;
    }
    const uint64_t count = (uint64_t)n[0] * n[1] * n[2];
    if (count > capacity) {
        if (threadIdx.x == 0) latch(status, FAULT_OVERFLOW);
        return;
    }
    for (uint32_t i = threadIdx.x; i < count; i += blockDim.x) {
        const uint32_t x = i % n[0], y = (i / n[0]) % n[1], z = i / (n[0] * n[1]);
        tile_mark[sc.tile_base + uint32_t(lo[0]) + x + sc.W * (uint32_t(lo[1]) + y + sc.W * (uint32_t(lo[2]) + z))] = 1u;
    }
}

hipError_t launch_mark_spheres(const SceneDev* scenes, const RigidDev& rg, uint32_t* tile_mark, uint32_t capacity,
                               uint32_t* status, hipStream_t s) {
    if (rg.count == 0) return hipSuccess;
    hipLaunchKernelGGL(k_mark_spheres, dim3(rg.count), dim3(256), 0, s, scenes, rg, tile_mark, capacity, status);
    return hipGetLastError();
}

// The global-atomic P2G of the particles a sparse pool deferred (escaped
// stencils, chunks that could not reduce in LDS, the global-atomic mode):
// the P2G pass's particle math (stress from the FP64 SVD of F,
// mpm.wgsl:532-599) once the compaction has given their tiles slots.  Sparse
// pools hold one scene of the shader model.
__global__ __launch_bounds__(256) void k_deferred_p2g(StepArgs a) {
    if (a.status[ST_FAULT] != 0u) return;
    const uint32_t n = a.status[ST_DEFER], cap = a.cap;
    const float* ps = a.ps;
    const SceneDev sc = const_load(a.scenes);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t slot = a.defer_list[i], boff = 4u * slot;
        float x[3], v[3], C[9], F[9];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            x[k] = plane_ld(ps, cap, CX + k, boff);
            v[k] = plane_ld(ps, cap, CV + k, boff);
        }
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            C[k] = plane_ld(ps, cap, CC + k, boff);
            F[k] = plane_ld(ps, cap, CF + k, boff);
        }
        const float jp = plane_ld(ps, cap, CJP, boff), m = plane_ld(ps, cap, CMASS, boff),
                    vol = plane_ld(ps, cap, CVOL, boff);
        const float* mrow = mat_row(a, sc, __float_as_uint(plane_ld(ps, cap, CMAT, boff)));
        float mu = sc.mu, lam = sc.lam;
        if (a.has_E) {
            const float E = plane_ld(ps, cap, CE, boff);
            mu = E / (2.0f * (1.0f + sc.poisson));
            lam = E * sc.poisson / ((1.0f + sc.poisson) * (1.0f - 2.0f * sc.poisson));
        }
        Scatter sp;
        Svd32 d;
        svd3<MODEL_SHADER>(F, d);
        affine_from_svd<MODEL_SHADER>(sc, mrow, d, mu, lam, jp, a.dt, vol, m, C, sp.A);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float xp = (x[k] - sc.origin[k]) * sc.inv_dx;
            const float bf = floorf(xp - 0.5f);
            sp.b[k] = int(bf) - sc.window[k];
            sp.fx[k] = xp - bf;
            sp.mv[k] = m * v[k];
        }
        sp.m = m;
        sp.on = true;
        sp.esc = true;
        sp.slot = slot;
        scatter_global(a, sc, sp);
    }
}

hipError_t launch_deferred_p2g(const StepArgs& a, int model, hipStream_t s) {
    if (model != MODEL_SHADER) return hipErrorInvalidValue;
    // the fused mode defers the few particles that escaped or whose chunk fell
    // back; the global-atomic mode all of them
    const unsigned blocks = std::max(1u, std::min<unsigned>((a.cap + 255) / 256, a.use_lds ? 512u : 4096u));
    hipLaunchKernelGGL(k_deferred_p2g, dim3(blocks), dim3(256), 0, s, a);
    return hipGetLastError();
}

__global__ void k_storage_layout(const float4* __restrict__ gmp, uint32_t cells, float* __restrict__ mass,
                                 float* __restrict__ mom) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < cells; i += gridDim.x * blockDim.x) {
        const float4 q = gmp[i];
        mass[i] = q.x;
        mom[3 * (size_t)i] = q.y;
        mom[3 * (size_t)i + 1] = q.z;
        mom[3 * (size_t)i + 2] = q.w;
    }
}

hipError_t launch_storage_to_host_layout(const float4* gmp, uint32_t cells, float* mass, float* mom, hipStream_t s) {
    const unsigned blocks = std::max(1u, std::min<unsigned>((cells + 255) / 256, 8192u));
    hipLaunchKernelGGL(k_storage_layout, dim3(blocks), dim3(256), 0, s, gmp, cells, mass, mom);
    return hipGetLastError();
}

}  // namespace mpm
