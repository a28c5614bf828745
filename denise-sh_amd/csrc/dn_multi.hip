// Several time steps per launch for grids that leave most of the chip
// idle (gfx950).  Same arithmetic, in the same order and rounding, as the
// tile step (dn_tile.hip); compiled with -ffp-contract=off.
//
// One workgroup owns 24 x 8 cells of one shot and holds the cells around them
// that T steps reach (T (2K-1) on every side) as well.  A thread keeps the
// fields, coefficients and CPML variables of its cells in registers; vy, sxy
// and syz are exchanged through LDS, two barriers per step; the region that
// is still right shrinks by 2K-1 cells per step and ends on the owned cells.
//
// What bounds it: latency.  A launch of the tile step lasts 3.9 us on a
// small grid (batch slot 0.85, fields 1.2, the two updates 1.4, the rest
// barriers and stores) and the next follows 1.4 us later; a step in here is
// two updates from LDS, so T of them share one load, one store and one
// launch.  The price is work: 1536 cells for 192 owned ones in the first step
// of FDORDER 4, so the rule (multi_limit in dn_core.cpp, with both sides'
// times) stops where that fills the chip.  400 x 120, one shot, microseconds
// per step, tiles -> several steps: FDORDER 4 forward 5.5 -> 2.5, gradient
// 6.6 -> 3.2; FDORDER 8 with L 2 6.0 -> 4.4, 6.9 -> 5.4.
// Shape (the same forward / gradient of FDORDER 4, whole calls of 2000 / 1500
// steps, ms): 24 x 8 cells and 4 steps 4.73 / 8.73; 32 x 8 and 3, 4, 5, 6
// steps 5.40 / 9.90, 4.95 / 9.32, 5.21 / 11.8, 4.99 / 9.26; 20 x 10 4.83 /
// 8.93; 16 x 16 5.02 / 9.46.  Steps of other orders: FDORDER 2 with 4, 6, 8
// 1.64, 1.46, 1.57 us per step; FDORDER 6 with 2, 3 3.44, 3.29.  The CPML
// profiles lie in LDS, not in registers, and the elastic kernels of FDORDER 2
// and 4 are held to 80 registers: two workgroups share a CU (500 x 160: 4.09
// -> 3.22 us per step, gradient 5.31 -> 4.86).  At that limit the storing one
// of FDORDER 4 spills one vector register (8 bytes) and 40 scalar ones into
// lanes of vector registers; the correlating one spilled 23 (+12 % at 400 x
// 120) and is not held to it.
//
// Everything the cells around the tile read is double-buffered (here also the
// stress CPML memory and the relaxation variables, which the single steps
// update in place).
#include "dn_internal.h"

#pragma clang fp contract(off)

#ifndef DN_MULTI_K
#error "compile with -DDN_MULTI_K=<FDORDER / 2>"
#endif

namespace dn {

namespace {

constexpr int kMThreads = 768;

// EX: launches that store FP32 snapshots or sum the pseudo-Hessian (forward),
// or correlate with FP32 snapshots (adjoint), in some of their steps
template <int K, int L, bool ADJ, bool EX>
__global__ __launch_bounds__(kMThreads, L == 0 && K <= 2 && !(ADJ && EX) ? 6 : 3) void k_multi(const StepArgs a)
{
    constexpr int T = multi_steps(K), H = 2 * K - 1, M = T * H, kMX = kMultiX, kMY = kMultiY;
    constexpr int LD = L > 0 ? L : 1;
    constexpr int W = kMX + 2 * M, HT = kMY + 2 * M, N = W * HT, NC = (N + kMThreads - 1) / kMThreads;
    __shared__ float lv[N], lx[N], lz[N];
    __shared__ float lkx[6 * W], lky[6 * HT];   // CPML K, a, b of the velocity, then of the stress
    const int w_ = blockIdx.x, lin = (w_ & 7) * a.tl_nblk8 + (w_ >> 3);
    if (lin >= a.tl_nblk) return;
    const int tile = lin / a.nshots, s = lin - tile * a.nshots;
    const int bx = tile / a.tl_ny, by = tile - bx * a.tl_ny;
    const Geo &g = a.g;
    const ShotSlot sl = a.slots[s];
    const int nt0 = *a.nt_base + a.nt;
    const int S = sl.shot, NTs = sl.nt;
    if (S < 0 || S >= a.nshots_all || nt0 > NTs) {
        if (S < 0 || S >= a.nshots_all) a.status[2] = 1;
        return;
    }
    const int steps = min(a.ms_steps, NTs - nt0 + 1);   // a record may end inside the launch
    const int c0 = 1 + bx * kMX, j0 = 1 + by * kMY;
    const int fw = g.fw, fw2 = 2 * g.fw, pn = fw2 + 1;
    const int nxny = g.nx * g.ny;
    const long long s0 = s;
    const float *__restrict__ vyi = a.vy_in + s0 * g.plane;
    const float *__restrict__ sxi = a.sxy_in + s0 * g.plane;
    const float *__restrict__ szi = a.syz_in + s0 * g.plane;
    const float *__restrict__ rqi = L > 0 ? a.rq_in + s0 * 2 * L * g.plane : nullptr;
    const float *__restrict__ pmlb = a.pml.Kx;
    const float *__restrict__ pxi = a.psx_in + s0 * g.ny * fw2, *__restrict__ pyi = a.psy_in + s0 * fw2 * g.nx;
    const float *__restrict__ wxi = a.pvx_in + s0 * g.ny * fw2, *__restrict__ wyi = a.pvy_in + s0 * fw2 * g.nx;

    // ---- the thread's cells ----
    int cr[NC], cq[NC], cj[NC], cw[NC];   // row and column in the workgroup's region, grid row, wrapped column
    bool in[NC], own[NC];
    float v[NC], sx[NC], sz[NC], b[NC], u1[NC], u2[NC];
    float rr[NC][LD], qq[NC][LD], dp[NC][LD], dd[NC][LD];   // relaxation variables and their coefficients
    unsigned off[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int e = min((int)threadIdx.x + i * kMThreads, N - 1);
        cr[i] = e / W;
        cq[i] = e - cr[i] * W;
        cj[i] = j0 - M + cr[i];
        const int c = c0 - M + cq[i];
        cw[i] = !g.periodic ? c : (c < 1 ? c + g.nx : (c > g.nx ? c - g.nx : c));
        in[i] = (int)threadIdx.x + i * kMThreads < N && cj[i] >= 1 && cj[i] <= g.ny && (g.periodic || (c >= 1 && c <= g.nx));
        own[i] = in[i] && cr[i] >= M && cr[i] < M + kMY && cq[i] >= M && cq[i] < M + kMX && c <= g.nx;
        // cells outside the grid read an edge cell, unused
        const int jj = min(max(cj[i], 1), g.ny), cc = min(max(cw[i], 1), g.nx);
        off[i] = (unsigned)((jj - 1 + g.yoff) * g.pitch + (cc - 1 + g.xoff));
        v[i] = vyi[off[i]];
        sx[i] = sxi[off[i]];
        sz[i] = szi[off[i]];
        b[i] = a.bfield[off[i]];
        if (L == 0) {
            const float2 u = *(const float2 *)(a.spk + 2 * (size_t)off[i]);
            u1[i] = u.x;
            u2[i] = u.y;
        } else {
            const float4 u = *(const float4 *)(a.spk + 4 * (size_t)off[i]);
            u1[i] = u.x;
            u2[i] = u.y;
            dp[i][0] = u.z;
            dd[i][0] = u.w;
#pragma unroll
            for (int l = 1; l < L; ++l) {
                const float2 w = *(const float2 *)(a.spk + (2 + 2 * l) * g.plane + 2 * (size_t)off[i]);
                dp[i][l] = w.x;
                dd[i][l] = w.y;
            }
#pragma unroll
            for (int l = 0; l + 1 < L; l += 2) {
                const float4 w = *(const float4 *)(rqi + 2 * l * g.plane + 4 * (size_t)off[i]);
                rr[i][l] = w.x;
                qq[i][l] = w.y;
                rr[i][l + 1] = w.z;
                qq[i][l + 1] = w.w;
            }
            if (L & 1) {
                const float2 w = *(const float2 *)(rqi + 2 * (L - 1) * g.plane + 2 * (size_t)off[i]);
                rr[i][L - 1] = w.x;
                qq[i][L - 1] = w.y;
            }
        }
    }
    // CPML variables and profiles, in workgroups that reach into an absorbing
    // region (uniform)
    const bool tpx = fw > 0 && !g.periodic && (c0 - M <= fw || c0 + kMX - 1 + M >= g.nx - fw + 1);
    const bool tpy = fw > 0 && ((!g.free_surf && j0 - M <= fw) || j0 + kMY - 1 + M >= g.ny - fw + 1);
    int xk[NC], yk[NC];
    float px[NC], py[NC], wx[NC], wy[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        xk[i] = yk[i] = 0;
        if (tpx && in[i]) xk[i] = cw[i] <= fw ? cw[i] : (cw[i] >= g.nx - fw + 1 ? cw[i] - g.nx + fw2 : 0);
        if (tpy && in[i])
            yk[i] = (!g.free_surf && cj[i] <= fw) ? cj[i] : (cj[i] >= g.ny - fw + 1 ? cj[i] - g.ny + fw2 : 0);
        if (xk[i] > 0) {
            const int o = (cj[i] - 1) * fw2 + (xk[i] - 1);
            px[i] = pxi[o];
            wx[i] = wxi[o];
        }
        if (yk[i] > 0) {
            const int o = (yk[i] - 1) * g.nx + (cw[i] - 1);
            py[i] = pyi[o];
            wy[i] = wyi[o];
        }
    }
    if (tpx) {
        for (int e = threadIdx.x; e < 6 * W; e += kMThreads) {
            const int f = e / W, c = c0 - M + (e - f * W);
            lkx[e] = pmlb[f * pn + min(max(c <= fw ? c : c - g.nx + fw2, 0), fw2)];
        }
    }
    if (tpy) {
        for (int e = threadIdx.x; e < 6 * HT; e += kMThreads) {
            const int f = e / HT, j = j0 - M + (e - f * HT);
            // no top frame under a free surface: its rows may be the bottom frame's (NY < 2 FW)
            const bool top = !g.free_surf && j <= fw;
            // Q2: the viscoelastic stress uses the full-grid y profile on top
            const int fp = (L > 0 && f >= 3 && top) ? f + 3 : f + 6;
            lky[e] = pmlb[fp * pn + min(max(top ? j : j - g.ny + fw2, 0), fw2)];
        }
    }
    // the gradient sums of the owned cells stay in registers over the steps
    float *__restrict__ grb = EX ? a.grad_rho + s0 * nxny : nullptr;
    float *__restrict__ gub = EX ? a.grad_u + s0 * nxny : nullptr;
    float *__restrict__ wab = EX ? a.wacc + s0 * nxny : nullptr;
    const bool sums = EX && (ADJ || a.hess);
    const bool energy = EX && (ADJ || a.store_mode != 0);
    float gr[NC], gu[NC], wa[NC], f0[NC], fy[NC], fu[NC];
    unsigned ci[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        ci[i] = own[i] ? (unsigned)((cj[i] - 1) * g.nx + (cw[i] - 1)) : 0u;
        if (sums) {
            gr[i] = grb[ci[i]];
            gu[i] = gub[ci[i]];
        }
        if (energy) wa[i] = wab[ci[i]];
    }
    // adjoint: the snapshot that step nt correlates with, loaded a step ahead
    auto corr_slot = [&](int nt) -> int {
        const int sf = NTs - nt + 1;
        return (EX && ADJ && sf >= 1 && (sf - 1) % a.dtinv == 0) ? (sf - 1) / a.dtinv : -1;
    };
    auto snap_load = [&](int slot) {
        const float *__restrict__ sn = a.snap + s0 * a.snap_shot_stride + (long long)slot * 3 * nxny;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            f0[i] = sn[ci[i]];
            fy[i] = sn[nxny + ci[i]];
            fu[i] = sn[2 * nxny + ci[i]];
        }
    };
    int slot = corr_slot(nt0);
    if (slot >= 0) snap_load(slot);
    // sources near the tile (uniform); the first one's samples of the launch
    const int sb = sl.src0, se = ADJ ? sl.src0 : sl.src1;
    auto near = [&](int si, int sj) -> bool {
        return sj >= j0 - M && sj < j0 + kMY + M && (g.periodic || (si >= c0 - M && si < c0 + kMX + M));
    };
    bool has_src = false;
    float sig[T];
#pragma unroll
    for (int t = 0; t < T; ++t) sig[t] = 0.0f;
    if (!ADJ && se > sb) {
        has_src = near(sl.si, sl.sj);
        if (has_src) {
#pragma unroll
            for (int t = 0; t < T; ++t) sig[t] = a.src_sig[(long long)sb * a.nt_max + min(nt0 - 1 + t, a.nt_max - 1)];
        }
        for (int l = sb + 1; l < se; ++l) has_src = has_src || near(a.src_i[l], a.src_j[l]);
    }
    // receivers of the cells and, in the adjoint, their residuals of the launch
    int ri[NC];
    float res[NC][T];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        ri[i] = -1;
        if (in[i]) {
            const int row = a.rec_row[cj[i]];
            if (row >= 0) ri[i] = a.rec_tab[row + cw[i]];
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            res[i][t] = 0.0f;
            if (ADJ && ri[i] >= 0) res[i][t] = a.resid[(s0 * a.ntr + ri[i]) * a.nt_max + min(nt0 - 1 + t, a.nt_max - 1)];
        }
    }
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int e = threadIdx.x + i * kMThreads;
        if (!in[i]) v[i] = sx[i] = sz[i] = 0.0f;
        if (e < N) {
            lv[e] = v[i];
            lx[e] = sx[i];
            lz[e] = sz[i];
        }
    }

    auto cpml = [](float kk, float ka, float kb, float &p, float &d) {
        p = kb * p + ka * d;
        d = d / kk + p;
    };
    // ---- the steps ----
#pragma unroll 1
    for (int t = 0; t < steps; ++t) {
        const int nt = nt0 + t;
        const bool onstep = ((nt - 1) % a.dtinv) == 0;
        const bool fstore = EX && !ADJ && a.store_mode != 0 && onstep;
        // hessian.c:91: stored steps 1..NTDTINV-1 of this shot
        const bool hsum = EX && !ADJ && a.hess && onstep && (nt - 1) / a.dtinv < (NTs + a.dtinv - 1) / a.dtinv - 1;
        const bool corr = slot >= 0;
        float *__restrict__ snw =
            fstore ? a.snap + s0 * a.snap_shot_stride + (long long)((nt - 1) / a.dtinv) * 3 * nxny : nullptr;
        __syncthreads();
        const int lo = t * H + K, hi = t * H + K - 1;   // new vy: cells lo .. size - hi - 1
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            if (!(in[i] && cr[i] >= lo && cr[i] < HT - hi && cq[i] >= lo && cq[i] < W - hi)) continue;
            const int e = threadIdx.x + i * kMThreads;
            float gx = a.hc[1] * (sx[i] - lx[e - 1]);
            float gy = a.hc[1] * (sz[i] - lz[e - W]);
#pragma unroll
            for (int m = 2; m <= K; ++m) {
                gx = gx + a.hc[m] * (lx[e + m - 1] - lx[e - m]);
                gy = gy + a.hc[m] * (lz[e + (m - 1) * W] - lz[e - m * W]);
            }
            if (xk[i] > 0) cpml(lkx[cq[i]], lkx[W + cq[i]], lkx[2 * W + cq[i]], px[i], gx);
            if (yk[i] > 0) cpml(lky[cr[i]], lky[HT + cr[i]], lky[2 * HT + cr[i]], py[i], gy);
            const float tsum = gx + gy, vold = v[i];
            if (EX && !ADJ && own[i] && (hsum || fstore)) {
                const float acc = (b[i] * tsum) / a.DH;   // vyp1, update_v_PML.c:184
                if (hsum) gr[i] = gr[i] + (acc * acc);
                if (fstore) snw[ci[i]] = acc;
            }
            // vyp1 = old vy (update_v_PML.c:189); denise.c:1589
            if (EX && ADJ && corr) gr[i] = gr[i] + (vold * f0[i]);
            float vn = vold + ((b[i] * a.DT) * tsum) / a.DH;
            if (!ADJ) {
                if (has_src) {
                    if (sl.sj == cj[i] && sl.si == cw[i]) vn = vn + sig[0];
                    for (int l = sb + 1; l < se; ++l)
                        if (a.src_j[l] == cj[i] && a.src_i[l] == cw[i])
                            vn = vn + a.src_sig[(long long)l * a.nt_max + (nt - 1)];
                }
            } else if (ri[i] >= 0) {
                vn = vn + res[i][0];
            }
            v[i] = vn;
            lv[e] = vn;
            if (own[i]) {
                if (!ADJ && a.seis != nullptr && ri[i] >= 0) a.seis[(s0 * a.ntr + ri[i]) * a.nt_max + (nt - 1)] = vn;
                // instability latch at the reference's probe cell
                if (cj[i] == (g.ny >> 1) && cw[i] == (g.nx >> 1) && !(vn == vn))
                    if (atomicCAS(&a.status[0], 0, nt) == 0) a.status[1] = S + 1;
            }
        }
#pragma unroll
        for (int k = 0; k + 1 < T; ++k) {
            sig[k] = sig[k + 1];
#pragma unroll
            for (int i = 0; i < NC; ++i) res[i][k] = res[i][k + 1];
        }
        __syncthreads();
        const int ms = (t + 1) * H;                     // stress: cells ms .. size - ms - 1
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            if (!(in[i] && cr[i] >= ms && cr[i] < HT - ms && cq[i] >= ms && cq[i] < W - ms)) continue;
            const int e = threadIdx.x + i * kMThreads;
            float vyx = a.hc[1] * (lv[e + 1] - v[i]);
            float vyy = a.hc[1] * (lv[e + W] - v[i]);
#pragma unroll
            for (int m = 2; m <= K; ++m) {
                vyx = vyx + a.hc[m] * (lv[e + m] - lv[e - m + 1]);
                vyy = vyy + a.hc[m] * (lv[e + m * W] - lv[e - (m - 1) * W]);
            }
            vyx = vyx * a.dhi;
            vyy = vyy * a.dhi;
            if (xk[i] > 0) cpml(lkx[3 * W + cq[i]], lkx[4 * W + cq[i]], lkx[5 * W + cq[i]], wx[i], vyx);
            if (yk[i] > 0) cpml(lky[3 * HT + cr[i]], lky[4 * HT + cr[i]], lky[5 * HT + cr[i]], wy[i], vyy);
            if (L == 0) {
                sx[i] = sx[i] + u1[i] * vyx;
                sz[i] = sz[i] + u2[i] * vyy;
            } else {
                float sumr = 0.0f, sumq = 0.0f;
#pragma unroll
                for (int l = 0; l < L; ++l) {
                    sumr += rr[i][l];
                    sumq += qq[i][l];
                }
                sx[i] = sx[i] + ((u1[i] * vyx) + (a.dthalbe * sumr));
                sz[i] = sz[i] + ((u2[i] * vyy) + (a.dthalbe * sumq));
                sumr = 0.0f;
                sumq = 0.0f;
#pragma unroll
                for (int l = 0; l < L; ++l) {
                    rr[i][l] = a.bip[l] * (rr[i][l] * a.cip[l] - (dp[i][l] * vyx));
                    qq[i][l] = a.bjm[l] * (qq[i][l] * a.cjm[l] - (dd[i][l] * vyy));
                    sumr += rr[i][l];
                    sumq += qq[i][l];
                }
                sx[i] = sx[i] + (a.dthalbe * sumr);
                sz[i] = sz[i] + (a.dthalbe * sumq);
            }
            lx[e] = sx[i];
            lz[e] = sz[i];
            if (EX && own[i]) {
                if (fstore) {
                    snw[nxny + ci[i]] = vyy;        // uy  (forward_prop_y)
                    snw[2 * nxny + ci[i]] = vyx;    // uyx (forward_prop_u)
                    wa[i] = wa[i] + v[i] * v[i];    // eprecond.c:11
                }
                if (hsum) {
                    const float eyx = 0.5f * vyx;   // hess_save.c:13 (exact in float)
                    gu[i] = gu[i] + ((vyy * vyy) + (eyx * eyx));
                }
                if (ADJ && corr) {
                    gu[i] = gu[i] + ((fu[i] * sx[i]) + (fy[i] * sz[i]));   // denise.c:1609
                    wa[i] = wa[i] + v[i] * v[i];
                }
            }
        }
        if (EX && ADJ) {
            slot = corr_slot(nt + 1);
            if (slot >= 0 && t + 1 < steps) snap_load(slot);
        }
    }

    // ---- the owned cells back ----
    float *__restrict__ vyo = a.vy_out + s0 * g.plane;
    float *__restrict__ sxo = a.sxy_out + s0 * g.plane;
    float *__restrict__ szo = a.syz_out + s0 * g.plane;
    float *__restrict__ rqo = L > 0 ? a.rq + s0 * 2 * L * g.plane : nullptr;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        if (!own[i]) continue;
        vyo[off[i]] = v[i];
        sxo[off[i]] = sx[i];
        szo[off[i]] = sz[i];
#pragma unroll
        for (int l = 0; l + 1 < L; l += 2)
            *(float4 *)(rqo + 2 * l * g.plane + 4 * (size_t)off[i]) =
                make_float4(rr[i][l], qq[i][l], rr[i][l + 1], qq[i][l + 1]);
        if (L & 1) *(float2 *)(rqo + 2 * (L - 1) * g.plane + 2 * (size_t)off[i]) = make_float2(rr[i][L - 1], qq[i][L - 1]);
        if (xk[i] > 0) {
            const long long o = s0 * g.ny * fw2 + (cj[i] - 1) * fw2 + (xk[i] - 1);
            a.psx_out[o] = px[i];
            a.pvx[o] = wx[i];
        }
        if (yk[i] > 0) {
            const long long o = s0 * fw2 * g.nx + (yk[i] - 1) * g.nx + (cw[i] - 1);
            a.psy_out[o] = py[i];
            a.pvy[o] = wy[i];
        }
        if (sums) {
            grb[ci[i]] = gr[i];
            gub[ci[i]] = gu[i];
        }
        if (energy) wab[ci[i]] = wa[i];
    }
}

template <int L> hipError_t launch_l(const StepArgs &a, bool adjoint, bool extra, hipStream_t st)
{
    constexpr int K = DN_MULTI_K;
    const dim3 grid((unsigned)(a.tl_nblk8 * 8)), block(kMThreads);
    if (adjoint) {
        if (extra)
            hipLaunchKernelGGL((k_multi<K, L, true, true>), grid, block, 0, st, a);
        else
            hipLaunchKernelGGL((k_multi<K, L, true, false>), grid, block, 0, st, a);
    } else {
        if (extra)
            hipLaunchKernelGGL((k_multi<K, L, false, true>), grid, block, 0, st, a);
        else
            hipLaunchKernelGGL((k_multi<K, L, false, false>), grid, block, 0, st, a);
    }
    return hipGetLastError();
}

}  // namespace

template <> hipError_t launch_multi_k<DN_MULTI_K>(const StepArgs &a, bool adjoint, bool extra, hipStream_t st)
{
    if (a.ms_steps < 1 || a.ms_steps > multi_steps(DN_MULTI_K)) return hipErrorInvalidValue;
    switch (a.g.L) {
    case 0: return launch_l<0>(a, adjoint, extra, st);
    case 1: return launch_l<1>(a, adjoint, extra, st);
    case 2: return launch_l<2>(a, adjoint, extra, st);
    case 3: return launch_l<3>(a, adjoint, extra, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace dn
