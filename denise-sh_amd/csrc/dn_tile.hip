// The fused time step on two-dimensional tiles (gfx950).  Same arithmetic,
// in the same order and rounding, as the strip kernel of dn_kernels.hip; the
// file is compiled once per stencil half-order (DN_TILE_K) with
// -ffp-contract=off.
//
// One workgroup of WX x WY waves owns a tile of 64 WX columns x WY RW rows of
// one shot.  It loads everything the tile needs at once, computes the new vy
// of the tile and of the cells around it that the tile's stress update reads
// (2K-1 rows and 2K-1 columns, recomputed by their owners too), exchanges
// them through LDS and updates the stress: two barriers, no loop.
//
// What bounds it: the latency of one chain (batch slot -> fields -> stores)
// where the tiles do not fill the chip, the bytes where they do.  The strip
// kernel walks R + 2K - 1 rows one after the other, each with a wait of its
// own, and recomputes 2K - 1 of them; here every load of a wave is issued
// before the first is used and before anything is stored (a load behind a
// store waits for the store on this chip), the tables a workgroup reads
// first come in one scalar load (ShotSlot), and only tiles that reach into
// an absorbing region touch the CPML arrays.  A tile starts on a 128-byte
// line and writes whole lines (kPadX 32: -6 % at 4000 x 800, +2 % at
// 1200 x 300 against 64-byte aligned rows).
// Microseconds per step, strips -> tiles (one box, graph replay):
// 400 x 120 elastic FDORDER 4, 1 shot 12.2 -> 5.4; 1200 x 300 viscoelastic
// FDORDER 8 L 2, 4 shots 35.5 -> 22.3, gradient of 8 shots 56.6 -> 43.1;
// gradient of 4000 x 800, 2 shots 118.6 -> 118 (both at the rate of a large
// copy).
// Shape: 64 columns, eight waves, one or two rows per wave (dn_core.cpp
// chooses).  Also measured at 1200 x 300 x 8 / 4000 x 800 x 2: four waves of
// two rows 41.7 / 117, of four rows 45.3 / 118; eight of four rows 47 / 125;
// 128 columns, 4 x 2 waves of two rows 50 / 126; sixteen waves 63 / 151.
//
// Order of the tiles.  A tile reads 2K-1 columns of its neighbours on each
// side, a whole line per row for each, and where the fields exceed the
// memory-side cache that is HBM traffic unless the neighbour ran just before.
// With all shots of a tile in turn and the tiles down a column, the next
// column was a column of tiles times all shots away; now groups of three
// shots (all up to four), an eighth of each group's tiles to each XCD, bands
// of eight columns of tiles, row by row.  Gcell-updates/s of the gradient
// (strips, one box; then down a column, now, another): 1200 x 300 with 24
// shots 55.8; 51.0, 57.3; with 16 50.9; 54.1, 57.6; 2000 x 400 with 9 55.8;
// 54.2, 56.9; 4000 x 800 with 2 56.8; 57.8, 60.2, with 4 57.4; 58.7, 62.1.
// Bands of 4, 8, 16 columns (pairs of shots): 1200 x 300 with 24 shots 56.9
// 56.9 56.5, 2000 x 400 with 9 56.2 57.2 57.3, 4000 x 800 with 2 59.8 60.2
// 60.2.  Whole groups to one XCD leave XCDs idle once a group's records end
// (1973 x 397, six uneven shots, 89.8 ms against 81.8 for pairs).
//
// Old and new vy, sxy, syz and the velocity CPML memory are separate buffers
// (ping-pong), so the reads of the cells around a tile never race with their
// owners' writes; the stress CPML and the relaxation memory variables are
// touched by their owner only and are updated in place.
#include "dn_internal.h"
#include <hip/hip_fp16.h>

#pragma clang fp contract(off)

#ifndef DN_TILE_K
#error "compile with -DDN_TILE_K=<FDORDER / 2>"
#endif

namespace dn {

namespace {

__device__ __forceinline__ float ldf(const float *base, unsigned boff)
{
    return *(const float *)((const char *)base + boff);
}
__device__ __forceinline__ void stf(float *base, unsigned boff, float v) { *(float *)((char *)base + boff) = v; }
__device__ __forceinline__ float2 ld2(const float *base, unsigned boff)
{
    return *(const float2 *)((const char *)base + boff);
}
__device__ __forceinline__ float4 ld4(const float *base, unsigned boff)
{
    return *(const float4 *)((const char *)base + boff);
}
__device__ __forceinline__ void st2(float *base, unsigned boff, float2 v) { *(float2 *)((char *)base + boff) = v; }
__device__ __forceinline__ void st4(float *base, unsigned boff, float4 v) { *(float4 *)((char *)base + boff) = v; }

__device__ __forceinline__ float wave_max(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ uint16_t f2bf16(float x)
{
    unsigned int u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf162f(unsigned h) { return __uint_as_float(h << 16); }
__device__ __forceinline__ float h2f(unsigned h) { return __half2float(__ushort_as_half((unsigned short)h)); }

// n / d with m = (2^32 - 1) / d: the estimate is at most one short
__device__ __forceinline__ int udiv(int n, int d, unsigned m)
{
    const int q = (int)__umulhi((unsigned)n, m);
    return n - q * d >= d ? q + 1 : q;
}

// EX as in k_step: 0 plain steps; 1 FP32 snapshots or FP16 staging, the
// pseudo-Hessian (forward), correlation with FP32 snapshots (adjoint); 2 BF16
// snapshots (forward), correlation with 16-bit snapshots (adjoint).
template <int K, int L, bool ADJ, int EX, int WX, int WY, int RW>
__global__ __launch_bounds__(kWave *WX *WY) void k_tile(const StepArgs a)
{
    constexpr bool S16 = ADJ && EX == 2, B16W = !ADJ && EX == 2, VISCO = L > 0;
    constexpr int LD = L > 0 ? L : 1;
    constexpr int H = 2 * K - 1;          // rows and columns of new vy around the tile (K-1 before, K after)
    constexpr int TX = kWave * WX;        // columns of the tile
    constexpr int OY = WY * RW;           // rows of the tile
    constexpr int VP = TX + H;         // columns of new vy (and of old syz)
    constexpr int XP = TX + 2 * H;     // columns of old sxy (2K-1 before, 2K-1 after)
    constexpr int NV = OY + H;            // rows of new vy (and of old sxy)
    constexpr int NZ = OY + 2 * H;        // rows of old syz
    constexpr int NT = kWave * WX * WY;
    constexpr int NQ = (H + WY - 1) / WY;                  // rows around the tile per wave
    constexpr int NSX = (2 * H * OY + NT - 1) / NT;        // side cells per thread: sxy beside the tile's rows,
    constexpr int NSZ = (H * (OY + H) + NT - 1) / NT;      // syz beside the tile,
    constexpr int NSV = (H * OY + NT - 1) / NT;            // new vy beside the tile
    __shared__ float lx[NV * XP];         // (j0-(K-1).., c0-(2K-1)..)
    __shared__ float lz[NZ * VP];         // (j0-(2K-1).., c0-(K-1)..)
    __shared__ float lv[NV * VP];         // (j0-(K-1).., c0-(K-1)..)

    // order: groups of shots, an eighth of each group's tiles to each XCD, and
    // in a group bands of eight columns of tiles, in a band row by row, each
    // tile for all shots of the group
    const int w_ = blockIdx.x, grp = udiv(w_ >> 3, a.tl_g8, a.tl_mg8);
    const bool full = grp < a.tl_full;
    const int gs = full ? a.tl_grp : a.tl_last;
    const int gl = (w_ & 7) * (full ? a.tl_g8 : a.tl_l8) + (w_ >> 3) - grp * a.tl_g8;
    if (gl >= gs * a.tl_tiles) return;
    const int tile = udiv(gl, gs, full ? a.tl_mgrp : a.tl_mlast), s = grp * a.tl_grp + gl - tile * gs;
    const int band = udiv(tile, a.tl_bblk, a.tl_mbblk), bl = tile - band * a.tl_bblk;
    const bool wide = band < a.tl_bfull;
    const int by = wide ? bl >> 3 : udiv(bl, a.tl_blast, a.tl_mblast), bx = 8 * band + bl - by * (wide ? 8 : a.tl_blast);
    const Geo &g = a.g;
    const ShotSlot sl = a.slots[s];
    const int nt = *a.nt_base + a.nt;
    const int S = sl.shot, NTs = sl.nt;
    if (S < 0 || S >= a.nshots_all || nt > NTs) {   // finished shots (uneven record lengths) rest
        // a stale or foreign shot map: touch nothing, reported by the host after the pass
        if (S < 0 || S >= a.nshots_all) a.status[2] = 1;
        return;
    }

    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const int wx = wv % WX, wy = wv / WX, lc = wx * kWave + lane;   // lc: column in the tile
    const int c0 = 1 + bx * TX, j0 = 1 + by * OY;
    const int fw = g.fw, fw2 = 2 * g.fw;
    const int nxny = g.nx * g.ny;
    // column of the cell an index beyond the edges stands for (BOUNDARY 1)
    auto wrapc = [&](int c) -> int { return !g.periodic ? c : (c < 1 ? c + g.nx : (c > g.nx ? c - g.nx : c)); };
    // byte offset of (j, c); rows below the frame's last but one read zeros there
    auto rowo = [&](int j) -> unsigned { return (unsigned)((min(j, g.ny + kPadY - 1) - 1 + g.yoff) * g.pitch) * 4u; };
    auto colo = [&](int c) -> unsigned { return (unsigned)(wrapc(c) - 1 + g.xoff) * 4u; };
    auto xkof = [&](int c) -> int {
        if (fw <= 0 || g.periodic || c < 1 || c > g.nx) return 0;
        return (c <= fw) ? c : ((c >= g.nx - fw + 1) ? c - g.nx + fw2 : 0);
    };
    auto ykof = [&](int r) -> int {
        if (fw <= 0 || r < 1 || r > g.ny) return 0;
        if (!g.free_surf && r <= fw) return r;
        return (r >= g.ny - fw + 1) ? r - g.ny + fw2 : 0;
    };
    auto inx = [&](int c) -> bool { return g.periodic || (c >= 1 && c <= g.nx); };

    const long long s0 = s;
    const float *__restrict__ vyi = a.vy_in + s0 * g.plane;
    const float *__restrict__ sxi = a.sxy_in + s0 * g.plane;
    const float *__restrict__ szi = a.syz_in + s0 * g.plane;
    float *__restrict__ vyo = a.vy_out + s0 * g.plane;
    float *__restrict__ sxo_ = a.sxy_out + s0 * g.plane;
    float *__restrict__ szo = a.syz_out + s0 * g.plane;
    float *__restrict__ rqb = VISCO ? a.rq + s0 * 2 * L * g.plane : nullptr;
    auto rqp = [&](int k) -> float * { return rqb + (long long)k * 4 * g.plane; };
    const float *__restrict__ bf = a.bfield;
    const float *__restrict__ pxi = a.psx_in + s0 * g.ny * fw2;
    float *__restrict__ pxo = a.psx_out + s0 * g.ny * fw2;
    const float *__restrict__ pyi = a.psy_in + s0 * fw2 * g.nx;
    float *__restrict__ pyo = a.psy_out + s0 * fw2 * g.nx;
    float *__restrict__ pvxb = a.pvx + s0 * g.ny * fw2;
    float *__restrict__ pvyb = a.pvy + s0 * fw2 * g.nx;
    const float *__restrict__ pmlb = a.pml.Kx;   // twelve packed profiles, stride 2 FW + 1
    const int pn = fw2 + 1;

    bool fstore = false, corr = false, hsum = false;
    int slot = 0;
    if (!EX) {
    } else if (!ADJ) {
        if (a.store_mode != 0 && ((nt - 1) % a.dtinv) == 0) {
            fstore = true;
            slot = (nt - 1) / a.dtinv;
        }
        // hessian.c:91: stored steps 1..NTDTINV-1 of this shot
        if (a.hess && ((nt - 1) % a.dtinv) == 0 && (nt - 1) / a.dtinv < (NTs + a.dtinv - 1) / a.dtinv - 1) hsum = true;
    } else {
        const int sf = NTs - nt + 1;   // forward step paired with this adjoint step
        if (((sf - 1) % a.dtinv) == 0) {
            corr = true;
            slot = (sf - 1) / a.dtinv;
        }
    }

    const long long shot_off = s0 * nxny;
    float *__restrict__ grb = (EX && a.grad_rho) ? a.grad_rho + shot_off : nullptr;
    float *__restrict__ gub = (EX && a.grad_u) ? a.grad_u + shot_off : nullptr;
    float *__restrict__ wab = (EX && a.wacc) ? a.wacc + shot_off : nullptr;
    const long long sbase = s0 * a.snap_shot_stride + (long long)slot * 3 * nxny;
    float *__restrict__ snw = (EX && a.snap) ? a.snap + sbase : nullptr;
    uint16_t *__restrict__ sn16 = (EX && a.snap16) ? a.snap16 + sbase : nullptr;
    float *__restrict__ stg = (EX && a.stage) ? a.stage + s0 * 3 * nxny : nullptr;
    // ---- loads: everything the tile needs, before anything waits or stores ----
    // a source in the tile or the cells around it (uniform)
    const int sb = sl.src0, se = ADJ ? sl.src0 : sl.src1;
    auto near = [&](int si, int sj) -> bool {
        return sj > j0 - K && sj < j0 + OY + K && (g.periodic || (si > c0 - K && si < c0 + TX + K));
    };
    bool has_src = false;
    float sig0 = 0.0f;                    // the shot's first source's sample of this step
    if (!ADJ && se > sb) {
        has_src = near(sl.si, sl.sj);
        if (has_src) sig0 = a.src_sig[(long long)sb * a.nt_max + (nt - 1)];
        for (int l = sb + 1; l < se; ++l) has_src = has_src || near(a.src_i[l], a.src_j[l]);
    }
    const int c = c0 + lc;
    const bool own_x = c <= g.nx;
    const unsigned co = colo(c);
    const int cw = wrapc(c);
    const int xk = xkof(c);
    const int jb = j0 + wy * RW;          // first own row of the wave
    float sx[RW], sz[RW], vo[RW], bb[RW];
#pragma unroll
    for (int t = 0; t < RW; ++t) {
        const unsigned o = rowo(jb + t) + co;
        sx[t] = ldf(sxi, o);
        sz[t] = ldf(szi, o);
        vo[t] = ldf(vyi, o);
        bb[t] = ldf(bf, o);
    }
    // receiver-table row of the own and the surrounding rows (-1: none)
    int rrow[RW], qrr[NQ], srr[NSV];
#pragma unroll
    for (int t = 0; t < RW; ++t) rrow[t] = (jb + t <= g.ny) ? a.rec_row[jb + t] : -1;
    // rows around the tile: new vy rows (K-1 above, K below), syz rows beyond
    float qsx[NQ], qhx[NQ], qsz[NQ], qvo[NQ], qbb[NQ], qfz[NQ];
    auto qrow = [&](int q) -> int { return q < K - 1 ? j0 - (K - 1) + q : j0 + OY + (q - (K - 1)); };
    auto qfar = [&](int q) -> int { return q < K ? j0 - H + q : j0 + OY + K + (q - K); };
    // column beside a row of the tile: H cells, K left and K-1 right (old sxy)
    const bool hl = wx == 0 && lane < K, hr = wx == WX - 1 && lane >= K && lane < H;
    const unsigned ho = colo(hl ? c0 - K + lane : (hr ? c0 + TX + (lane - K) : c));
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int q = wy + n * WY;
        qsx[n] = qhx[n] = qsz[n] = qvo[n] = qbb[n] = qfz[n] = 0.0f;
        qrr[n] = -1;
        if (q < H) {
            const int j = qrow(q);
            if (ADJ && j >= 1 && j <= g.ny) qrr[n] = a.rec_row[j];
            const unsigned r = rowo(j);
            qsx[n] = ldf(sxi, r + co);
            qhx[n] = ldf(sxi, r + ho);
            qsz[n] = ldf(szi, r + co);
            qvo[n] = ldf(vyi, r + co);
            qbb[n] = ldf(bf, r + co);
            qfz[n] = ldf(szi, rowo(qfar(q)) + co);
        }
    }
    // cells beside the tile (flat over the workgroup)
    float ssx[NSX], ssz[NSZ], svo[NSV], sbb[NSV];
#pragma unroll
    for (int n = 0; n < NSX; ++n) {
        const int e = min((int)threadIdx.x + n * NT, 2 * H * OY - 1);
        const int r = e / (2 * H), k = e - r * (2 * H);
        const int cc = k < H ? c0 - H + k : c0 + TX + (k - H);
        ssx[n] = ldf(sxi, rowo(j0 + r) + colo(cc));
    }
    auto vside = [&](int k) -> int { return k < K - 1 ? c0 - (K - 1) + k : c0 + TX + (k - (K - 1)); };
#pragma unroll
    for (int n = 0; n < NSZ; ++n) {
        const int e = min((int)threadIdx.x + n * NT, H * (OY + H) - 1);
        const int r = e / H, k = e - r * H;
        ssz[n] = ldf(szi, rowo(j0 - K + r) + colo(vside(k)));
    }
#pragma unroll
    for (int n = 0; n < NSV; ++n) {
        const int e = min((int)threadIdx.x + n * NT, H * OY - 1);
        const int r = e / H, k = e - r * H;
        const unsigned o = rowo(j0 + r) + colo(vside(k));
        svo[n] = ldf(vyi, o);
        sbb[n] = ldf(bf, o);
        srr[n] = (ADJ && j0 + r <= g.ny) ? a.rec_row[j0 + r] : -1;
    }
    // velocity CPML: the memory variables and profiles (K, a, b) of the own
    // and the surrounding rows, in tiles that reach into an absorbing region
    // (uniform); the cells beside the tile and the stress load theirs later,
    // which keeps them out of the registers here
    const bool tpx = fw > 0 && !g.periodic && (c0 - (K - 1) <= fw || c0 + TX - 1 + K >= g.nx - fw + 1);
    const bool tpy = fw > 0 && ((!g.free_surf && j0 - (K - 1) <= fw) || j0 + OY - 1 + K >= g.ny - fw + 1);
    auto pxo_of = [&](int j, int k) -> unsigned { return (unsigned)((j - 1) * fw2 + (k - 1)) * 4u; };
    auto pyo_of = [&](int k, int ccw) -> unsigned { return (unsigned)((k - 1) * g.nx + (ccw - 1)) * 4u; };
    float px[RW], py[RW], qpx[NQ], qpy[NQ], cx[3], cy[RW][3], cqy[NQ][3];
    if (tpx && xk > 0) {
#pragma unroll
        for (int f = 0; f < 3; ++f) cx[f] = pmlb[f * pn + xk];
#pragma unroll
        for (int t = 0; t < RW; ++t)
            if (jb + t <= g.ny) px[t] = ldf(pxi, pxo_of(jb + t, xk));
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            const int q = wy + n * WY, j = qrow(q);
            if (q < H && j >= 1 && j <= g.ny) qpx[n] = ldf(pxi, pxo_of(j, xk));
        }
    }
    if (tpy) {
#pragma unroll
        for (int t = 0; t < RW; ++t) {
            const int yk = ykof(jb + t);
            if (yk > 0) {
#pragma unroll
                for (int f = 0; f < 3; ++f) cy[t][f] = pmlb[(6 + f) * pn + yk];
                if (inx(c)) py[t] = ldf(pyi, pyo_of(yk, cw));
            }
        }
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            const int q = wy + n * WY, yk = q < H ? ykof(qrow(q)) : 0;
            if (yk > 0) {
#pragma unroll
                for (int f = 0; f < 3; ++f) cqy[n][f] = pmlb[(6 + f) * pn + yk];
                if (inx(c)) qpy[n] = ldf(pyi, pyo_of(yk, cw));
            }
        }
    }
    // static coefficients and memory variables of the own cells
    float s1[RW], s2[RW], dp[RW][LD], dd[RW][LD], rr[RW][LD], qq[RW][LD];
#pragma unroll
    for (int t = 0; t < RW; ++t) {
        const unsigned o = rowo(jb + t) + co;
        if (!VISCO) {
            const float2 v = ld2(a.spk, o * 2u);
            s1[t] = v.x;
            s2[t] = v.y;
        } else {
            const float4 v = ld4(a.spk, o * 4u);
            s1[t] = v.x;
            s2[t] = v.y;
            dp[t][0] = v.z;
            dd[t][0] = v.w;
#pragma unroll
            for (int l = 1; l < L; ++l) {
                const float2 u = ld2(a.spk + 4 * g.plane + 2 * (long long)(l - 1) * g.plane, o * 2u);
                dp[t][l] = u.x;
                dd[t][l] = u.y;
            }
#pragma unroll
            for (int l = 0; l + 1 < L; l += 2) {
                const float4 u = ld4(rqp(l / 2), o * 4u);
                rr[t][l] = u.x;
                qq[t][l] = u.y;
                rr[t][l + 1] = u.z;
                qq[t][l + 1] = u.w;
            }
            if (L & 1) {
                const float2 u = ld2(rqp(L / 2), o * 2u);
                rr[t][L - 1] = u.x;
                qq[t][L - 1] = u.y;
            }
        }
    }

    // accumulators and stored snapshots of the own cells, where this step uses
    // them (every lane loads, at element 0 where it owns nothing)
    float egr[RW], ef0[RW], ewa[RW], egu[RW], efy[RW], efu[RW];
    unsigned eh0[RW], ehy[RW], ehu[RW];
    if (EX) {
#pragma unroll
        for (int t = 0; t < RW; ++t) {
            const unsigned ci = (jb + t <= g.ny && own_x) ? (unsigned)((jb + t - 1) * g.nx + (cw - 1)) : 0u;
            if ((ADJ && corr) || (!ADJ && hsum)) {
                egr[t] = grb[ci];
                egu[t] = gub[ci];
            }
            if ((ADJ && corr) || (!ADJ && fstore)) ewa[t] = wab[ci];
            if (ADJ && corr) {
                if (S16) {
                    eh0[t] = sn16[ci];
                    ehy[t] = sn16[nxny + ci];
                    ehu[t] = sn16[2 * nxny + ci];
                } else {
                    ef0[t] = snw[ci];
                    efy[t] = snw[nxny + ci];
                    efu[t] = snw[2 * nxny + ci];
                }
            }
        }
    }

    // receivers: index of the own cells (-1: none), and the residuals that
    // enter the new vy of the adjoint
    int ri[RW];
    float res[RW], qres[NQ], sres[NSV];
    bool qrec[NQ], srec[NSV];
#pragma unroll
    for (int t = 0; t < RW; ++t) {
        ri[t] = -1;
        if (rrow[t] >= 0 && inx(c)) {
            ri[t] = a.rec_tab[rrow[t] + cw];
            if (ADJ && ri[t] >= 0) res[t] = a.resid[(s0 * a.ntr + ri[t]) * a.nt_max + (nt - 1)];
        }
    }
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        qrec[n] = false;
        if (ADJ && qrr[n] >= 0 && inx(c)) {
            const int r = a.rec_tab[qrr[n] + cw];
            qrec[n] = r >= 0;
            if (r >= 0) qres[n] = a.resid[(s0 * a.ntr + r) * a.nt_max + (nt - 1)];
        }
    }
#pragma unroll
    for (int n = 0; n < NSV; ++n) {
        srec[n] = false;
        if (ADJ && srr[n] >= 0) {
            const int cc = vside(min((int)threadIdx.x + n * NT, H * OY - 1) % H);
            if (inx(cc)) {
                const int r = a.rec_tab[srr[n] + wrapc(cc)];
                srec[n] = r >= 0;
                if (r >= 0) sres[n] = a.resid[(s0 * a.ntr + r) * a.nt_max + (nt - 1)];
            }
        }
    }

    // ---- old stress into LDS ----------------------------------------------
#pragma unroll
    for (int t = 0; t < RW; ++t) {
        lx[(wy * RW + t + K - 1) * XP + H + lc] = sx[t];
        lz[(wy * RW + t + H) * VP + K - 1 + lc] = sz[t];
    }
    auto qlv = [&](int q) -> int { return q < K - 1 ? q : OY + q; };              // lx, lv row of qrow(q)
    auto qlf = [&](int q) -> int { return q < K ? q : OY + 2 * K - 1 + q; };      // lz row of qfar(q)
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int q = wy + n * WY;
        if (q < H) {
            lx[qlv(q) * XP + H + lc] = qsx[n];
            if (hl || hr) lx[qlv(q) * XP + (hl ? H - K + lane : TX + H + (lane - K))] = qhx[n];
            lz[(qlv(q) + K) * VP + K - 1 + lc] = qsz[n];
            lz[qlf(q) * VP + K - 1 + lc] = qfz[n];
        }
    }
#pragma unroll
    for (int n = 0; n < NSX; ++n) {
        const int e = (int)threadIdx.x + n * NT;
        if (e < 2 * H * OY) {
            const int r = e / (2 * H), k = e - r * (2 * H);
            lx[(r + K - 1) * XP + (k < H ? k : TX + k)] = ssx[n];
        }
    }
    auto vscol = [&](int k) -> int { return k < K - 1 ? k : TX + k; };         // lz, lv column of vside(k)
#pragma unroll
    for (int n = 0; n < NSZ; ++n) {
        const int e = (int)threadIdx.x + n * NT;
        if (e < H * (OY + H)) {
            const int r = e / H, k = e - r * H;
            lz[(r + K - 1) * VP + vscol(k)] = ssz[n];
        }
    }
    __syncthreads();

    // ---- new vy -------------------------------------------------------------
    // x-CPML (update_v_PML.c: left, c <= FW, or right, c >= NX-FW+1) and
    // y-CPML (top without a free surface, or bottom) of one derivative
    auto cpml = [](const float *k, float &p, float &d) {
        p = k[2] * p + k[1] * d;
        d = d / k[0] + p;
    };
    // new vy of cell (j, ccw) from the sum of the derivatives: update, then
    // sources (forward) or the cell's residual (adjoint)
    auto velocity = [&](int j, int ccw, float tsum, float vold, float b, bool rec, float r) -> float {
        float vn = vold + ((b * a.DT) * tsum) / a.DH;
        if (ADJ) {
            if (rec) vn = vn + r;
        } else if (has_src) {
            if (sl.sj == j && sl.si == ccw) vn = vn + sig0;
            for (int l = sb + 1; l < se; ++l)
                if (a.src_j[l] == j && a.src_i[l] == ccw) vn = vn + a.src_sig[(long long)l * a.nt_max + (nt - 1)];
        }
        return vn;
    };
    auto xsum = [&](const float *p) -> float {   // p: the cell in lx
        float v = a.hc[1] * (p[0] - p[-1]);
#pragma unroll
        for (int m = 2; m <= K; ++m) v = v + a.hc[m] * (p[m - 1] - p[-m]);
        return v;
    };
    auto ysum = [&](const float *p, int st) -> float {   // p: the cell in lz or in a register window
        float v = a.hc[1] * (p[0] - p[-st]);
#pragma unroll
        for (int m = 2; m <= K; ++m) {
            const float hy = (K == 6 && m == 6) ? a.hcy6 : a.hc[m];
            v = v + hy * (p[(m - 1) * st] - p[-m * st]);
        }
        return v;
    };

    // BF16 snapshots (EX 2 forward): the ring of maxima of k_step: snapshot k
    // is scaled by the exponent of the largest |x| of snapshot k - 1
    float enc[3] = {1.0f, 1.0f, 1.0f};
    if (B16W && fstore) {
        unsigned int *ring = a.stage_max + s0 * 9;
        const int kp = (slot + 2) % 3, kc = (slot + 1) % 3;
        const bool first = tile == 0 && threadIdx.x == 0;
#pragma unroll
        for (int f = 0; f < 3; ++f) {
            const float m = __uint_as_float(ring[kp * 3 + f]);
            int e = 0;
            if (m > 0.0f && isfinite(m)) {
                (void)frexpf(m, &e);
                e = min(max(e, -100), 100);
            }
            enc[f] = ldexpf(1.0f, -e);
            if (first) {
                ring[kc * 3 + f] = 0u;
                a.snap_scale[(s0 * (a.snap_shot_stride / (3 * nxny)) + slot) * 3 + f] = ldexpf(1.0f, e);
            }
        }
    }
    float dsc[3] = {1.0f, 1.0f, 1.0f};
    if (S16 && corr) {
        const float *scp = a.snap_scale + (s0 * (a.snap_shot_stride / (3 * nxny)) + slot) * 3;
        dsc[0] = scp[0];
        dsc[1] = scp[1];
        dsc[2] = scp[2];
    }
    auto decode = [&](unsigned h, float scale) -> float { return (a.snap_kind == 1 ? bf162f(h) : h2f(h)) * scale; };
    float smx0 = 0.0f, smx1 = 0.0f, smx2 = 0.0f;

#pragma unroll
    for (int n = 0; n < NSV; ++n) {
        const int e = (int)threadIdx.x + n * NT;
        if (e < H * OY) {
            const int r = e / H, k = e - r * H;
            const int j = j0 + r, cc = vside(k);
            float vn = 0.0f;
            if (j <= g.ny && inx(cc)) {
                const int lk = vscol(k), ccw = wrapc(cc);
                float gx = xsum(lx + (r + K - 1) * XP + K + lk);
                float gy = ysum(lz + (r + H) * VP + lk, VP);
                if (tpx) {
                    const int kx = xkof(cc);
                    if (kx > 0) {
                        const float ck[3] = {pmlb[0 * pn + kx], pmlb[1 * pn + kx], pmlb[2 * pn + kx]};
                        float p = ldf(pxi, pxo_of(j, kx));
                        cpml(ck, p, gx);
                    }
                }
                if (tpy) {
                    const int yk = ykof(j);
                    if (yk > 0) {
                        const float ck[3] = {pmlb[6 * pn + yk], pmlb[7 * pn + yk], pmlb[8 * pn + yk]};
                        float p = ldf(pyi, pyo_of(yk, ccw));
                        cpml(ck, p, gy);
                    }
                }
                vn = velocity(j, ccw, gx + gy, svo[n], sbb[n], srec[n], sres[n]);
            }
            lv[(r + K - 1) * VP + vscol(k)] = vn;
        }
    }
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int q = wy + n * WY;
        if (q < H) {
            const int j = qrow(q);
            float vn = 0.0f;
            if (j >= 1 && j <= g.ny && inx(c)) {
                float gx = xsum(lx + qlv(q) * XP + H + lc);
                float gy = ysum(lz + (qlv(q) + K) * VP + K - 1 + lc, VP);
                if (tpx && xk > 0) cpml(cx, qpx[n], gx);
                if (tpy && ykof(j) > 0) cpml(cqy[n], qpy[n], gy);
                vn = velocity(j, cw, gx + gy, qvo[n], qbb[n], qrec[n], qres[n]);
            }
            lv[qlv(q) * VP + K - 1 + lc] = vn;
        }
    }
    float vnew[RW];
    {
        float zw[RW + H];
#pragma unroll
        for (int t = 0; t < RW + H; ++t)
            zw[t] = (t >= K && t < K + RW) ? sz[t - K] : lz[(wy * RW + t + K - 1) * VP + K - 1 + lc];
#pragma unroll
        for (int t = 0; t < RW; ++t) {
            const int j = jb + t;
            float vn = 0.0f;
            if (j <= g.ny && inx(c)) {
                const bool own = own_x;
                float gx = xsum(lx + (wy * RW + t + K - 1) * XP + H + lc);
                float gy = ysum(zw + K + t, 1);
                if (tpx && xk > 0) {
                    cpml(cx, px[t], gx);
                    if (own) stf(pxo, pxo_of(j, xk), px[t]);
                }
                if (tpy) {
                    const int yk = ykof(j);
                    if (yk > 0) {
                        cpml(cy[t], py[t], gy);
                        if (own) stf(pyo, pyo_of(yk, cw), py[t]);
                    }
                }
                const float tsum = gx + gy;
                vn = velocity(j, cw, tsum, vo[t], bb[t], ri[t] >= 0, res[t]);
                const unsigned ci = (unsigned)((j - 1) * g.nx + (cw - 1));
                if (EX && !ADJ && hsum && own) {
                    const float acc = (bb[t] * tsum) / a.DH;   // vyp1 (hess_utty)
                    grb[ci] = egr[t] + (acc * acc);
                }
                if (EX && !ADJ && fstore && own) {
                    const float acc = (bb[t] * tsum) / a.DH;   // vyp1, update_v_PML.c:184
                    if (B16W) {
                        sn16[ci] = f2bf16(acc * enc[0]);
                        smx0 = fmaxf(smx0, fabsf(acc));
                    } else if (a.store_mode == 1) {
                        snw[ci] = acc;
                    } else {
                        stg[ci] = acc;
                        smx0 = fmaxf(smx0, fabsf(acc));
                    }
                }
                if (EX && ADJ && corr && own) {
                    // vyp1 = old vy (update_v_PML.c:189); denise.c:1589
                    const float f0 = S16 ? decode(eh0[t], dsc[0]) : ef0[t];
                    grb[ci] = egr[t] + (vo[t] * f0);
                }
                // instability latch at the reference's probe cell
                if (j == (g.ny >> 1) && own && c == (g.nx >> 1) && !(vn == vn))
                    if (atomicCAS(&a.status[0], 0, nt) == 0) a.status[1] = S + 1;
            }
            vnew[t] = vn;
            lv[(wy * RW + t + K - 1) * VP + K - 1 + lc] = vn;
        }
    }
    // the stress CPML of the own cells
    float wx_[RW], wy_[RW], sx_[3], sy_[RW][3];
    if (tpx && xk > 0) {
#pragma unroll
        for (int f = 0; f < 3; ++f) sx_[f] = pmlb[(3 + f) * pn + xk];
#pragma unroll
        for (int t = 0; t < RW; ++t)
            if (jb + t <= g.ny) wx_[t] = ldf(pvxb, pxo_of(jb + t, xk));
    }
    if (tpy) {
#pragma unroll
        for (int t = 0; t < RW; ++t) {
            const int yk = ykof(jb + t);
            if (yk > 0) {
                // Q2: the viscoelastic stress uses the full-grid y profile on top
                const int b0 = (VISCO && !g.free_surf && jb + t <= fw) ? 6 : 9;
#pragma unroll
                for (int f = 0; f < 3; ++f) sy_[t][f] = pmlb[(b0 + f) * pn + yk];
                if (own_x) wy_[t] = ldf(pvyb, pyo_of(yk, cw));
            }
        }
    }
    __syncthreads();

    // ---- stress ---------------------------------------------------------------
    {
        float vw[RW + H];
#pragma unroll
        for (int t = 0; t < RW + H; ++t)
            vw[t] = (t >= K - 1 && t < K - 1 + RW) ? vnew[t - (K - 1)] : lv[(wy * RW + t) * VP + K - 1 + lc];
#pragma unroll
        for (int t = 0; t < RW; ++t) {
            const int js = jb + t;
            if (js > g.ny || !own_x) continue;
            const unsigned gs = rowo(js) + co;
            stf(vyo, gs, vnew[t]);
            if (!ADJ && a.seis != nullptr && ri[t] >= 0)
                a.seis[(s0 * a.ntr + ri[t]) * a.nt_max + (nt - 1)] = vnew[t];
            const float *lvy = lv + (wy * RW + t + K - 1) * VP + K - 1 + lc;
            const float *p = vw + K - 1 + t;
            float vyx = a.hc[1] * (lvy[1] - lvy[0]);
            float vyy = a.hc[1] * (p[1] - p[0]);
#pragma unroll
            for (int m = 2; m <= K; ++m) {
                vyx = vyx + a.hc[m] * (lvy[m] - lvy[-m + 1]);
                vyy = vyy + a.hc[m] * (p[m] - p[-m + 1]);
            }
            vyx = vyx * a.dhi;
            vyy = vyy * a.dhi;
            if (tpx && xk > 0) {   // update_s_*_PML.c: x-CPML of the stress
                cpml(sx_, wx_[t], vyx);
                stf(pvxb, pxo_of(js, xk), wx_[t]);
            }
            if (tpy) {
                const int yk = ykof(js);
                if (yk > 0) {
                    cpml(sy_[t], wy_[t], vyy);
                    stf(pvyb, pyo_of(yk, cw), wy_[t]);
                }
            }
            float sxn, syn;
            if (!VISCO) {
                sxn = sx[t] + s1[t] * vyx;
                syn = sz[t] + s2[t] * vyy;
            } else {
                float sumr = 0.0f, sumq = 0.0f;
#pragma unroll
                for (int l = 0; l < L; ++l) {
                    sumr += rr[t][l];
                    sumq += qq[t][l];
                }
                sxn = sx[t] + ((s1[t] * vyx) + (a.dthalbe * sumr));
                syn = sz[t] + ((s2[t] * vyy) + (a.dthalbe * sumq));
                sumr = 0.0f;
                sumq = 0.0f;
#pragma unroll
                for (int l = 0; l < L; ++l) {
                    rr[t][l] = a.bip[l] * (rr[t][l] * a.cip[l] - (dp[t][l] * vyx));
                    qq[t][l] = a.bjm[l] * (qq[t][l] * a.cjm[l] - (dd[t][l] * vyy));
                    sumr += rr[t][l];
                    sumq += qq[t][l];
                }
#pragma unroll
                for (int l = 0; l + 1 < L; l += 2)
                    st4(rqp(l / 2), gs * 4u, make_float4(rr[t][l], qq[t][l], rr[t][l + 1], qq[t][l + 1]));
                if (L & 1) st2(rqp(L / 2), gs * 2u, make_float2(rr[t][L - 1], qq[t][L - 1]));
                sxn = sxn + (a.dthalbe * sumr);
                syn = syn + (a.dthalbe * sumq);
            }
            stf(sxo_, gs, sxn);
            stf(szo, gs, syn);
            if (EX) {
                const unsigned ci = (unsigned)((js - 1) * g.nx + (cw - 1));
                const float vc = vnew[t];
                if (!ADJ && fstore) {
                    if (B16W) {
                        uint16_t *b0 = sn16 + ci;
                        b0[nxny] = f2bf16(vyy * enc[1]);       // uy
                        b0[2 * nxny] = f2bf16(vyx * enc[2]);   // uyx
                    } else {
                        float *b0 = (a.store_mode == 1 ? snw : stg) + ci;
                        b0[nxny] = vyy;        // uy  (forward_prop_y)
                        b0[2 * nxny] = vyx;    // uyx (forward_prop_u)
                    }
                    smx1 = fmaxf(smx1, fabsf(vyy));
                    smx2 = fmaxf(smx2, fabsf(vyx));
                    wab[ci] = ewa[t] + vc * vc;   // eprecond.c:11
                }
                if (!ADJ && hsum) {
                    const float eyx = 0.5f * vyx;     // hess_save.c:13 (exact in float)
                    gub[ci] = egu[t] + ((vyy * vyy) + (eyx * eyx));
                }
                if (ADJ && corr) {
                    const float fy = S16 ? decode(ehy[t], dsc[1]) : efy[t];
                    const float fu = S16 ? decode(ehu[t], dsc[2]) : efu[t];
                    gub[ci] = egu[t] + ((fu * sxn) + (fy * syn));   // denise.c:1609
                    wab[ci] = ewa[t] + vc * vc;
                }
            }
        }
    }

    // per-snapshot max |x| for the reduced-precision codecs (FP16 staging:
    // the scale of this snapshot; BF16: the scale of the next one): over the
    // workgroup, then one atomic per field where it raises the maximum
    if (EX && !ADJ && fstore && (B16W || a.store_mode == 2)) {
        __shared__ float red[WX * WY][3];
        const float m0 = wave_max(smx0), m1 = wave_max(smx1), m2 = wave_max(smx2);
        if (lane == 0) {
            red[wv][0] = m0;
            red[wv][1] = m1;
            red[wv][2] = m2;
        }
        __syncthreads();
        if (threadIdx.x < 3) {
            unsigned int *mx = (B16W ? a.stage_max + s0 * 9 + (slot % 3) * 3 : a.stage_max + s0 * 3) + threadIdx.x;
            float m = red[0][threadIdx.x];
            for (int k = 1; k < WX * WY; ++k) m = fmaxf(m, red[k][threadIdx.x]);
            const unsigned int bits = __float_as_uint(m);
            if (bits > __atomic_load_n(mx, __ATOMIC_RELAXED)) atomicMax(mx, bits);
        }
    }
}

template <int K, int L, int WX, int WY, int RW>
hipError_t launch_shape(const StepArgs &a, bool adjoint, bool extra, hipStream_t st)
{
    const dim3 grid((unsigned)(a.tl_nblk8 * 8)), block(kWave * WX * WY);
    if (a.tl_w != kWave * WX || a.tl_h != WY * RW) return hipErrorInvalidValue;
    if (adjoint) {
        if (extra && a.snap_kind != 0)
            hipLaunchKernelGGL((k_tile<K, L, true, 2, WX, WY, RW>), grid, block, 0, st, a);
        else if (extra)
            hipLaunchKernelGGL((k_tile<K, L, true, 1, WX, WY, RW>), grid, block, 0, st, a);
        else
            hipLaunchKernelGGL((k_tile<K, L, true, 0, WX, WY, RW>), grid, block, 0, st, a);
    } else {
        if (extra && a.store_mode == 3)
            hipLaunchKernelGGL((k_tile<K, L, false, 2, WX, WY, RW>), grid, block, 0, st, a);
        else if (extra)
            hipLaunchKernelGGL((k_tile<K, L, false, 1, WX, WY, RW>), grid, block, 0, st, a);
        else
            hipLaunchKernelGGL((k_tile<K, L, false, 0, WX, WY, RW>), grid, block, 0, st, a);
    }
    return hipGetLastError();
}

template <int K, int L>
hipError_t launch_kl(const StepArgs &a, bool adjoint, bool extra, hipStream_t st)
{
    switch (a.tl_rw) {
    case 1: return launch_shape<K, L, 1, 8, 1>(a, adjoint, extra, st);
    case 2: return launch_shape<K, L, 1, 8, 2>(a, adjoint, extra, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

template <int K> hipError_t launch_tile_k(const StepArgs &a, int L, bool adjoint, bool extra, hipStream_t st);

template <>
hipError_t launch_tile_k<DN_TILE_K>(const StepArgs &a, int L, bool adjoint, bool extra, hipStream_t st)
{
    switch (L) {
    case 0: return launch_kl<DN_TILE_K, 0>(a, adjoint, extra, st);
    case 1: return launch_kl<DN_TILE_K, 1>(a, adjoint, extra, st);
    case 2: return launch_kl<DN_TILE_K, 2>(a, adjoint, extra, st);
    case 3: return launch_kl<DN_TILE_K, 3>(a, adjoint, extra, st);
    case 4: return launch_kl<DN_TILE_K, 4>(a, adjoint, extra, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace dn
