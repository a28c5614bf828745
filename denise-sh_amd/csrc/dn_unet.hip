// Kernels of the learned diagonal-Hessian preconditioner: a 4-level U-Net of
// 3x3 convolutions in BF16 with FP32 accumulation on the CDNA4 matrix cores
// (v_mfma_f32_16x16x32_bf16), stored channels-last ([n][H][W][C], C a
// multiple of 16), plus the pooling, upsampling, loss and Adam kernels of
// its training.  Host side: dn_unet.cpp.
#include "dn_unet.h"

#include <algorithm>

namespace dn {

typedef float f4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t u_f2bf(float x)
{
    // round to nearest even (finite inputs)
    unsigned int u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float u_bf2f(uint16_t h) { return __uint_as_float(((unsigned int)h) << 16); }

// 8 BF16 values: one 16-byte MFMA operand per lane
typedef unsigned short u8v __attribute__((ext_vector_type(8)));
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f4v mfma32(u8v a, u8v b, f4v c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8v, a), __builtin_bit_cast(bf8v, b), c, 0, 0,
                                                   0);
}

// ---------------------------------------------------------------------------
// 3x3 "same" convolution as an implicit GEMM on MFMA 16x16x32 (bf16 in, fp32
// accumulate): D[co][px] = sum over k = (tap, ci) of W[tap][co][ci] *
// X[px + shift(tap)][ci].  K is walked in groups of 8 input channels of one
// tap; one MFMA takes 4 groups: lane quarter kq = lane / 16 supplies group
// 4i + kq, A = W[tap][co = lane % 16][8 channels] and B = X[pixel lane % 16
// + shift][8 channels] (16 bytes each), and receives D[4kq + r][lane % 16],
// r = 0..3.  The weights of groups past the last tap are zero.
//
// The layers move 2 (CI + Co) bytes per pixel for 18 CI Co operations: at 16
// channels 72 operations per byte, so the bytes bound them, if enough loads
// are in flight.  A wave owns 16 NT columns and up to 16 NM output channels
// and walks down a strip of rows: each input row is loaded once, while the
// row before it is multiplied, and enters the accumulators of the three
// output rows it belongs to, in the order ky = 0, 1, 2 of the sum.  All nine
// taps' weights are staged in LDS once, so the walk has no barrier.  One row
// per workgroup, each row's weights staged and waited for and each input row
// loaded for three output rows, took 118 us for 16 -> 16 channels at 800 x
// 4000 and 168 us for 80 -> 32 at half of it; now 47 us (4.4 TB/s) and 81.
//
// CAT: the input is the concatenation of an up-sampled tensor (CU channels at
// half resolution, nearest) and a skip tensor, read from both where they are:
// the concatenated copy (243 us per layer at 800 x 4000) is never written.
// The groups stay in the order of the concatenated channels, so the sums round
// as those over a concatenated copy; with all groups of one part first, without
// the second loads, 48 -> 16 took 95 us instead of 105, but every activation
// behind it may round to another bfloat16.
// ---------------------------------------------------------------------------
constexpr int cat_up(int CI) { return CI == 112 ? 64 : (CI == 80 ? 48 : 32); }
// groups 4i..4i+3 of cb groups per tap, the first b0 of them up-sampled: does
// MFMA i read up-sampled (up) or skip channels; how many MFMAs below n read both
constexpr bool cat_reads(int i, int cb, int b0, bool up)
{
    for (int g = 4 * i; g < 4 * i + 4 && g < 3 * cb; ++g)
        if ((g % cb < b0) == up) return true;
    return false;
}
constexpr int cat_both(int n, int cb, int b0)
{
    int k = 0;
    for (int i = 0; i < n; ++i) k += cat_reads(i, cb, b0, true) && cat_reads(i, cb, b0, false);
    return k;
}

// One row of a tensor as a buffer resource: an offset outside [0, bytes)
// reads zero and stores nothing, which is the convolution's padding, without
// a branch (behind a branch the compiler waits for every access in flight).
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t row_rsrc(const void *p, int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, 0x00027000);
}
typedef unsigned int u4v __attribute__((ext_vector_type(4)));
typedef unsigned int u2v __attribute__((ext_vector_type(2)));

template <int CI, int NM, int NT, bool CAT>
__global__ __launch_bounds__(256, 2) void k_conv3x3(ConvArgs a)
{
    // the input's parts: the up-sampled and the skip tensor, or one tensor
    constexpr int C0 = CAT ? cat_up(CI) : CI, C1 = CI - C0;
    constexpr int CB = CI / 8, B0 = C0 / 8;      // 8-channel groups per tap, of the first part
    constexpr int NKI = (3 * CB + 3) / 4;        // MFMAs per kernel row
    constexpr int N2 = cat_both(NKI, CB, B0);    // of them with groups of both parts
    constexpr int SW = 16 * NM + 1;     // LDS entries per group (+ 1 against bank conflicts)
    __shared__ u8v sw[3 * NKI * 4 * SW];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nl = lane & 15, kq = lane >> 4;
    const int strip = a.strip0 + (int)blockIdx.y, img = strip / a.hblocks, hb = strip - img * a.hblocks;
    const int y0 = (hb * 4 + wave) * a.rows, y1 = min(y0 + a.rows, a.H);   // output rows of the wave
    const int x0 = blockIdx.x * (16 * NT);
    const int cg = blockIdx.z * (16 * NM);
    const int nmt = min(NM, (a.Co - cg) >> 4);
    for (int e = threadIdx.x; e < 3 * NKI * 4 * 16 * NM; e += 256) {
        const int co = e % (16 * NM), kg = e / (16 * NM);      // kg = ky * 4 NKI + group
        const int ky = kg / (4 * NKI), g = kg - ky * (4 * NKI);
        u8v v = u8v{0, 0, 0, 0, 0, 0, 0, 0};
        if (g < 3 * CB && cg + co < a.Co) {
            const int kx = g / CB, cb = g - kx * CB;
            v = *(const u8v *)(a.w + ((long long)(3 * ky + kx) * a.Co + cg + co) * CI + 8 * cb);
        }
        sw[kg * SW + co] = v;
    }
    float bias[NM][4];
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int co = cg + m * 16 + 4 * kq + r;
            bias[m][r] = (a.bias && co < a.Co) ? a.bias[co] : 0.0f;
        }
    __syncthreads();
    if (y0 >= y1) return;

    // input fragment i, t of row yi: the groups of the one part; those of the
    // other part and past the last tap read zero
    auto load = [&](int yi, int i, int t, bool up) -> u8v {
        const int g = 4 * i + kq, kx = g / CB, cb = g - kx * CB, px = x0 + 16 * t + nl + kx - 1;
        const bool half = CAT && up;               // the part at half resolution
        const int w = half ? a.W >> 1 : a.W, c = up ? C0 : C1;
        const uint16_t *row = half ? a.up + (long long)(img * (a.H >> 1) + (yi >> 1)) * w * c
                                   : a.x + (long long)(img * a.H + yi) * w * c;
        // px >> 1: -1 stays -1, W becomes W / 2
        int off = ((half ? px >> 1 : px) * c + 8 * (up ? cb : cb - B0)) * 2;
        if (CAT && (cb < B0) != up) off = -16;
        if (4 * NKI > 3 * CB && g >= 3 * CB) off = -16;
        return __builtin_bit_cast(u8v, __builtin_amdgcn_raw_buffer_load_b128(row_rsrc(row, w * c * 2), off, 0, 0));
    };
    // An MFMA whose groups are of both parts takes the union of two loads: the
    // sum keeps the order of the concatenated channels.
    u8v b[NKI][NT], b2[N2 > 0 ? N2 : 1][NT];
    auto fetch = [&](int yi, int i) {
        const bool up = cat_reads(i, CB, B0, true);
#pragma unroll
        for (int t = 0; t < NT; ++t) b[i][t] = load(yi, i, t, up);
        if (up && cat_reads(i, CB, B0, false)) {
#pragma unroll
            for (int t = 0; t < NT; ++t) b2[cat_both(i, CB, B0)][t] = load(yi, i, t, false);
        }
    };
    f4v acc[3][NM][NT];
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[q][m][t] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    const int ya = max(y0 - 1, 0), yb = min(y1, a.H - 1);      // input rows
#pragma unroll
    for (int i = 0; i < NKI; ++i) fetch(ya, i);

    const int orow = a.W * a.Co * 2;                           // bytes of an output (or mask) row
    auto ooff = [&](int t, int m) -> int { return ((x0 + 16 * t + nl) * a.Co + cg + m * 16 + 4 * kq) * 2; };
    auto finish = [&](int y, f4v (&ac)[NM][NT], const u2v (&mk)[NM][NT]) {
        const long long row = (long long)(img * a.H + y) * a.W;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                if (m < nmt) {
                    float v[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        v[r] = ac[m][t][r] + bias[m][r];
                        if (a.relu) v[r] = fmaxf(v[r], 0.0f);
                    }
                    if (a.mask) {
                        if (!(u_bf2f((uint16_t)(mk[m][t].x & 0xffffu)) > 0.0f)) v[0] = 0.0f;
                        if (!(u_bf2f((uint16_t)(mk[m][t].x >> 16)) > 0.0f)) v[1] = 0.0f;
                        if (!(u_bf2f((uint16_t)(mk[m][t].y & 0xffffu)) > 0.0f)) v[2] = 0.0f;
                        if (!(u_bf2f((uint16_t)(mk[m][t].y >> 16)) > 0.0f)) v[3] = 0.0f;
                    }
                    if (a.y16) {
                        const u2v o = u2v{(unsigned)u_f2bf(v[0]) | ((unsigned)u_f2bf(v[1]) << 16),
                                          (unsigned)u_f2bf(v[2]) | ((unsigned)u_f2bf(v[3]) << 16)};
                        __builtin_amdgcn_raw_buffer_store_b64(o, row_rsrc(a.y16 + row * a.Co, orow), ooff(t, m), 0, 0);
                    }
                    if (a.y1 && m == 0) {   // channel 0: lanes kq 0 of the first tile
                        const int off = (kq == 0 && cg == 0) ? (x0 + 16 * t + nl) * 4 : -4;
                        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[0]), row_rsrc(a.y1 + row, a.W * 4), off, 0, 0);
                    }
                }
                ac[m][t] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
            }
    };
    // the ReLU mask of output row y, asked for before the next input row
    auto masks = [&](int y, u2v (&mk)[NM][NT]) {
        const rsrc_t rs = row_rsrc(a.mask ? a.mask + (long long)(img * a.H + max(y, 0)) * a.W * a.Co : a.w, a.mask ? orow : 0);
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int t = 0; t < NT; ++t)
                if (m < nmt) mk[m][t] = __builtin_amdgcn_raw_buffer_load_b64(rs, ooff(t, m), 0, 0);
    };
    // one input row: output rows yi+1 (ky 0), yi (ky 1), yi-1 (ky 2, complete
    // after it) in the accumulators a0, a1, a2
    auto step = [&](int yi, f4v (&a0)[NM][NT], f4v (&a1)[NM][NT], f4v (&a2)[NM][NT]) {
        const bool d0 = yi + 1 < y1, d1 = yi >= y0 && yi < y1, d2 = yi - 1 >= y0;   // uniform
        const int yn = min(yi + 1, yb);
        u2v mk[NM][NT];
        if (a.mask) masks(yi - 1, mk);
#pragma unroll
        for (int i = 0; i < NKI; ++i) {
            if (cat_reads(i, CB, B0, true) && cat_reads(i, CB, B0, false)) {
#pragma unroll
                for (int t = 0; t < NT; ++t) b[i][t] |= b2[cat_both(i, CB, B0)][t];
            }
            auto mult = [&](int ky, f4v (&ac)[NM][NT]) {
                const u8v *w = sw + (ky * 4 * NKI + 4 * i + kq) * SW + nl;
#pragma unroll
                for (int m = 0; m < NM; ++m)
                    if (m < nmt) {
                        const u8v av = w[16 * m];
#pragma unroll
                        for (int t = 0; t < NT; ++t) ac[m][t] = mfma32(av, b[i][t], ac[m][t]);
                    }
            };
            if (d0) mult(0, a0);
            if (d1) mult(1, a1);
            if (d2) mult(2, a2);
            fetch(yn, i);
        }
        if (d2) finish(yi - 1, a2, mk);
    };
    auto last = [&](int y, f4v (&ac)[NM][NT]) {               // the image's last row
        u2v mk[NM][NT];
        if (a.mask) masks(y, mk);
        finish(y, ac, mk);
    };
    // the accumulators take turns: after a row, a2's is free for row yi+2
    int yi = ya;
    for (; yi + 2 <= yb; yi += 3) {
        step(yi, acc[0], acc[1], acc[2]);
        step(yi + 1, acc[2], acc[0], acc[1]);
        step(yi + 2, acc[1], acc[2], acc[0]);
    }
    if (yi <= yb) {
        step(yi, acc[0], acc[1], acc[2]);
        if (yi + 1 <= yb) {
            step(yi + 1, acc[2], acc[0], acc[1]);
            if (yb == y1 - 1) last(yb, acc[0]);
        } else if (yb == y1 - 1) {
            last(yb, acc[1]);
        }
    } else if (yb == y1 - 1) {
        last(yb, acc[2]);
    }
}

// The second dimension of a grid takes 65536 workgroups; the rows (strips,
// images) of a large batch go in several launches: f(first, count).  With the
// rows in the first dimension, where one launch takes them all, 16 -> 32
// channels took 20.4 us instead of 17.7 and k_pool_bwd<16> 48 instead of 44
// (4 x 304 x 1200).
template <typename F> static hipError_t by_grid_y(long long rows, F f)
{
    constexpr long long kMost = 65535;
    for (long long r0 = 0; r0 < rows; r0 += kMost) {
        const hipError_t e = f(r0, (unsigned)std::min(kMost, rows - r0));
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int CI, int NM, int NT, bool CAT> static hipError_t conv_launch(ConvArgs a, hipStream_t st)
{
    // rows per wave: a strip of R rows loads R + 2; shorter where the image
    // would leave CUs without a workgroup
    const int cols = (a.W + 16 * NT - 1) / (16 * NT), z = (a.Co + 16 * NM - 1) / (16 * NM);
    int R = 12;
    while (R > 2 && (long long)cols * z * a.n * ((a.H + 4 * R - 1) / (4 * R)) < 1024) R /= 2;
    a.rows = R;
    a.hblocks = (a.H + 4 * R - 1) / (4 * R);
    return by_grid_y((long long)a.n * a.hblocks, [&](long long s0, unsigned strips) {
        a.strip0 = (int)s0;
        hipLaunchKernelGGL((k_conv3x3<CI, NM, NT, CAT>), dim3((unsigned)cols, strips, (unsigned)z), dim3(256), 0, st, a);
        return hipGetLastError();
    });
}

hipError_t launch_conv3x3(const ConvArgs &a, hipStream_t st)
{
    if (a.Co % 16 || a.Co < 16 || a.n < 1 || a.H < 1 || a.W < 1) return hipErrorInvalidValue;
    if (a.up && ((a.H | a.W) & 1)) return hipErrorInvalidValue;
    // output channel tiles per wave: all of them up to four, 5 as 3 + 2, 7 as 4 + 3
    // (112 input channels: one, its weights would fill the LDS of a CU)
    const int tiles = a.Co / 16, nm = a.Ci == 112 ? 1 : (tiles <= 4 ? tiles : (tiles == 5 ? 3 : 4));
    switch ((a.up ? 10000 : 0) + a.Ci * 10 + nm) {   // the layers and their data gradients
    case 161: return conv_launch<16, 1, 4, false>(a, st);
    case 162: return conv_launch<16, 2, 2, false>(a, st);
    case 163: return conv_launch<16, 3, 2, false>(a, st);
    case 321: return conv_launch<32, 1, 4, false>(a, st);
    case 322: return conv_launch<32, 2, 2, false>(a, st);
    case 323: return conv_launch<32, 3, 2, false>(a, st);
    case 482: return conv_launch<48, 2, 2, false>(a, st);
    case 483: return conv_launch<48, 3, 2, false>(a, st);
    case 484: return conv_launch<48, 4, 2, false>(a, st);
    case 643: return conv_launch<64, 3, 2, false>(a, st);
    case 644: return conv_launch<64, 4, 2, false>(a, st);
    case 10481: return conv_launch<48, 1, 2, true>(a, st);
    case 10802: return conv_launch<80, 2, 2, true>(a, st);
    case 11121: return conv_launch<112, 1, 2, true>(a, st);
    default: return hipErrorInvalidValue;
    }
}

// ---------------------------------------------------------------------------
// Weight gradient dW[tap][co][ci] = sum_p dY[p][co] * X[p + shift(tap)][ci]
// as a GEMM over pixels (K) on MFMA 16x16x32, with the bias gradient
// db[co] = sum_p dY[p][co] (an operand of ones).  A workgroup (4 waves) walks
// down rows y0..y1-1 of one image in a column segment of 128 pixels.  The
// rows are staged in LDS as they lie in memory (channels last, 16-byte
// accesses, loaded a row ahead) and read back transposed, four pixels of one
// channel per lane, by ds_read_b64_tr_b16: A = dY^T (co = lane % 16) and
// B = X (ci = lane % 16), 8 pixels per lane quarter, the taps as pixel and row
// offsets.  Wave w multiplies pixels 32 w..32 w + 31 into all the workgroup's
// tiles; their sum over the waves, in wave order, is the workgroup's partial,
// and the partials are added in order (deterministic).
//
// Bytes bound it where one workgroup takes all nine taps (KYS 1: the X rows
// rotate through three LDS slots and are loaded once); where the accumulators
// allow three taps only (KYS 3) blockIdx.y selects ky, and blockIdx.z a group
// of NTB input-channel tiles.  Transposing by 2-byte LDS stores, each X row
// stored for three kx and loaded for three ky, took 140 us (16 -> 16 channels,
// 4 x 304 x 1200) and 312 us (48 -> 16); now 25 and 49.  Of the layers only
// 112 -> 48 spills: 8 registers, 20 bytes per lane.
// ---------------------------------------------------------------------------
constexpr int kSegPx = 128;    // pixels per segment

typedef short s4v __attribute__((ext_vector_type(4)));

// 8 pixels (rows of `pitch` elements) of 16 channels, transposed: p points at
// the lane's 4 channels of its pixel, see tr_lane
__device__ __forceinline__ u8v tr_read(const uint16_t *p, int pitch)
{
    typedef __attribute__((address_space(3))) s4v *lds_t;
    const s4v a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)p);
    const s4v b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(p + 4 * pitch));
    return u8v{(unsigned short)a.x, (unsigned short)a.y, (unsigned short)a.z, (unsigned short)a.w,
               (unsigned short)b.x, (unsigned short)b.y, (unsigned short)b.z, (unsigned short)b.w};
}

constexpr bool wgrad_cat(int CI, int CO) { return CI >= 80 || (CI == 48 && CO == 16); }

template <int CI, int CO, int KYS, int NTB>
__global__ __launch_bounds__(256, 2) void k_wgrad(WgradArgs a)
{
    constexpr bool CAT = wgrad_cat(CI, CO);              // the input is [up-sampled | skip]
    constexpr int NMT = CO / 16, NNT = CI / 16, TAPS = 9 / KYS, NR = KYS == 1 ? 3 : 1;
    constexpr int CW = 16 * NTB, BW = CW / 8;            // input channels of the workgroup
    constexpr int XP = kSegPx + 2;                       // X pixels per row (x0 - 1 .. x0 + 128)
    constexpr int ND = (kSegPx * (CO / 8) + 255) / 256, NX = (XP * BW + 255) / 256;
    constexpr int NTILE = TAPS * NMT * NTB;
    constexpr int RED = 4;                               // tiles summed over the waves per turn
    constexpr int SXN = NR * XP * CW, SDN = kSegPx * CO;
    __shared__ __attribute__((aligned(16))) uint16_t lds[SXN + SDN > RED * 4 * 512 ? SXN + SDN : RED * 4 * 512];
    uint16_t *sx = lds, *sdy = lds + SXN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nl = lane & 15, kq = lane >> 4;
    const int ky0 = KYS == 1 ? 0 : blockIdx.y, c8g = blockIdx.z * BW;
    const int seg = blockIdx.x % a.nseg, chunk = blockIdx.x / a.nseg;
    const int img = chunk / a.hchunks, y0 = (chunk - img * a.hchunks) * a.chunk_rows;
    const int y1 = min(y0 + a.chunk_rows, a.H), x0 = seg * kSegPx;
    f4v acc[TAPS][NMT][NTB], accb[NMT];
#pragma unroll
    for (int m = 0; m < NMT; ++m) {
        accb[m] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int p = 0; p < TAPS; ++p)
#pragma unroll
            for (int t = 0; t < NTB; ++t) acc[p][m][t] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    }
    u8v rd[ND], rx[NX];
    // zero outside the row (buffer range) and, by an empty range, for a row
    // outside the image
    auto fetch_x = [&](int yy) {
        const bool in = yy >= 0 && yy < a.H;
        const long long xr = in ? (long long)(img * a.H + yy) : 0;
        constexpr int CU = CAT ? cat_up(CI) : 0, CS = CI - CU;
        const rsrc_t s0 = row_rsrc(a.x + xr * a.W * CS, in ? a.W * CS * 2 : 0);
        if (!CAT) {
#pragma unroll
            for (int k = 0; k < NX; ++k) {
                const int e = (int)threadIdx.x + 256 * k, jj = e / BW, c8 = c8g + e - jj * BW;
                const int off = c8 < CI / 8 ? ((x0 + jj - 1) * CI + 8 * c8) * 2 : -16;
                rx[k] = __builtin_bit_cast(u8v, __builtin_amdgcn_raw_buffer_load_b128(s0, off, 0, 0));
            }
        } else {   // up-sampled and skip channels, as in k_conv3x3: one of the two reads zero
            const long long ur = in ? (long long)(img * (a.H >> 1) + (yy >> 1)) : 0;
            const int wu = a.W >> 1;
            const rsrc_t su = row_rsrc(a.up + ur * wu * CU, in ? wu * CU * 2 : 0);
#pragma unroll
            for (int k = 0; k < NX; ++k) {
                const int e = (int)threadIdx.x + 256 * k, jj = e / BW, c8 = c8g + e - jj * BW, px = x0 + jj - 1;
                const bool up = c8 < CU / 8, skip = !up && c8 < CI / 8;
                const u8v vu = __builtin_bit_cast(
                    u8v, __builtin_amdgcn_raw_buffer_load_b128(su, up ? ((px >> 1) * CU + 8 * c8) * 2 : -16, 0, 0));
                const u8v vs = __builtin_bit_cast(
                    u8v, __builtin_amdgcn_raw_buffer_load_b128(s0, skip ? (px * CS + 8 * c8 - CU) * 2 : -16, 0, 0));
                rx[k] = vu | vs;
            }
        }
    };
    auto fetch_d = [&](int y) {
        const rsrc_t sd = row_rsrc(a.dy + (long long)(img * a.H + y) * a.W * CO, a.W * CO * 2);
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            const int e = (int)threadIdx.x + 256 * k, j = e / (CO / 8), c8 = e - j * (CO / 8);
            const int off = j < kSegPx ? ((x0 + j) * CO + 8 * c8) * 2 : -16;
            rd[k] = __builtin_bit_cast(u8v, __builtin_amdgcn_raw_buffer_load_b128(sd, off, 0, 0));
        }
    };
    auto store_x = [&](int slot) {
#pragma unroll
        for (int k = 0; k < NX; ++k) {
            const int e = (int)threadIdx.x + 256 * k;
            if (e < XP * BW) *(u8v *)(sx + slot * (XP * CW) + 8 * e) = rx[k];
        }
    };
    auto store_d = [&]() {
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            const int e = (int)threadIdx.x + 256 * k;
            if (e < kSegPx * (CO / 8)) *(u8v *)(sdy + 8 * e) = rd[k];
        }
    };
    // the transposed read's lane: lanes 4 r + q of a quarter supply channels
    // 4 q.. of pixel r, lane n receives channel n of pixels 0..3
    const int tp = 32 * wave + 8 * kq + (nl >> 2), tc = 4 * (nl & 3);
    if (KYS == 1) {
        // rows y0 - 1 and y0; row yy lives in slot (yy + 3) % 3
        fetch_x(y0 - 1);
        store_x((y0 + 2) % 3);
        fetch_x(y0);
        store_x(y0 % 3);
    }
    fetch_x(KYS == 1 ? y0 + 1 : y0 + ky0 - 1);
    fetch_d(y0);
    const u8v ones = u8v{0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80};
    for (int y = y0; y < y1; ++y) {
        __syncthreads();   // the row before is consumed
        store_x(KYS == 1 ? (y + 1) % 3 : 0);
        store_d();
        __syncthreads();
        // the next row's loads go out before this one is multiplied
        const int yn = min(y + 1, y1 - 1);
        fetch_x(KYS == 1 ? yn + 1 : yn + ky0 - 1);
        fetch_d(yn);
        u8v av[NMT];
#pragma unroll
        for (int m = 0; m < NMT; ++m) {
            av[m] = tr_read(sdy + tp * CO + 16 * m + tc, CO);
            if (ky0 == 0 && blockIdx.z == 0) accb[m] = mfma32(av[m], ones, accb[m]);
        }
#pragma unroll
        for (int p = 0; p < TAPS; ++p) {
            const int kx = p % 3, slot = KYS == 1 ? (y + p / 3 + 2) % 3 : 0;   // row y + ky - 1
            const uint16_t *bx = sx + slot * (XP * CW) + (tp + kx) * CW + tc;
#pragma unroll
            for (int t = 0; t < NTB; ++t) {
                const u8v bv = tr_read(bx + 16 * t, CW);
#pragma unroll
                for (int m = 0; m < NMT; ++m) acc[p][m][t] = mfma32(av[m], bv, acc[p][m][t]);
            }
        }
    }
    // sums over the waves, RED tiles per turn; element (lane, j) of a tile is
    // co = 16 m + 4 (lane / 16) + j, ci = lane % 16
    float *red = (float *)lds;
    auto turn = [&](int tile0, int nt, auto get, auto put) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < RED; ++q)
            if (q < nt) *(f4v *)(red + ((q * 4 + wave) * 64 + lane) * 4) = get(tile0 + q);
        __syncthreads();
        const int e = threadIdx.x;
#pragma unroll
        for (int q = 0; q < RED; ++q)
            if (q < nt) {
                const float *r = red + q * 1024 + e;
                put(tile0 + q, ((r[0] + r[256]) + r[512]) + r[768]);
            }
    };
    const int el = threadIdx.x >> 2, ej = threadIdx.x & 3;
    float *part = a.part + (long long)blockIdx.x * 9 * CO * CI;
#pragma unroll
    for (int t0 = 0; t0 < NTILE; t0 += RED)
        turn(t0, NTILE - t0 < RED ? NTILE - t0 : RED,
             [&](int q) { return acc[q / (NMT * NTB)][q / NTB % NMT][q % NTB]; },
             [&](int q, float v) {
                 const int p = q / (NMT * NTB), m = q / NTB % NMT, t = q % NTB;
                 const int tap = KYS == 1 ? p : 3 * ky0 + p;
                 const int co = 16 * m + 4 * (el >> 4) + ej, ci = 8 * c8g + 16 * t + (el & 15);
                 if (NNT % NTB == 0 || ci < CI) part[((long long)tap * CO + co) * CI + ci] = v;
             });
    if (ky0 == 0 && blockIdx.z == 0)
        turn(0, NMT, [&](int q) { return accb[q < NMT ? q : 0]; },
             [&](int q, float v) {
                 if ((el & 15) == 0) a.bpart[(long long)blockIdx.x * CO + 16 * q + 4 * (el >> 4) + ej] = v;
             });
}

// dw[e] = sum over c of part[c][e] and, behind them, db[e] from bpart: four
// waves take a quarter of the partials each, in order, for 64 elements, and
// the quarters are added in order (one wave over all of 512 partials and a
// launch of its own for db: 10.4 + 4.7 us per layer, now 9.3)
__global__ __launch_bounds__(256) void k_reduce_chunks(int nchunks, int len, const float *part, float *dw, int blen,
                                                       const float *bpart, float *db)
{
    __shared__ float sh[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nb = (len + 63) / 64;
    const bool bias = (int)blockIdx.x >= nb;
    const int n = bias ? blen : len, e = ((int)blockIdx.x - (bias ? nb : 0)) * 64 + lane;
    const float *src = (bias ? bpart : part) + min(e, n - 1);
    const int c0 = (int)((long long)nchunks * wave / 4), c1 = (int)((long long)nchunks * (wave + 1) / 4);
    float s = 0.0f;
    int c = c0;
    for (; c + 32 <= c1; c += 32) {   // 32 are read before the first is added
        float p[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) p[k] = src[(long long)(c + k) * n];
#pragma unroll
        for (int k = 0; k < 32; ++k) s += p[k];
    }
    for (; c < c1; ++c) s += src[(long long)c * n];
    sh[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && e < n) (bias ? db : dw)[e] = ((sh[0][lane] + sh[1][lane]) + sh[2][lane]) + sh[3][lane];
}

// the layers' (input, output) channel pairs: taps per workgroup and input
// channel tiles per workgroup, as the accumulators allow
static bool wgrad_all_taps(int Ci, int Co) { return Ci * Co <= 1024; }

// column segments and row chunks: about 512 workgroups of partials (256 where
// blockIdx.y triples them), a chunk within one image
static void wgrad_split(int n, int H, int W, int Ci, int Co, int &nseg, int &hchunks, int &rows)
{
    nseg = (W + kSegPx - 1) / kSegPx;
    const int want = std::max(1, (wgrad_all_taps(Ci, Co) ? 512 : 256) / (nseg * n));
    rows = std::max(1, (H + want - 1) / want);
    hchunks = (H + rows - 1) / rows;
}

int wgrad_chunks(int n, int H, int W, int Ci, int Co)
{
    int nseg, hchunks, rows;
    wgrad_split(n, H, W, Ci, Co, nseg, hchunks, rows);
    return n * nseg * hchunks;
}

template <int CI, int CO, int KYS, int NTB> static void wgrad_launch(const WgradArgs &a, int nch, hipStream_t st)
{
    constexpr int Z = (CI / 16 + NTB - 1) / NTB;
    static_assert((KYS == 1) == (CI * CO <= 1024), "as wgrad_all_taps");
    hipLaunchKernelGGL((k_wgrad<CI, CO, KYS, NTB>), dim3(nch, KYS, Z), dim3(256), 0, st, a);
}

hipError_t launch_wgrad(WgradArgs a, float *dw, float *db, hipStream_t st)
{
    if (a.n < 1 || a.H < 1 || a.W < 1 || (a.up && ((a.H | a.W) & 1))) return hipErrorInvalidValue;
    wgrad_split(a.n, a.H, a.W, a.Ci, a.Co, a.nseg, a.hchunks, a.chunk_rows);
    const int nch = wgrad_chunks(a.n, a.H, a.W, a.Ci, a.Co);
    switch ((a.up ? 1000000 : 0) + a.Ci * 1000 + a.Co) {   // the network's layers
    case 16016: wgrad_launch<16, 16, 1, 1>(a, nch, st); break;
    case 16032: wgrad_launch<16, 32, 1, 1>(a, nch, st); break;
    case 32032: wgrad_launch<32, 32, 1, 2>(a, nch, st); break;
    case 32048: wgrad_launch<32, 48, 3, 2>(a, nch, st); break;
    case 48048: wgrad_launch<48, 48, 3, 3>(a, nch, st); break;
    case 48064: wgrad_launch<48, 64, 3, 3>(a, nch, st); break;
    case 64064: wgrad_launch<64, 64, 3, 2>(a, nch, st); break;
    case 1112048: wgrad_launch<112, 48, 3, 4>(a, nch, st); break;
    case 1080032: wgrad_launch<80, 32, 3, 5>(a, nch, st); break;
    case 1048016: wgrad_launch<48, 16, 1, 3>(a, nch, st); break;
    default: return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int len = 9 * a.Co * a.Ci;
    hipLaunchKernelGGL(k_reduce_chunks, dim3((unsigned)((len + 63) / 64 + (a.Co + 63) / 64)), dim3(256), 0, st, nch, len,
                       a.part, dw, a.Co, a.bpart, db);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// 2x2 average pooling and the adjoints of pooling and nearest upsampling with
// the ReLU mask of the activation they feed.  Bytes only: one thread per 8
// channels of a pixel (16-byte accesses), one image row per blockIdx.y, so
// the only division is by the channel count, a constant.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void unpack8(const uint16_t *p, float (&f)[8])
{
    const u8v v = *(const u8v *)p;
#pragma unroll
    for (int k = 0; k < 8; ++k) f[k] = u_bf2f(v[k]);
}

template <int C> __global__ void k_pool(long long row0, int H, int W, const uint16_t *x, uint16_t *y)
{
    constexpr int C8 = C / 8;
    const int w = W / 2, e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= w * C8) return;
    const int xo = e / C8, c = 8 * (e - xo * C8);
    const long long row = row0 + blockIdx.y;              // image * H/2 + y
    const uint16_t *b = x + ((2 * row * W + 2 * xo) * C + c);
    float p[8], q[8], r[8], t[8];
    unpack8(b, p);
    unpack8(b + C, q);
    unpack8(b + (long long)W * C, r);
    unpack8(b + (long long)W * C + C, t);
    u8v o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = u_f2bf(0.25f * ((p[k] + q[k]) + (r[k] + t[k])));
    *(u8v *)(y + (row * w + xo) * C + c) = o;
}

// dact[p][c] = (act > 0) * (0.25 * dpool[p/2][c] + dcat[p][off + c])
template <int C>
__global__ void k_pool_bwd(long long row0, int H, int W, const uint16_t *dpool, const uint16_t *dcat, int ccat,
                           int off, const uint16_t *act, uint16_t *dact)
{
    constexpr int C8 = C / 8;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= W * C8) return;
    const int x = e / C8, c = 8 * (e - x * C8);
    const long long row = row0 + blockIdx.y, p = row * W + x;   // row: image * H + y
    const long long img = row / H, yl = (row - img * H) / 2;
    float dp[8], dc[8], ac[8];
    unpack8(dpool + ((img * (H / 2) + yl) * (W / 2) + x / 2) * C + c, dp);
    unpack8(dcat + p * ccat + off + c, dc);
    unpack8(act + p * C + c, ac);
    u8v o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = ac[k] > 0.0f ? u_f2bf(0.25f * dp[k] + dc[k]) : (uint16_t)0;
    *(u8v *)(dact + p * C + c) = o;
}

// dlow[q][c] = (act_low > 0) * sum over the 2x2 children of dcat[child][c], c < CU
template <int CU>
__global__ void k_up_bwd(long long row0, int H, int W, int Ccat, const uint16_t *dcat, const uint16_t *act_low,
                         uint16_t *dlow)
{
    constexpr int C8 = CU / 8;
    const int w = W / 2, e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= w * C8) return;
    const int xo = e / C8, c = 8 * (e - xo * C8);
    const long long row = row0 + blockIdx.y;              // image * H/2 + y
    const uint16_t *b = dcat + ((2 * row * W + 2 * xo) * Ccat + c);
    const long long q = (row * w + xo) * CU + c;
    float p0[8], p1[8], p2[8], p3[8], ac[8];
    unpack8(b, p0);
    unpack8(b + Ccat, p1);
    unpack8(b + (long long)W * Ccat, p2);
    unpack8(b + (long long)W * Ccat + Ccat, p3);
    unpack8(act_low + q, ac);
    u8v o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = ac[k] > 0.0f ? u_f2bf((p0[k] + p1[k]) + (p2[k] + p3[k])) : (uint16_t)0;
    *(u8v *)(dlow + q) = o;
}

static dim3 grid_for(long long total)
{
    return dim3((unsigned)std::max<long long>(1, std::min<long long>(8192, (total + 255) / 256)));
}

hipError_t launch_pool(int n, int H, int W, int C, const uint16_t *x, uint16_t *y, hipStream_t st)
{
    const unsigned nb = (unsigned)((W / 2 * (C / 8) + 255) / 256);
    return by_grid_y((long long)n * (H / 2), [&](long long r0, unsigned rows) {
        const dim3 g(nb, rows);
        switch (C) {
        case 16: hipLaunchKernelGGL(k_pool<16>, g, dim3(256), 0, st, r0, H, W, x, y); break;
        case 32: hipLaunchKernelGGL(k_pool<32>, g, dim3(256), 0, st, r0, H, W, x, y); break;
        case 48: hipLaunchKernelGGL(k_pool<48>, g, dim3(256), 0, st, r0, H, W, x, y); break;
        default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    });
}
hipError_t launch_pool_bwd(int n, int H, int W, int C, const uint16_t *dpool, const uint16_t *dcat, int ccat, int off,
                           const uint16_t *act, uint16_t *dact, hipStream_t st)
{
    const unsigned nb = (unsigned)((W * (C / 8) + 255) / 256);
    return by_grid_y((long long)n * H, [&](long long r0, unsigned rows) {
        const dim3 g(nb, rows);
        switch (C) {
        case 16: hipLaunchKernelGGL(k_pool_bwd<16>, g, dim3(256), 0, st, r0, H, W, dpool, dcat, ccat, off, act, dact); break;
        case 32: hipLaunchKernelGGL(k_pool_bwd<32>, g, dim3(256), 0, st, r0, H, W, dpool, dcat, ccat, off, act, dact); break;
        case 48: hipLaunchKernelGGL(k_pool_bwd<48>, g, dim3(256), 0, st, r0, H, W, dpool, dcat, ccat, off, act, dact); break;
        default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    });
}
hipError_t launch_up_bwd(int n, int H, int W, int Cu, int Ccat, const uint16_t *dcat, const uint16_t *act_low,
                         uint16_t *dlow, hipStream_t st)
{
    const unsigned nb = (unsigned)((W / 2 * (Cu / 8) + 255) / 256);
    return by_grid_y((long long)n * (H / 2), [&](long long r0, unsigned rows) {
        const dim3 g(nb, rows);
        switch (Cu) {
        case 32: hipLaunchKernelGGL(k_up_bwd<32>, g, dim3(256), 0, st, r0, H, W, Ccat, dcat, act_low, dlow); break;
        case 48: hipLaunchKernelGGL(k_up_bwd<48>, g, dim3(256), 0, st, r0, H, W, Ccat, dcat, act_low, dlow); break;
        case 64: hipLaunchKernelGGL(k_up_bwd<64>, g, dim3(256), 0, st, r0, H, W, Ccat, dcat, act_low, dlow); break;
        default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    });
}

// ---------------------------------------------------------------------------
// Input packing, output extraction, loss, parameter casts and Adam
// ---------------------------------------------------------------------------
// x [n][3][H][W] fp32 (planar) -> [n][H][W][16] bf16 with channels 3..15
// zero: one pixel per thread
__global__ void k_pack_input(long long im0, long long hw, const float *x, uint16_t *xp)
{
    const long long r = blockIdx.x * (long long)blockDim.x + threadIdx.x, im = im0 + blockIdx.y;
    if (r >= hw) return;
    const float *b = x + im * 3 * hw + r;
    const u8v z = u8v{0, 0, 0, 0, 0, 0, 0, 0};
    u8v v = z;
    v[0] = u_f2bf(b[0]);
    v[1] = u_f2bf(b[hw]);
    v[2] = u_f2bf(b[2 * hw]);
    u8v *o = (u8v *)(xp + (im * hw + r) * 16);
    o[0] = v;
    o[1] = z;
}

// loss = mean (y[p] - t[p])^2 ; dy[p][c] = c == 0 ? 2 (y - t) / P : 0
__global__ void k_mse(long long P, const float *y, const float *t, uint16_t *dy, double *part)
{
    __shared__ double sh[256];
    double acc = 0.0;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < P; p += (long long)gridDim.x * blockDim.x) {
        const float d = y[p] - t[p];
        acc += (double)d * (double)d;
        if (dy) {
            const u8v z = u8v{0, 0, 0, 0, 0, 0, 0, 0};
            u8v v = z;
            v[0] = u_f2bf(2.0f * d / (float)P);
            u8v *o = (u8v *)(dy + p * 16);
            o[0] = v;
            o[1] = z;
        }
    }
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// fp32 master W [9][Co][Ci] -> bf16 W and bf16 W^T for the data gradient:
// wt[8 - tap][ci][co] = w[tap][co][ci]
__global__ void k_cast_weights(int Co, int Ci, const float *w32, uint16_t *w16, uint16_t *wt16)
{
    const long long total = 9LL * Co * Ci;
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int ci = (int)(e % Ci);
        const int co = (int)((e / Ci) % Co);
        const int tap = (int)(e / ((long long)Ci * Co));
        const uint16_t v = u_f2bf(w32[e]);
        w16[e] = v;
        wt16[((long long)(8 - tap) * Ci + ci) * Co + co] = v;
    }
}

__global__ void k_adam(long long n, float *w, const float *g, float *m, float *v, float lr_t, float b1, float b2,
                       float eps)
{
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < n; e += (long long)gridDim.x * blockDim.x) {
        const float gi = g[e];
        const float mi = b1 * m[e] + (1.0f - b1) * gi;
        const float vi = b2 * v[e] + (1.0f - b2) * gi * gi;
        m[e] = mi;
        v[e] = vi;
        w[e] = w[e] - lr_t * mi / (sqrtf(vi) + eps);
    }
}

hipError_t launch_pack_input(int n, int H, int W, const float *x, uint16_t *xp, hipStream_t st)
{
    const long long hw = (long long)H * W;
    return by_grid_y(n, [&](long long im0, unsigned images) {
        hipLaunchKernelGGL(k_pack_input, dim3((unsigned)((hw + 255) / 256), images), dim3(256), 0, st, im0, hw, x, xp);
        return hipGetLastError();
    });
}
hipError_t launch_mse(long long P, const float *y, const float *t, uint16_t *dy, double *part, int nblocks,
                      hipStream_t st)
{
    hipLaunchKernelGGL(k_mse, dim3(nblocks), dim3(256), 0, st, P, y, t, dy, part);
    return hipGetLastError();
}
hipError_t launch_cast_weights(int Co, int Ci, const float *w32, uint16_t *w16, uint16_t *wt16, hipStream_t st)
{
    hipLaunchKernelGGL(k_cast_weights, grid_for(9LL * Co * Ci), dim3(256), 0, st, Co, Ci, w32, w16, wt16);
    return hipGetLastError();
}
hipError_t launch_adam(long long n, float *w, const float *g, float *m, float *v, float lr_t, float b1, float b2,
                       float eps, hipStream_t st)
{
    hipLaunchKernelGGL(k_adam, grid_for(n), dim3(256), 0, st, n, w, g, m, v, lr_t, b1, b2, eps);
    return hipGetLastError();
}

}  // namespace dn
