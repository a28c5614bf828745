// Source-time-function estimate by Wiener deconvolution (stf.c:11-250) on
// the device, with the project's own FFT.
//
// For one shot with observed traces d_i, modelled traces m_i (modelled with
// the current source signal s) and Npad = 2^(ceil(log2 ns) + 2):
//   S_n[k] = sum_i ntr D_i[k] conj(M_i[k]),  S_d[k] = sum_i ntr |M_i[k]|^2
//   Ebar   = sum_i sum_k S_d^(i)[k] / (Npad ntr)   (S_d^(i): the running sum
//            after trace i, as stf.c:165-168 accumulates it)
//   STF    = Re IFFT( FFT(s) S_n / (S_d + EPS_STF ntr Ebar) )[0..ns-1]
// Killed and muted traces are zero (stf.c:57-112); NORMALIZE 1 scales each
// trace by its largest |sample| over samples 2..ns, NORMALIZE 2 the observed
// trace to the modelled trace's (util.c:489-579).  The reference transforms
// with FFTW's +1 sign forward and -1 inverse; for real input this gives the
// same real part as the usual convention used here.  Sums run in FP64 in a
// fixed order; the reference accumulates Ebar in float.
//
// FFT: radix-2 decimation in time, a bit-reversal gather then log2(Npad)
// butterfly stages over kBatchPts points at once, complex double.  The stages run
// in LDS, eight in the pass that gathers the traces and up to seven in each
// pass after it: two passes over HBM instead of one per stage for 2^15
// points, with the same butterflies.  The call for 240 traces of 5000 samples
// (Npad 2^15): 2.67 ms with a pass per stage over all traces, 1.29 with these
// over all traces (four launches of about 75 us), 1.03 in batches.
#include "dn_core.h"

#include <algorithm>
#include <cmath>
#include <vector>

using namespace dn;

namespace {

struct cd {
    double re, im;
};

__device__ inline cd cmul(cd a, cd b) { return cd{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }

// w[k] = exp(i pi k / (N / 2)), k < N / 2: the twiddles of every stage
__global__ void k_twiddles(int N, cd *__restrict__ w)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= N / 2) return;
    double sn, cs;
    sincospi((double)k / (double)(N / 2), &sn, &cs);
    w[k] = cd{cs, sn};
}

constexpr int kFirstBits = 8, kNextBits = 7;
constexpr int kFirstPts = 512, kNextPts = 1024;   // points of a workgroup of 256 threads
// points of the traces transformed together (at least one trace): 16 MB per
// array, so the passes and the sums find them in the memory-side cache and a
// call does not allocate the spectra of all traces (250 MB for 240 traces of
// 5000 samples; memory that was freed before is cleared at some 40 GB/s when
// it is allocated again, 7.4 ms per call after a thousand calls).  The call
// with 2^18, 2^19, 2^20, 2^21 points: 1.52, 1.23, 1.03, 1.23 ms
constexpr int kBatchPts = 1 << 20;

__device__ inline void butterfly(cd &a, cd &b, cd w, int sign)
{
    const cd b1 = cmul(b, cd{w.re, sign * w.im}), a0 = a;
    a = cd{a0.re + b1.re, a0.im + b1.im};
    b = cd{a0.re - b1.re, a0.im - b1.im};
}

// x [ntr][ns] float (row stride ld) -> X [ntr][N] complex after the first
// `bits` stages (sign +1): gathered in bit-reversed order, zero padding beyond
// ns; mute[i] != 0 gives a zero trace; samples 2..ns are divided by scale[i]
// (mul = 0) or multiplied by it (mul = 1), sample 1 is kept (util.c:502-520,
// 545-571).  With src the points come from there, already in that order
// (then sign applies).  A workgroup takes kFirstPts consecutive points.
__global__ __launch_bounds__(256) void k_fft_first(int ntr, int ns, int ld, int logN, int bits,
                                                   const float *__restrict__ x, const unsigned char *__restrict__ mute,
                                                   const float *__restrict__ scale, int mul, const cd *src, int sign,
                                                   const cd *__restrict__ tw, cd *X)
{
    __shared__ cd p[kFirstPts];
    const long long total = (long long)ntr << logN, g0 = (long long)blockIdx.x * kFirstPts;
#pragma unroll
    for (int k = 0; k < kFirstPts / 256; ++k) {
        const long long g = g0 + threadIdx.x + 256 * k;
        cd v{0.0, 0.0};
        if (g < total) {
            if (src) {
                v = src[g];
            } else {
                const int i = (int)(g >> logN);
                const unsigned r = (unsigned)(g & ((1LL << logN) - 1));
                const int j = (int)(__builtin_bitreverse32(r) >> (32 - logN));
                if (j < ns && !(mute && mute[i])) {
                    float f = x[(long long)i * ld + j];
                    if (scale && j >= 1) f = mul ? f * scale[i] : f / scale[i];
                    v.re = (double)f;
                }
            }
        }
        p[threadIdx.x + 256 * k] = v;
    }
    for (int q = 0; q < bits; ++q) {
        __syncthreads();
        const int b = threadIdx.x, pos = b & ((1 << q) - 1), i0 = ((b >> q) << (q + 1)) + pos;
        butterfly(p[i0], p[i0 + (1 << q)], tw[(size_t)pos << (logN - 1 - q)], sign);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kFirstPts / 256; ++k) {
        const long long g = g0 + threadIdx.x + 256 * k;
        if (g < total) X[g] = p[threadIdx.x + 256 * k];
    }
}

// stages s0 .. s0 + bits - 1 in place: a workgroup takes, of one span of
// 2^(s0 + bits) points, the 2^bits points 2^s0 apart of C consecutive columns
__global__ __launch_bounds__(256) void k_fft_next(int logN, int s0, int bits, int logC, int sign,
                                                  const cd *__restrict__ tw, cd *__restrict__ X)
{
    __shared__ cd p[kNextPts];
    const int C = 1 << logC, pts = 1 << (bits + logC);
    const long long wg = blockIdx.x;
    const int lo0 = (int)(wg & ((1LL << (s0 - logC)) - 1)) << logC;
    cd *base = X + ((wg >> (s0 - logC)) << (s0 + bits)) + lo0;
    for (int e = threadIdx.x; e < pts; e += 256) p[e] = base[((size_t)(e >> logC) << s0) + (e & (C - 1))];
    for (int q = 0; q < bits; ++q) {
        __syncthreads();
        for (int b = threadIdx.x; b < pts / 2; b += 256) {
            const int c = b & (C - 1), kb = b >> logC;               // butterfly kb of column c
            const int pos = kb & ((1 << q) - 1), k0 = ((kb >> q) << (q + 1)) + pos;
            const size_t ang = ((size_t)pos << s0) + lo0 + c;        // of 2^(s0 + q)
            butterfly(p[(k0 << logC) + c], p[((k0 + (1 << q)) << logC) + c], tw[ang << (logN - 1 - s0 - q)], sign);
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < pts; e += 256) base[((size_t)(e >> logC) << s0) + (e & (C - 1))] = p[e];
}

// per-trace scales of NORMALIZE 1 / 2 (max |x| over samples 2..ns, 0 -> 1)
__global__ void k_trace_max(int ntr, int ns, int ld, const float *__restrict__ x, float *__restrict__ mx)
{
    const int i = blockIdx.x;
    float m = 0.0f, mn = 0.0f;
    for (int j = 1 + threadIdx.x; j < ns; j += blockDim.x) {
        const float v = x[(long long)i * ld + j];
        m = fmaxf(m, v);
        mn = fminf(mn, v);
    }
    __shared__ float sm[256], sn[256];
    sm[threadIdx.x] = m;
    sn[threadIdx.x] = mn;
    __syncthreads();
    for (int o = blockDim.x / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            sm[threadIdx.x] = fmaxf(sm[threadIdx.x], sm[threadIdx.x + o]);
            sn[threadIdx.x] = fminf(sn[threadIdx.x], sn[threadIdx.x + o]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const float a = sm[0], b = fabsf(sn[0]);
        float t = (a > b) ? a : b;
        if (t == 0.0f) t = 1.0f;
        mx[i] = t;
    }
}

// NORMALIZE 2: the observed trace times max_syn / max_obs (util.c:570)
__global__ void k_norm_ratio(int ntr, const float *mx_syn, const float *mx_obs, float *ratio)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ntr) ratio[i] = mx_syn[i] / mx_obs[i];
}

// S_n, S_d and the per-frequency share of Ebar (sum over the running sums);
// n_all traces in all, ntr of them in D and M, behind those summed before
// (more: some were)
__global__ void k_wiener_sums(int n_all, int ntr, bool more, int N, const cd *__restrict__ D, const cd *__restrict__ M, cd *__restrict__ sn,
                              double *__restrict__ sd, double *__restrict__ erow)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= N) return;
    const double n = (double)n_all;
    cd a{0.0, 0.0};
    double d = 0.0, e = 0.0;
    if (more) {
        a = sn[k];
        d = sd[k];
        e = erow[k];
    }
    auto add = [&](const cd &dd, const cd &mm) {
        const cd nd{n * dd.re, n * dd.im}, nm{n * mm.re, n * mm.im};
        const cd p = cmul(nd, cd{mm.re, -mm.im});
        a.re += p.re;
        a.im += p.im;
        d += nm.re * mm.re + nm.im * mm.im;
        e += d;
    };
    int i = 0;
    for (; i + 8 <= ntr; i += 8) {   // eight traces are read before the first is added
        cd dd[8], mm[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            dd[q] = D[(long long)(i + q) * N + k];
            mm[q] = M[(long long)(i + q) * N + k];
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) add(dd[q], mm[q]);
    }
    for (; i < ntr; ++i) add(D[(long long)i * N + k], M[(long long)i * N + k]);
    sn[k] = a;
    sd[k] = d;
    erow[k] = e;
}

// fixed-order sum of erow (one block)
__global__ void k_sum_fixed(int N, const double *__restrict__ v, double *__restrict__ out)
{
    __shared__ double sm[256];
    double a = 0.0;
    int k = threadIdx.x;
    for (; k + 15 * 256 < N; k += 16 * 256) {
        double x[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) x[q] = v[k + 256 * q];
#pragma unroll
        for (int q = 0; q < 16; ++q) a += x[q];
    }
    for (; k < N; k += 256) a += v[k];
    sm[threadIdx.x] = a;
    __syncthreads();
    for (int o = blockDim.x / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) sm[threadIdx.x] += sm[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = sm[0];
}

// D_s = FFT(s) S_n / (S_d + eps), written bit-reversed for the inverse pass
__global__ void k_wiener_div(int N, int logN, const cd *__restrict__ S, const cd *__restrict__ sn,
                             const double *__restrict__ sd, const double *__restrict__ eps, cd *__restrict__ out)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= N) return;
    const double den = sd[k] + *eps;
    const cd q{sn[k].re / den, sn[k].im / den};
    const unsigned r = __builtin_bitreverse32((unsigned)k) >> (32 - logN);
    out[r] = cmul(S[k], q);
}

__global__ void k_eps(const double *esum, int N, int ntr, float eps_stf, double *eps)
{
    // stf.c:170-174: Ebar = Ebar / (Npad ntr); the regulariser EPS_STF ntr Ebar
    const float ebar = (float)(*esum / ((double)N * (double)ntr));
    *eps = (double)((eps_stf * (float)ntr) * ebar);
}

__global__ void k_stf_out(int ns, int N, const cd *__restrict__ x, float *__restrict__ stf)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < ns) stf[j] = (float)(x[j].re / (double)N);
}

unsigned blocks(long long n, int b = 256) { return (unsigned)((n + b - 1) / b); }

// device buffers of one call, cut from one allocation
struct StfDev {
    hipStream_t st = nullptr;
    char *mem = nullptr;
    size_t used = 0;
    float *obs = nullptr, *syn = nullptr, *sig = nullptr, *stf = nullptr, *mx = nullptr;
    unsigned char *mute = nullptr;
    cd *D = nullptr, *M = nullptr, *S = nullptr, *sn = nullptr, *Y = nullptr, *tw = nullptr;
    double *sd = nullptr, *erow = nullptr, *esum = nullptr;
    // sizes first (mem null: only `used` grows), then pointers
    template <typename T> void take(T *&p, size_t n)
    {
        if (mem) p = (T *)(mem + used);
        used += (n * sizeof(T) + 255) / 256 * 256;
    }
    void layout(size_t ntr, size_t ns, size_t N, size_t batch)
    {
        used = 0;
        take(obs, ntr * ns);
        take(syn, ntr * ns);
        take(sig, ns);
        take(stf, ns);
        take(mx, 4 * ntr);
        take(mute, ntr);
        take(D, batch * N);
        take(M, batch * N);
        take(S, N);
        take(sn, N);
        take(Y, N);
        take(tw, N / 2);
        take(sd, N);
        take(erow, N);
        take(esum, 2);
    }
    void release()
    {
        if (mem) (void)hipFree(mem);
        if (st) (void)hipStreamDestroy(st);
        *this = StfDev{};
    }
};

#define SCHK(x)                                                                                  \
    do {                                                                                         \
        hipError_t e_ = (x);                                                                     \
        if (e_ != hipSuccess) {                                                                  \
            R.release();                                                                         \
            return dn_fail(nullptr, "%s: %s", #x, hipGetErrorString(e_));                        \
        }                                                                                        \
    } while (0)

// the stages after the first pass, of ntr transforms
void fft_rest(cd *X, int ntr, int logN, int sign, const cd *tw, hipStream_t st)
{
    for (int s0 = kFirstBits; s0 < logN;) {
        const int bits = std::min(kNextBits, logN - s0);
        const int logC = std::min(s0, 10 - bits);   // kNextPts points
        const long long wgs = (long long)ntr << (logN - bits - logC);
        hipLaunchKernelGGL(k_fft_next, dim3((unsigned)wgs), dim3(256), 0, st, logN, s0, bits, logC, sign, tw, X);
        s0 += bits;
    }
}

// transforms of ntr float traces (sign +1)
void fft_traces(int ntr, int ns, int logN, const float *x, const unsigned char *mute, const float *scale, int mul,
                const cd *tw, cd *X, hipStream_t st)
{
    hipLaunchKernelGGL(k_fft_first, dim3(blocks((long long)ntr << logN, kFirstPts)), dim3(256), 0, st, ntr, ns, ns, logN,
                       std::min(kFirstBits, logN), x, mute, scale, mul, (const cd *)nullptr, 1, tw, X);
    fft_rest(X, ntr, logN, 1, tw, st);
}

}  // namespace

extern "C" int dn_stf(int ntr, int ns, const float *obs, const float *syn, const float *signal,
                      const unsigned char *mute, const dn_stf_opts *o, float *stf)
{
    if (ntr < 1 || ns < 2 || !obs || !syn || !signal || !o || !stf) return dn_fail(nullptr, "dn_stf: bad arguments");
    if (o->normalize < 0 || o->normalize > 2) return dn_fail(nullptr, "dn_stf: NORMALIZE must be 0, 1 or 2");
    // stf.c:38: Npad = 2^(ceil(log2 ns) + 2)
    const int logN = (int)std::ceil(std::log((double)ns) / std::log(2.0)) + 2;
    if (logN > 26) return dn_fail(nullptr, "dn_stf: record too long");
    const int N = 1 << logN;
    const int batch = std::max(1, std::min(ntr, kBatchPts / N));
    StfDev R;
    SCHK(hipStreamCreateWithFlags(&R.st, hipStreamNonBlocking));
    const size_t nd = (size_t)ntr * ns;
    R.layout(ntr, ns, N, batch);
    SCHK(hipMalloc((void **)&R.mem, R.used));
    R.layout(ntr, ns, N, batch);
    hipStream_t st = R.st;
    SCHK(hipMemcpyAsync(R.obs, obs, nd * sizeof(float), hipMemcpyHostToDevice, st));
    SCHK(hipMemcpyAsync(R.syn, syn, nd * sizeof(float), hipMemcpyHostToDevice, st));
    SCHK(hipMemcpyAsync(R.sig, signal, (size_t)ns * sizeof(float), hipMemcpyHostToDevice, st));
    std::vector<unsigned char> mu(ntr, 0);
    if (mute)
        for (int i = 0; i < ntr; ++i) mu[i] = mute[i] ? 1 : 0;
    SCHK(hipMemcpyAsync(R.mute, mu.data(), (size_t)ntr, hipMemcpyHostToDevice, st));
    // normalisation of samples 2..ns (muted traces are zero whatever the scale)
    const float *sc_syn = nullptr, *sc_obs = nullptr;
    int mul_obs = 0;
    if (o->normalize) {
        float *mxs = R.mx, *mxo = R.mx + ntr;
        hipLaunchKernelGGL(k_trace_max, dim3(ntr), dim3(256), 0, st, ntr, ns, ns, R.syn, mxs);
        hipLaunchKernelGGL(k_trace_max, dim3(ntr), dim3(256), 0, st, ntr, ns, ns, R.obs, mxo);
        if (o->normalize == 1) {
            sc_syn = mxs;
            sc_obs = mxo;
        } else {
            hipLaunchKernelGGL(k_norm_ratio, dim3(blocks(ntr)), dim3(256), 0, st, ntr, mxs, mxo, R.mx + 2 * ntr);
            sc_obs = R.mx + 2 * ntr;
            mul_obs = 1;
        }
    }
    hipLaunchKernelGGL(k_twiddles, dim3(blocks(N / 2)), dim3(256), 0, st, N, R.tw);
    fft_traces(1, ns, logN, R.sig, nullptr, nullptr, 0, R.tw, R.S, st);
    for (int i = 0; i < ntr; i += batch) {
        const int n = std::min(batch, ntr - i);
        fft_traces(n, ns, logN, R.obs + (size_t)i * ns, R.mute + i, sc_obs ? sc_obs + i : nullptr, mul_obs, R.tw, R.D, st);
        fft_traces(n, ns, logN, R.syn + (size_t)i * ns, R.mute + i, sc_syn ? sc_syn + i : nullptr, 0, R.tw, R.M, st);
        hipLaunchKernelGGL(k_wiener_sums, dim3(blocks(N)), dim3(256), 0, st, ntr, n, i > 0, N, R.D, R.M, R.sn, R.sd,
                           R.erow);
    }
    hipLaunchKernelGGL(k_sum_fixed, dim3(1), dim3(256), 0, st, N, R.erow, R.esum);
    hipLaunchKernelGGL(k_eps, dim3(1), dim3(1), 0, st, R.esum, N, ntr, o->eps_stf, R.esum + 1);
    hipLaunchKernelGGL(k_wiener_div, dim3(blocks(N)), dim3(256), 0, st, N, logN, R.S, R.sn, R.sd, R.esum + 1, R.Y);
    hipLaunchKernelGGL(k_fft_first, dim3(blocks(N, kFirstPts)), dim3(256), 0, st, 1, ns, ns, logN,
                       std::min(kFirstBits, logN), (const float *)nullptr, (const unsigned char *)nullptr,
                       (const float *)nullptr, 0, R.Y, -1, R.tw, R.Y);
    fft_rest(R.Y, 1, logN, -1, R.tw, st);
    hipLaunchKernelGGL(k_stf_out, dim3(blocks(ns)), dim3(256), 0, st, ns, N, R.Y, R.stf);
    SCHK(hipGetLastError());
    SCHK(hipMemcpyAsync(stf, R.stf, (size_t)ns * sizeof(float), hipMemcpyDeviceToHost, st));
    SCHK(hipStreamSynchronize(st));
    R.release();
    return 0;
}

// stf.c on the context: the shot's observed data, its synthetics from the
// current signal, the context's trace kill / offset mute plus OFFSETC_STF
extern "C" int dn_stf_shot(dn_ctx *c, int shot, const dn_stf_opts *o, float *stf)
{
    if (!c || !o || !stf) return dn_fail(c, "dn_stf_shot: NULL argument");
    if (shot < 0 || shot >= c->nshots) return dn_fail(c, "dn_stf_shot: shot %d outside 0..%d", shot, c->nshots - 1);
    if (!c->d_obs) return dn_fail(c, "dn_stf_shot: set the observed data first");
    const int ntr = c->ntr, nt_max = c->nt_max, ns = c->shot_nt[shot];
    std::vector<float> syn((size_t)ntr * nt_max), obs((size_t)ntr * nt_max), sig(nt_max);
    if (dn_forward_shots(c, std::vector<int>{shot}, syn.data())) return -1;
    HIPCHK(c, hipMemcpy(obs.data(), c->d_obs + (size_t)shot * ntr * nt_max, obs.size() * sizeof(float),
                        hipMemcpyDeviceToHost));
    HIPCHK(c, hipMemcpy(sig.data(), c->d_sig + (size_t)c->src_off[shot] * nt_max, nt_max * sizeof(float),
                        hipMemcpyDeviceToHost));
    // [ntr][ns] rows of the shot's record length
    std::vector<float> o2((size_t)ntr * ns), s2((size_t)ntr * ns);
    for (int r = 0; r < ntr; ++r)
        for (int j = 0; j < ns; ++j) {
            o2[(size_t)r * ns + j] = obs[(size_t)r * nt_max + j];
            s2[(size_t)r * ns + j] = syn[(size_t)r * nt_max + j];
        }
    std::vector<unsigned char> mute(ntr, 0);
    const dn_ctx::DataCond &d = c->dc;
    const float DH = c->p.dh;
    const int l0 = c->src_off[shot];
    const float xs = d.offset_mute ? d.src_x[shot] : (float)c->src_i[l0] * DH;
    const float ys = d.offset_mute ? d.src_y[shot] : (float)c->src_j[l0] * DH;
    for (int r = 0; r < ntr; ++r) {
        if (d.on && d.trkill && d.kill[(size_t)shot * d.kill_ntr + r] == 1) mute[r] = 1;   // stf.c:46-64
        const float xr = (float)c->rec_i[r] * DH, yr = (float)c->rec_j[r] * DH;
        const float offset = (float)std::sqrt((double)(((xs - xr) * (xs - xr)) + ((ys - yr) * (ys - yr))));
        if (d.on && d.offset_mute == 1 && offset >= d.offsetc) mute[r] = 1;                  // stf.c:67-90
        if (d.on && d.offset_mute == 2 && offset <= d.offsetc) mute[r] = 1;
        if (o->offsetc_stf > 0.0f && std::fabs(offset) >= o->offsetc_stf) mute[r] = 1;        // stf.c:93-110
    }
    if (dn_stf(ntr, ns, o2.data(), s2.data(), sig.data(), mute.data(), o, stf)) return dn_fail(c, "%s", dn_last_error(nullptr));
    return 0;
}
