// vk_frontend.hip — the Whisper front end on gfx950: log-mel spectrogram
// (crates/vokra-models/src/whisper/mel.rs:123-183, fused form
// crates/vokra-ops/src/fused_logmel.rs:80-175) and 1-D convolution
// (crates/vokra-backend-cpu/src/kernels/mod.rs:583-822) for the encoder's conv
// stem (crates/vokra-models/src/whisper/encoder.rs:58-108).
//
// The log-mel is one pass from samples to log10 energies (a real FFT per frame in
// LDS, the power spectrum, the filter bank's nonzero weights) and one for the
// per-clip (max(v, gmax - 8) + 4) / 4 normalisation. Convolution is im2col + the
// f32 matrix-core GEMM (the encoder's conv stem has kernels of its own,
// vk_stem.hip).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "vk_common.h"

namespace vk {

namespace fe {
constexpr int NS = 480000, NFFT = 400, HOP = 160, NFR = 3000, NB = 201, PAD = 200;
constexpr int FR = 16;              // frames per workgroup of the transform
constexpr int NC = NFFT / 2;        // complex points
constexpr int PW = 205;             // floats per frame's power row (odd: frames on distinct banks)
}  // namespace fe

// numpy mode="reflect" (crates/vokra-ops/src/stft.rs:269-285) for the
// single reflection the 200-sample centre padding needs.
__device__ __forceinline__ int fe_reflect(int i, int n) { return i < 0 ? -i : (i >= n ? 2 * (n - 1) - i : i); }

__device__ __forceinline__ float2 fe_add(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 fe_sub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 fe_mul(float2 a, float2 b) {
    return make_float2(fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ float2 fe_mul_mi(float2 a) { return make_float2(a.y, -a.x); }  // * -i

// Forward DFT of 4 / 8 / 5 points in place (natural order in and out).
__device__ __forceinline__ void fe_dft4(float2& a, float2& b, float2& c, float2& d) {
    const float2 s0 = fe_add(a, c), s1 = fe_sub(a, c), s2 = fe_add(b, d), s3 = fe_mul_mi(fe_sub(b, d));
    a = fe_add(s0, s2);
    b = fe_add(s1, s3);
    c = fe_sub(s0, s2);
    d = fe_sub(s1, s3);
}
__device__ __forceinline__ void fe_dft8(float2 (&x)[8]) {
    float2 e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
    fe_dft4(e[0], e[1], e[2], e[3]);
    fe_dft4(o[0], o[1], o[2], o[3]);
    const float h = 0.70710678118654752440f;
    o[1] = make_float2(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x));   // * exp(-i pi / 4)
    o[2] = fe_mul_mi(o[2]);
    o[3] = make_float2(h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y));  // * exp(-3 i pi / 4)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        x[k] = fe_add(e[k], o[k]);
        x[k + 4] = fe_sub(e[k], o[k]);
    }
}
__device__ __forceinline__ void fe_dft5(float2 (&x)[5]) {
    const float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;  // cos(2 pi / 5), cos(4 pi / 5)
    const float s1 = 0.95105651629515357212f, s2 = 0.58778525229247312917f;   // sin
    const float2 a = fe_add(x[1], x[4]), b = fe_add(x[2], x[3]), d = fe_sub(x[1], x[4]), f = fe_sub(x[2], x[3]);
    const float2 u1 = make_float2(fmaf(c2, b.x, fmaf(c1, a.x, x[0].x)), fmaf(c2, b.y, fmaf(c1, a.y, x[0].y)));
    const float2 u2 = make_float2(fmaf(c1, b.x, fmaf(c2, a.x, x[0].x)), fmaf(c1, b.y, fmaf(c2, a.y, x[0].y)));
    const float2 v1 = make_float2(fmaf(s2, f.x, s1 * d.x), fmaf(s2, f.y, s1 * d.y));
    const float2 v2 = make_float2(fmaf(-s1, f.x, s2 * d.x), fmaf(-s1, f.y, s2 * d.y));
    x[0] = fe_add(x[0], fe_add(a, b));
    x[1] = make_float2(u1.x + v1.y, u1.y - v1.x);
    x[4] = make_float2(u1.x - v1.y, u1.y + v1.x);
    x[2] = make_float2(u2.x + v2.y, u2.y - v2.x);
    x[3] = make_float2(u2.x - v2.y, u2.y + v2.x);
}

// out[b][m][t] = log10(max(mel energy, 1e-10)) of frame t of clip b (zero-padded
// / trimmed to 480000 samples, reflect-padded by 200, windowed: mel.rs:134-137,
// fused_logmel.rs:135-138), FR frames per workgroup, and the workgroup's maximum
// into partial[b][wg].
// Bound: LDS and arithmetic of a few thousand flops per frame; the samples and
// the result are 1.9 + 1.5 MB per clip. A 400-point real transform is a 200-point
// complex one of (even, odd) samples, 200 = 8 x 25 as eight 25-point sequences:
// 8-point transforms over n = 25 n1 + n2, twiddles W200^(n2 k1), then 25 = 5 x 5,
// every pass in place in LDS (25 k1 + 5 c + d holds bin k1 + 8 (c + 5 d) at the
// end). It replaces a 402 x 400 f32 GEMM over materialised frames, a dense
// filter-bank GEMM and the passes between them: log-mel of 4 clips, 128 bands,
// 114 -> 25 us, and its rounding error is that of ~10 stages, not of 400-term sums:
// relative 2-norm of the result against 64 bits 1.5e-7, the GEMMs 2.6e-7.
// fb: per band {first bin, end bin} as ints, then the dense [n_mels][201] weights.
__global__ __launch_bounds__(256) void vk_log_mel(const float* __restrict__ pcm, int n_samples,
                                                  const float* __restrict__ win, const float2* __restrict__ tw_g,
                                                  const float* __restrict__ fb, int n_mels, float* __restrict__ out,
                                                  float* __restrict__ partial) {
    using namespace fe;
    __shared__ float2 z[FR][NC];
    __shared__ float pw[FR][PW];
    __shared__ float2 tw[NFFT];  // W400^j
    __shared__ float red[4];
    __shared__ int bad_lo[FR], bad_hi[FR];  // first and last bin of each frame whose power is not finite
    const int tid = threadIdx.x, b = blockIdx.y, t0 = blockIdx.x * FR;
    if (tid < FR) {
        bad_lo[tid] = NB;
        bad_hi[tid] = -1;
    }
    const float* clip = pcm + (size_t)b * n_samples;
    for (int i = tid; i < NFFT; i += 256) tw[i] = tw_g[i];
    for (int i = tid; i < FR * NC; i += 256) {
        const int f = i / NC, n = i - f * NC, t = t0 + f;
        float2 v = make_float2(0.0f, 0.0f);
        if (t < NFR) {
            const int p0 = fe_reflect(t * HOP + 2 * n - PAD, NS), p1 = fe_reflect(t * HOP + 2 * n + 1 - PAD, NS);
            v.x = (p0 < n_samples ? clip[p0] : 0.0f) * win[2 * n];
            v.y = (p1 < n_samples ? clip[p1] : 0.0f) * win[2 * n + 1];
        }
        z[f][n] = v;
    }
    __syncthreads();
    for (int i = tid; i < FR * 25; i += 256) {
        const int f = i / 25, n2 = i - f * 25;
        float2 x[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) x[q] = z[f][25 * q + n2];
        fe_dft8(x);
        z[f][n2] = x[0];
#pragma unroll
        for (int q = 1; q < 8; ++q) z[f][25 * q + n2] = fe_mul(x[q], tw[2 * n2 * q]);  // W200^(n2 q), 2 * 24 * 7 < 400
    }
    __syncthreads();
    for (int i = tid; i < FR * 40; i += 256) {
        const int f = i / 40, r = i - f * 40, k1 = r / 5, q = r - k1 * 5;
        float2* s = &z[f][25 * k1 + q];
        float2 x[5];
#pragma unroll
        for (int a = 0; a < 5; ++a) x[a] = s[5 * a];
        fe_dft5(x);
        s[0] = x[0];
#pragma unroll
        for (int c = 1; c < 5; ++c) s[5 * c] = fe_mul(x[c], tw[16 * q * c]);  // W25^(q c), 16 * 16 < 400
    }
    __syncthreads();
    for (int i = tid; i < FR * 40; i += 256) {
        const int f = i / 40, r = i - f * 40;
        float2* s = &z[f][5 * r];
        float2 x[5] = {s[0], s[1], s[2], s[3], s[4]};
        fe_dft5(x);
#pragma unroll
        for (int a = 0; a < 5; ++a) s[a] = x[a];
    }
    __syncthreads();
    // X[k] = (Z[k] + conj Z[200 - k]) / 2 - i W400^k (Z[k] - conj Z[200 - k]) / 2, and X[200 - k] from the same two
    for (int i = tid; i < FR * 101; i += 256) {
        const int f = i / 101, k = i - f * 101, kr = k == 0 ? 0 : NC - k;
        auto at = [](int q) {
            const int k1 = q & 7, k2 = q >> 3, d = k2 / 5;
            return 25 * k1 + 5 * (k2 - 5 * d) + d;
        };
        const float2 u = z[f][at(k)], v = z[f][at(kr)];
        const float2 e = make_float2(0.5f * (u.x + v.x), 0.5f * (u.y - v.y));
        const float2 o = fe_mul(make_float2(0.5f * (u.y + v.y), 0.5f * (v.x - u.x)), tw[k]);
        const float2 p = fe_add(e, o), m = fe_sub(e, o);
        const float pk = fmaf(p.x, p.x, p.y * p.y), pr = fmaf(m.x, m.x, m.y * m.y);
        pw[f][k] = pk;
        pw[f][NC - k] = pr;
        if (!__builtin_isfinite(pk) || !__builtin_isfinite(pr)) {
            atomicMin(&bad_lo[f], __builtin_isfinite(pk) ? NC - k : k);
            atomicMax(&bad_hi[f], __builtin_isfinite(pr) ? k : NC - k);
        }
    }
    __syncthreads();
    const int2* range = reinterpret_cast<const int2*>(fb);
    const float* w = fb + 2 * n_mels;
    float mx = -INFINITY;
    for (int i = tid; i < FR * n_mels; i += 256) {
        const int f = i % FR, m = i / FR, t = t0 + f;  // consecutive threads: consecutive frames
        if (t >= NFR) continue;
        const int2 rg = range[m];
        float v = 0.0f;
        for (int k = rg.x; k < rg.y; ++k) v = fmaf(pw[f][k], w[(size_t)m * NB + k], v);
        // the reference's sum runs over every bin: a zero weight makes NaN of a power that is not finite
        if (bad_lo[f] < rg.x || bad_hi[f] >= rg.y) v = __builtin_nanf("");
        const float l = log10f(v > 1e-10f ? v : 1e-10f);
        out[((size_t)b * n_mels + m) * NFR + t] = l;
        mx = fmaxf(mx, l);
    }
    mx = vk_group_maxf<64>(mx);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    if (tid == 0) partial[(size_t)b * gridDim.x + blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// out = (max(out, gmax - 8) + 4) / 4 with gmax the clip's maximum (every
// workgroup reduces the clip's partials itself; mel.rs:176-181).
__global__ __launch_bounds__(256) void vk_logmel_norm(float* __restrict__ out, int n_mels,
                                                      const float* __restrict__ partial, int n_partial) {
    __shared__ float red[4];
    const int b = blockIdx.y;
    float mx = -INFINITY;
    for (int i = threadIdx.x; i < n_partial; i += 256) mx = fmaxf(mx, partial[(size_t)b * n_partial + i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, VK_WAVE));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    const float floor_v = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])) - 8.0f;
    const size_t n = (size_t)n_mels * fe::NFR;
    float* o = out + (size_t)b * n;
    const size_t i0 = (size_t)blockIdx.x * 256 + threadIdx.x, step = (size_t)gridDim.x * 256;
    if ((reinterpret_cast<uintptr_t>(out) & 15) == 0) {  // n is a multiple of 4
        float4* o4 = reinterpret_cast<float4*>(o);
        for (size_t i = i0; i < n / 4; i += step) {
            float4 v = o4[i];
            v.x = (fmaxf(v.x, floor_v) + 4.0f) / 4.0f;
            v.y = (fmaxf(v.y, floor_v) + 4.0f) / 4.0f;
            v.z = (fmaxf(v.z, floor_v) + 4.0f) / 4.0f;
            v.w = (fmaxf(v.w, floor_v) + 4.0f) / 4.0f;
            o4[i] = v;
        }
        return;
    }
    for (size_t i = i0; i < n; i += step) o[i] = (fmaxf(o[i], floor_v) + 4.0f) / 4.0f;
}

// im2col of x [in_ch][in_len] (zero outside 0..in_len): col[c * kernel + kk][t],
// the reference's layout (mod.rs:794-806).
__global__ void vk_im2col(const float* __restrict__ x, int in_ch, int in_len, int kernel, int stride, int padding,
                          int out_len, float* __restrict__ col) {
    const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (size_t)out_len * in_ch * kernel) return;
    const size_t t = gid % out_len, r = gid / out_len;
    const size_t c = r / kernel;
    const long pos = (long)t * stride + (long)(r % kernel) - padding;
    col[gid] = (pos >= 0 && pos < in_len) ? x[c * in_len + (size_t)pos] : 0.0f;
}

// out[oc][t] += bias[oc] (the reference adds the bias after its GEMM, mod.rs:814-820).
__global__ void vk_add_row_bias(float* __restrict__ out, const float* __restrict__ bias, int rows, int cols) {
    const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (size_t)rows * cols) return;
    out[gid] = out[gid] + bias[gid / cols];
}

// ---------------------------------------------------------------------------
// Host-side tables (built once per context, in double, cast to f32 as the
// reference does).

// Periodic Hann (crates/vokra-ops/src/window.rs:31,42-55).
void fe_hann_periodic(std::vector<float>& w) {
    w.resize(fe::NFFT);
    for (int n = 0; n < fe::NFFT; ++n) {
        const double x = 2.0 * M_PI * (double)n / (double)fe::NFFT;
        w[n] = (float)(0.5 - 0.5 * std::cos(x));
    }
}

// W400^j = exp(-2 pi i j / 400), j = 0 .. 399, as (cos, -sin) pairs.
void fe_twiddles(std::vector<float>& t) {
    t.resize(2 * fe::NFFT);
    for (int j = 0; j < fe::NFFT; ++j) {
        const double th = 2.0 * M_PI * (double)j / (double)fe::NFFT;
        t[2 * j] = (float)std::cos(th);
        t[2 * j + 1] = (float)-std::sin(th);
    }
}

// Slaney mel scale and the filter bank of crates/vokra-ops/src/mel.rs:29-130
// (triangles linear in Hz, Slaney norm), the Whisper front end's choice
// (crates/vokra-ops/src/frontend.rs:62-80).
static double fe_hz_to_mel(double f) {
    const double f_sp = 200.0 / 3.0, min_log_hz = 1000.0, min_log_mel = min_log_hz / f_sp;
    const double logstep = std::log(6.4) / 27.0;
    return f >= min_log_hz ? min_log_mel + std::log(f / min_log_hz) / logstep : f / f_sp;
}
static double fe_mel_to_hz(double mel) {
    const double f_sp = 200.0 / 3.0, min_log_hz = 1000.0, min_log_mel = min_log_hz / f_sp;
    const double logstep = std::log(6.4) / 27.0;
    return mel >= min_log_mel ? min_log_hz * std::exp(logstep * (mel - min_log_mel)) : f_sp * mel;
}
void fe_mel_filterbank(int n_mels, std::vector<float>& w) {
    const double sr = 16000.0, lo = fe_hz_to_mel(0.0), hi = fe_hz_to_mel(sr / 2.0);
    std::vector<double> band(n_mels + 2);
    for (int i = 0; i < n_mels + 2; ++i) band[i] = fe_mel_to_hz(lo + (hi - lo) * (double)i / (double)(n_mels + 1));
    w.assign((size_t)n_mels * fe::NB, 0.0f);
    for (int m = 0; m < n_mels; ++m) {
        const double left = band[m], center = band[m + 1], right = band[m + 2];
        for (int k = 0; k < fe::NB; ++k) {
            const double f = (double)k * sr / (double)fe::NFFT;
            const double lower = center > left ? (f - left) / (center - left) : 0.0;
            const double upper = right > center ? (right - f) / (right - center) : 0.0;
            const float v = (float)std::max(0.0, std::min(lower, upper));
            w[(size_t)m * fe::NB + k] = (float)((double)v * (2.0 / (right - left)));
        }
    }
}

// The filter bank as vk_log_mel reads it: per band its first and end nonzero
// bin (the bits of two ints; an empty band 0, 0), then the dense weights.
void fe_mel_ranges(int n_mels, const std::vector<float>& w, std::vector<float>& packed) {
    packed.assign(2 * (size_t)n_mels, 0.0f);
    for (int m = 0; m < n_mels; ++m) {
        int lo = fe::NB, hi = 0;
        for (int k = 0; k < fe::NB; ++k)
            if (w[(size_t)m * fe::NB + k] != 0.0f) {
                lo = std::min(lo, k);
                hi = k + 1;
            }
        if (hi == 0) lo = 0;
        std::memcpy(&packed[2 * m], &lo, 4);
        std::memcpy(&packed[2 * m + 1], &hi, 4);
    }
    packed.insert(packed.end(), w.begin(), w.end());
}

int fe_n_frames() { return fe::NFR; }

int logmel_n_partial() { return (fe::NFR + fe::FR - 1) / fe::FR; }

hipError_t launch_log_mel(hipStream_t s, const float* pcm, int batch, int n_samples, int n_mels, const float* win,
                          const float* tw, const float* fb, float* out, float* partial) {
    const int np = logmel_n_partial();
    hipLaunchKernelGGL(vk_log_mel, dim3(np, batch), dim3(256), 0, s, pcm, n_samples, win,
                       reinterpret_cast<const float2*>(tw), fb, n_mels, out, partial);
    hipLaunchKernelGGL(vk_logmel_norm, dim3(128, batch), dim3(256), 0, s, out, n_mels, partial, np);
    return hipGetLastError();
}

hipError_t launch_im2col(hipStream_t s, const float* x, int in_ch, int in_len, int kernel, int stride, int padding,
                         int out_len, float* col) {
    const size_t total = (size_t)out_len * in_ch * kernel;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(vk_im2col, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, x, in_ch, in_len, kernel,
                       stride, padding, out_len, col);
    return hipGetLastError();
}

hipError_t launch_add_row_bias(hipStream_t s, float* out, const float* bias, int rows, int cols) {
    const size_t total = (size_t)rows * cols;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(vk_add_row_bias, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, out, bias, rows, cols);
    return hipGetLastError();
}

}  // namespace vk
