// vk_stem.hip — the encoder's conv stem (crates/vokra-models/src/whisper/
// encoder.rs:58-104) on the fp16 matrix cores at f32 precision.
//
// Both convolutions (kernel 3) are GEMMs over rows that already lie in memory:
// with the input kept time-major, [clip][frame + 1][channel] and a zero row
// before and after each clip, output frame t of a stride-s convolution reads the
// 3 C consecutive values from padded row s t on. So there is no im2col pass;
// weights are stored [out][tap][channel].
//
// Precision: every f32 operand x is x * 2^e = hi + lo, two fp16 values, with e
// chosen so that the largest magnitude of the tensor (the log-mel: of the clip)
// lands in 2^13 .. 2^14 (exact: a power of two); each product runs as three MFMAs, hi*hi + hi*lo +
// lo*hi, f32 accumulation, and the sum is scaled back. hi + lo carries x to
// 2^-23 of itself down to 2^-16 of the tensor's maximum and to 2^-39 of that
// maximum below, and the sums take a third of the f32 MFMA's rounding steps (16
// x 16 x 32 against 16 x 16 x 4). Scales: the weights' once at set_stem, the
// log-mel's from each clip's largest finite magnitude (one pass; a clip's result
// does not depend on its batch), the first convolution's
// output from the bound L1(w) * max|x| + max|b| (|gelu(y)| <= |y|).
// Error against 64 bits at Whisper-large dims (relative 2-norm of the stem's
// output): 7.6e-7, the f32 GEMMs 1.2e-6; d 384 .. 1024: 3.9e-7 .. 7e-7 against
// 5.8e-7 .. 9.9e-7.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "vk_common.h"
#include "vk_launch.h"

namespace vk {

typedef _Float16 vk_sh8 __attribute__((ext_vector_type(8)));

namespace stem {
constexpr int PARTS = 64;  // partial maxima per clip of the log-mel
}

__device__ __forceinline__ float stem_exp2i(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }  // -126..127

// hi = fp16(x), lo = fp16(x - hi); an infinite or NaN x keeps lo = 0.
__device__ __forceinline__ void stem_split(float x, uint16_t& hi, uint16_t& lo) {
    const _Float16 h = (_Float16)x;
    const float r = x - (float)h;
    const _Float16 l = (_Float16)(r == r && fabsf(r) <= 3.40282347e38f ? r : 0.0f);
    hi = __builtin_bit_cast(uint16_t, h);
    lo = __builtin_bit_cast(uint16_t, l);
}

// e with 2^13 <= m * 2^e < 2^14 (0 for m = 0), within the exponents of a normal scale.
__device__ __forceinline__ int stem_exponent(double m) {
    if (!(m > 0.0)) return 0;
    return min(max(13 - ilogb(m), -120), 120);
}

// Largest finite |x| per workgroup of a clip's n values: part[clip][PARTS].
__global__ __launch_bounds__(256) void vk_stem_absmax(const float* __restrict__ x, size_t n, float* __restrict__ part) {
    __shared__ float red[4];
    const float* xc = x + (size_t)blockIdx.y * n;
    uint32_t m = 0;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)stem::PARTS * 256) {
        const uint32_t b = __float_as_uint(xc[i]) & 0x7fffffffu;
        m = max(m, b < 0x7f800000u ? b : 0u);
    }
    const float w = vk_group_max<64>(__uint_as_float(m));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = w;
    __syncthreads();
    if (threadIdx.x == 0)
        part[blockIdx.y * stem::PARTS + blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// log-mel [clip][m][frame] -> hi / lo [clip][nf + 2][mp] (zero rows at both ends,
// zero channels from m on), through a 64 x 64 LDS tile; also the zero rows of the
// second convolution's input and the clip's scales:
// scal[clip] = {e of the log-mel, e of the first convolution's output}.
__global__ __launch_bounds__(256) void vk_stem_mel(const float* __restrict__ x, int nm, int mp, int nf,
                                                   const float* __restrict__ part, float l1max, float bmax,
                                                   uint16_t* __restrict__ ahi, uint16_t* __restrict__ alo,
                                                   uint16_t* __restrict__ hhi, uint16_t* __restrict__ hlo, int d,
                                                   int2* __restrict__ scal) {
    __shared__ float tile[64][65];
    __shared__ float clip_max;
    const int tid = threadIdx.x, b = blockIdx.z, f0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
    static_assert(stem::PARTS == 64, "one wave reduces a clip's partials");
    if (tid < 64) {
        const float w = vk_group_max<64>(part[b * stem::PARTS + tid]);
        if (tid == 0) clip_max = w;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int c = (tid >> 6) + 4 * i, f = tid & 63;  // consecutive lanes: consecutive frames
        tile[f][c] = (c0 + c < nm && f0 + f < nf) ? x[((size_t)b * nm + c0 + c) * nf + f0 + f] : 0.0f;
    }
    __syncthreads();
    const float xmax = clip_max;
    const int e = stem_exponent((double)xmax);
    const float s = stem_exp2i(e);
    if (blockIdx.x == 0 && blockIdx.y == 0) {
        if (tid == 0) scal[b] = make_int2(e, stem_exponent((double)l1max * (double)xmax + (double)bmax));
        for (int i = tid; i < d; i += 256) {
            const size_t first = (size_t)b * (nf + 2) * d + i, end = first + (size_t)(nf + 1) * d;
            hhi[first] = hlo[first] = hhi[end] = hlo[end] = 0;
        }
    }
    const size_t base = (size_t)b * (nf + 2) * mp;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int f = (tid >> 6) + 4 * i, c = tid & 63;
        if (c0 + c >= mp) continue;
        if (f0 + f < nf) {
            uint16_t hi, lo;
            stem_split(tile[f][c] * s, hi, lo);
            const size_t o = base + (size_t)(f0 + f + 1) * mp + c0 + c;
            ahi[o] = hi;
            alo[o] = lo;
        }
        if (f0 == 0 && f == 0) ahi[base + c0 + c] = alo[base + c0 + c] = 0;
        if (f0 + f == nf - 1) {
            const size_t o = base + (size_t)(nf + 1) * mp + c0 + c;
            ahi[o] = alo[o] = 0;
        }
    }
}

// conv weights [out][channel][3] f32 -> hi / lo [out][3][cp] of w * 2^e
// (channels from c on zero).
__global__ void vk_stem_pack(const float* __restrict__ w, int out, int c, int cp, float scale,
                             uint16_t* __restrict__ hi, uint16_t* __restrict__ lo) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)out * 3 * cp) return;
    const int ch = (int)(i % cp), tap = (int)(i / cp % 3);
    const size_t o = i / cp / 3;
    uint16_t h = 0, l = 0;
    if (ch < c) stem_split(w[(o * c + ch) * 3 + tap] * scale, h, l);
    hi[i] = h;
    lo[i] = l;
}

// ---------------------------------------------------------------------------
// The convolution GEMM: out[r][n] = gelu(bias[n] + sum_k A(r, k) W(n, k)), row r =
// clip r / rpc, frame r % rpc, whose k values start at clip * clip_stride + frame
// * row_stride halves. Then either (SPLIT) hi / lo of out * 2^scal[clip].y into the next
// convolution's padded rows, or + pos[frame][n] as f32.
//
// Bound: the matrix cores (three fp16 MFMAs per product). 2 x 2 waves of 16 WT x
// 16 WT tiles, 32 values of k per stage, two stages in LDS so that two
// workgroups share a CU (128 KB): a stage's operands are read into registers, the
// workgroup meets, the stage after next is requested into the same buffer by
// direct loads, and 3 WT^2 MFMAs run over it. LDS rows hold 32 halves (64
// bytes); chunk c of row r sits at 4 r + (c ^ (r / 4 % 4)), which puts the 16
// rows that a 16-lane read takes on all 64 banks.
// Measured at Whisper-large dims, four clips (us): the whole stem 757 -> 325 (im2col 70 + 16,
// f32 GEMMs 167 + 539, positions 19 before; convolutions 98 + 246 now, the second 59
// GFLOP at 240 TFLOP/s, 720 of MFMA work); one clip at d 384 152 -> 52.
template <int WT, bool SPLIT>
__global__ __launch_bounds__(256, 2) void vk_stem_gemm(const uint16_t* __restrict__ ahi, const uint16_t* __restrict__ alo,
                                                       int m, int rpc, size_t clip_stride, int row_stride,
                                                       const uint16_t* __restrict__ whi, const uint16_t* __restrict__ wlo,
                                                       int n, int k, const float* __restrict__ bias, const int2* __restrict__ scal,
                                                       int w_exp, float* __restrict__ out,
                                                       const float* __restrict__ pos, uint16_t* __restrict__ ohi,
                                                       uint16_t* __restrict__ olo) {
    constexpr int T = 32 * WT;                   // workgroup tile rows / columns
    constexpr int MAT = T * 64;                  // bytes of one matrix of a stage
    constexpr int Q = T / 16 / 4;                // 1 KiB loads (16 rows) per wave and matrix
    constexpr int LOADS = 4 * Q;
    __shared__ __align__(16) uint8_t lds[2][4 * MAT];  // A hi, A lo, W hi, W lo
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int tiles_m = (m + T - 1) / T, tiles = gridDim.x, L = blockIdx.x, per = tiles / 8;
    const int t = per * 8 == tiles ? (L % 8) * per + L / 8 : L;
    const int m0 = (t % tiles_m) * T, n0 = (t / tiles_m) * T;
    // lane l of a load writes LDS slot l = 4 row + chunk', chunk' = chunk ^ (row / 4 % 4)
    size_t ao[Q], wo[Q];  // halves
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int r = 16 * (wave * Q + q) + (lane >> 2), c = 8 * ((lane & 3) ^ ((r >> 2) & 3));
        const int ar = min(m0 + r, m - 1), clip = ar / rpc;
        ao[q] = (size_t)clip * clip_stride + (size_t)(ar - clip * rpc) * row_stride + c;
        wo[q] = (size_t)min(n0 + r, n - 1) * k + c;
    }
    const uint32_t base = __builtin_amdgcn_readfirstlane(vk_lds_addr(&lds[0][0]) + wave * Q * 1024);
    auto issue = [&](int st, int buf) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const uint32_t d = base + buf * (4 * MAT) + q * 1024;
            vk_dma_b128(ahi + ao[q] + 32 * (size_t)st, d);
            vk_dma_b128(alo + ao[q] + 32 * (size_t)st, d + MAT);
            vk_dma_b128(whi + wo[q] + 32 * (size_t)st, d + 2 * MAT);
            vk_dma_b128(wlo + wo[q] + 32 * (size_t)st, d + 3 * MAT);
        }
    };
    vk_f32x4 acc[WT][WT];
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) acc[i][j] = (vk_f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    // operand reads: row lane % 16 of a 16-row subtile, chunk lane / 16
    const int lr = lane & 15, slot = (4 * lr + ((lane >> 4) ^ (lr >> 2))) * 16;
    const int n_st = k / 32, last = n_st - 1;
    issue(0, 0);
    issue(min(1, last), 1);
#pragma unroll 1
    for (int st = 0; st < n_st; ++st) {
        const int buf = st & 1;
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(LOADS) : "memory");  // stage st has landed everywhere
        const uint8_t* p = &lds[buf][0];
        vk_sh8 ah[WT], al[WT], bh[WT], bl[WT];
#pragma unroll
        for (int i = 0; i < WT; ++i) {
            ah[i] = *reinterpret_cast<const vk_sh8*>(p + (wm * WT + i) * 1024 + slot);
            al[i] = *reinterpret_cast<const vk_sh8*>(p + MAT + (wm * WT + i) * 1024 + slot);
            bh[i] = *reinterpret_cast<const vk_sh8*>(p + 2 * MAT + (wn * WT + i) * 1024 + slot);
            bl[i] = *reinterpret_cast<const vk_sh8*>(p + 3 * MAT + (wn * WT + i) * 1024 + slot);
        }
        VK_LDS_BARRIER();  // every wave has stage st in registers
        issue(min(st + 2, last), buf);
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
            for (int j = 0; j < WT; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], bl[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[i], bh[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], bh[j], acc[i][j], 0, 0, 0);
            }
    }
    vk_wait_vm<0>();  // nothing may land in LDS after the workgroup has ended
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = m0 + (wm * WT + i) * 16 + 4 * (lane >> 4) + r;
            if (row >= m) continue;
            const int clip = row / rpc, fr = row - clip * rpc;
            const int2 sc = scal[clip];
            const int unscale = -((SPLIT ? sc.x : sc.y) + w_exp);
            const float s2 = stem_exp2i(sc.y);
#pragma unroll
            for (int j = 0; j < WT; ++j) {
                const int col = n0 + (wn * WT + j) * 16 + lr;
                if (col >= n) continue;
                const float y = vk_gelu_as(bias[col] + ldexpf(acc[i][j][r], unscale));
                if (SPLIT) {
                    uint16_t hi, lo;
                    stem_split(y * s2, hi, lo);
                    const size_t o = ((size_t)clip * (rpc + 2) + fr + 1) * n + col;
                    ohi[o] = hi;
                    olo[o] = lo;
                } else {
                    out[(size_t)row * n + col] = y + pos[(size_t)fr * n + col];
                }
            }
        }
}

// The exponent of a weight tensor's scale: its largest finite magnitude to 2^13.
int stem_weight_exponent(const float* w, size_t n) {
    int32_t m[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // magnitudes order as their bits
    auto mag = [&](size_t i) {
        int32_t v;
        memcpy(&v, w + i, 4);
        v &= 0x7fffffff;
        return v < 0x7f800000 ? v : 0;
    };
    size_t i = 0;
    for (; i + 8 <= n; i += 8)
        for (int j = 0; j < 8; ++j) m[j] = std::max(m[j], mag(i + j));
    for (; i < n; ++i) m[0] = std::max(m[0], mag(i));
    const int32_t top = *std::max_element(m, m + 8);
    float f;
    memcpy(&f, &top, 4);
    return f > 0.0f ? std::min(std::max(13 - std::ilogb(f), -120), 120) : 0;
}

hipError_t launch_stem_pack(hipStream_t s, const float* w, int out, int c, int cp, int e, void* hi, void* lo) {
    const size_t total = (size_t)out * 3 * cp;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(vk_stem_pack, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, w, out, c, cp,
                       std::ldexp(1.0f, e), (uint16_t*)hi, (uint16_t*)lo);
    return hipGetLastError();
}

size_t stem_scalars(size_t batch) { return batch * (2 + stem::PARTS); }

// 128 x 128 tiles unless they leave CUs idle, then 64 x 64.
template <bool SPLIT>
static hipError_t go_stem(hipStream_t s, const void* ahi, const void* alo, int m, int rpc, size_t clip_stride,
                          int row_stride, const void* whi, const void* wlo, int n, int k, const float* bias,
                          const int2* scal, int we, float* out, const float* pos, void* ohi, void* olo) {
    const size_t big = (size_t)((m + 127) / 128) * ((n + 127) / 128), small = (size_t)((m + 63) / 64) * ((n + 63) / 64);
    if (small > (size_t)INT32_MAX || k % 32 != 0 || k < 32) return hipErrorInvalidValue;
    if (big >= 256)
        hipLaunchKernelGGL((vk_stem_gemm<4, SPLIT>), dim3((unsigned)big), dim3(256), 0, s, (const uint16_t*)ahi,
                           (const uint16_t*)alo, m, rpc, clip_stride, row_stride, (const uint16_t*)whi,
                           (const uint16_t*)wlo, n, k, bias, scal, we, out, pos, (uint16_t*)ohi, (uint16_t*)olo);
    else
        hipLaunchKernelGGL((vk_stem_gemm<2, SPLIT>), dim3((unsigned)small), dim3(256), 0, s, (const uint16_t*)ahi,
                           (const uint16_t*)alo, m, rpc, clip_stride, row_stride, (const uint16_t*)whi,
                           (const uint16_t*)wlo, n, k, bias, scal, we, out, pos, (uint16_t*)ohi, (uint16_t*)olo);
    return hipGetLastError();
}

hipError_t launch_stem(hipStream_t s, const float* mel, int batch, int nm, int nf, int nc, int d, const StemW& w,
                       const StemBufs& b, float* out) {
    if (batch == 0) return hipSuccess;
    const int mp = stem_channels(nm);
    int2* scal = reinterpret_cast<int2*>(b.scal);
    float* part = b.scal + 2 * (size_t)batch;
    hipLaunchKernelGGL(vk_stem_absmax, dim3(stem::PARTS, batch), dim3(256), 0, s, mel, (size_t)nm * nf, part);
    hipLaunchKernelGGL(vk_stem_mel, dim3((nf + 63) / 64, (mp + 63) / 64, batch), dim3(256), 0, s, mel, nm, mp, nf, part,
                       w.l1max, w.bmax, (uint16_t*)b.ahi, (uint16_t*)b.alo, (uint16_t*)b.hhi, (uint16_t*)b.hlo, d, scal);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    e = go_stem<true>(s, b.ahi, b.alo, batch * nf, nf, (size_t)(nf + 2) * mp, mp, w.w1hi, w.w1lo, d, 3 * mp, w.b1,
                      scal, w.e1, nullptr, nullptr, b.hhi, b.hlo);
    if (e != hipSuccess) return e;
    return go_stem<false>(s, b.hhi, b.hlo, batch * nc, nc, (size_t)(nf + 2) * d, 2 * d, w.w2hi, w.w2lo, d, 3 * d, w.b2,
                          scal, w.e2, out, w.pos, nullptr, nullptr);
}

}  // namespace vk
