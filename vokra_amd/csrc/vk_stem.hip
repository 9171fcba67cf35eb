// vk_stem.hip — the encoder's conv stem (crates/vokra-models/src/whisper/
// encoder.rs:58-104) on the bf16 matrix cores with whole f32 operands.
//
// Both convolutions (kernel 3) are GEMMs over rows that already lie in memory: with
// a zero row before and after each clip, output frame t of a stride-s convolution
// reads padded rows s t, s t + 1 and s t + 2. So there is no im2col pass.
//
// Precision: every f32 value is the sum of three bf16 values, x = p0 + p1 + p2, each
// the rounding of what the ones before leave: exact whatever its neighbours'
// magnitudes, since bf16 has f32's exponents (fp16 halves under a scale per tensor
// lose the bits of what is small beside its largest value; here only |x| < 2^-108
// does, to 2^-126 of an absolute error). A product
// runs as the six p_i q_j with i + j <= 2 in f32 accumulators, p0 q0 apart from the
// five smaller ones; what is left out is below 2^-24 of the product. One
// v_mfma_f32_32x32x16_bf16 takes the place of eight f32 ones, so the sums have
// shorter chains of roundings than an f32 GEMM's. Values that are not finite keep
// p1 = p2 = 0 and leave outputs that are not finite: those are computed again with
// f32 products of the recombined operands.
// Error against 64 bits at Whisper-large dims (relative 2-norm of the stem's
// output): 4.7e-7, f32 GEMMs 1.2e-6; d 384 .. 1024: 2.7e-7 .. 3.9e-7 against 5.8e-7 ..
// 9.7e-7.
//
// Layouts, chosen so that the 1 KiB operand fragments of a stage (32 rows or output
// channels by 16 k) are contiguous in memory, in the order the lanes hold them:
//   log-mel parts       [3][clip][channel / 16][frame + 1][16]
//   first convolution's [3][clip][channel / 16][parity][(frame + 1) / 2][16]
//   weights             [3][out / 32][tap * channels / 16][lane][8]
#include <algorithm>

#include "vk_common.h"
#include "vk_launch.h"

namespace vk {

typedef float vk_f32x16s __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float stem_f(uint16_t p) { return __uint_as_float((uint32_t)p << 16); }

// x = p0 + p1 + p2. A finite x that would round to an infinite p0 takes the largest
// finite one (what it leaves still fits p1 + p2).
__device__ __forceinline__ void stem_split(float x, uint16_t (&p)[3]) {
    const bool finite = (__float_as_uint(x) & 0x7fffffffu) < 0x7f800000u;
    p[0] = __builtin_bit_cast(uint16_t, (__bf16)x);
    if (finite && (p[0] & 0x7fffu) == 0x7f80u) p[0] -= 1;
    const float r1 = finite ? x - stem_f(p[0]) : 0.0f;
    p[1] = __builtin_bit_cast(uint16_t, (__bf16)r1);
    p[2] = __builtin_bit_cast(uint16_t, (__bf16)(r1 - stem_f(p[1])));
}

// 16 values -> 32 bytes of each part
__device__ __forceinline__ void stem_store16(const float (&v)[16], uint16_t* at, size_t part) {
    uint32_t w[3][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        uint16_t a[3], b[3];
        stem_split(v[2 * i], a);
        stem_split(v[2 * i + 1], b);
#pragma unroll
        for (int p = 0; p < 3; ++p) w[p][i] = a[p] | ((uint32_t)b[p] << 16);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int i = 0; i < 2; ++i)
            reinterpret_cast<uint4*>(at + p * part)[i] =
                make_uint4(w[p][4 * i], w[p][4 * i + 1], w[p][4 * i + 2], w[p][4 * i + 3]);
}

// log-mel [clip][m][frame] -> its parts, one thread per (clip, 16 channels, padded
// row): zero rows at both ends, zero channels from nm on. The threads past those
// clear the end rows of the second convolution's input (d / 16 channel blocks).
__global__ __launch_bounds__(256) void vk_stem_mel(const float* __restrict__ x, size_t batch, int nm, int nf,
                                                   uint16_t* __restrict__ a, int d, uint16_t* __restrict__ h) {
    const int rows = nf + 2, cbs = (nm + 15) / 16, hcb = d / 16, hp = (nf + 3) / 2;
    const size_t n_mel = batch * cbs * rows;
    size_t gid = (size_t)blockIdx.x * 256 + threadIdx.x;
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = 0.0f;
    if (gid < n_mel) {
        const int row = (int)(gid % rows);
        const size_t cc = gid / rows, clip = cc / cbs;
        const int c0 = 16 * (int)(cc % cbs);
        if (row > 0 && row <= nf) {
            const float* src = x + (clip * nm + c0) * nf + (row - 1);
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (c0 + i < nm) v[i] = src[(size_t)i * nf];
        }
        stem_store16(v, a + gid * 16, n_mel * 16);
        return;
    }
    gid -= n_mel;
    if (gid >= batch * hcb * 2) return;
    const int row = (gid & 1) ? nf + 1 : 0;
    const size_t at = ((gid >> 1) * 2 + (row & 1)) * hp + (row >> 1);
    stem_store16(v, h + at * 16, batch * hcb * 2 * hp * 16);
}

// conv weights [out][channel][3] f32 -> their parts in fragment order, one thread
// per lane's eight values (channels from c on zero).
__global__ __launch_bounds__(256) void vk_stem_pack(const float* __restrict__ w, int out, int c, uint16_t* __restrict__ wp) {
    const int cbs = (c + 15) / 16, ks_n = 3 * cbs;
    const size_t n = (size_t)(out / 32) * ks_n * 64, gid = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (gid >= n) return;
    const int lane = (int)(gid & 63), ks = (int)((gid >> 6) % ks_n), tap = ks / cbs, c0 = 16 * (ks - tap * cbs) + 8 * (lane >> 5);
    const size_t o = (gid >> 6) / ks_n * 32 + (lane & 31);
    uint32_t q[3][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint16_t a[3], b[3];
        stem_split(c0 + 2 * i < c ? w[(o * c + c0 + 2 * i) * 3 + tap] : 0.0f, a);
        stem_split(c0 + 2 * i + 1 < c ? w[(o * c + c0 + 2 * i + 1) * 3 + tap] : 0.0f, b);
#pragma unroll
        for (int p = 0; p < 3; ++p) q[p][i] = a[p] | ((uint32_t)b[p] << 16);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) reinterpret_cast<uint4*>(wp)[p * n + gid] = make_uint4(q[p][0], q[p][1], q[p][2], q[p][3]);
}

// One convolution's rows: row r = clip r / rpc, frame r % rpc; its k step (tap, cb)
// starts at clip * clip + frame * 16 + cb * block + tap_off[tap] halves of a part.
struct StemRows {
    const uint16_t* a;
    size_t part, clip, block, tap1, tap2;
    int m, rpc, cbs;
};

// ---------------------------------------------------------------------------
// The convolution GEMM: out[r][n] = gelu(bias[n] + sum_k A(r, k) W(n, k)), then either
// (SPLIT) its three parts into the next convolution's rows, or + pos[frame][n] as f32.
//
// Bound: the matrix cores (six bf16 MFMAs per product). 2 x 2 waves of 32 WT output
// channels by 32 WT frames, stages of 16 k through a ring of three in LDS, filled by
// direct loads two stages ahead. WT = 2 reads 12 fragments per stage for 24 MFMAs of
// 32 clocks (about 64 bytes per clock and CU of the LDS's 128) and leaves room for two
// workgroups per CU, whose barriers and reads fall on each other's MFMAs. Output
// channels are on the row side of the accumulators, so a lane holds four
// consecutive ones of a frame and stores them as a vector. Workgroups of one XCD walk
// the output channels first: they share both the frames' and the weights' fragments
// in its L2.
// Measured at Whisper-large dims, four clips: the whole stem 757 us as im2col, f32 GEMMs
// and a position pass -> 380 (convolutions 96 + 300, the second 354 GFLOP of MFMA work at
// 1.18 PFLOP/s of the 1.40 that MFMAs alone reach; fp16 halves 310); one clip at d 384 153 -> 38.
template <int WT, bool SPLIT>
__global__ __launch_bounds__(256, 2) void vk_stem_gemm(const StemRows A, const uint16_t* __restrict__ wp, int n,
                                                       const float* __restrict__ bias, float* __restrict__ out,
                                                       const float* __restrict__ pos, uint16_t* __restrict__ op,
                                                       size_t op_part, int op_half) {
    constexpr int WAVES = 4, NS = 3, FR = 2 * WT;         // fragments per part and side
    constexpr int LT = 6 * FR, LP = LT / WAVES;           // 1 KiB loads per stage / per wave
    constexpr int STAGE = LT * 1024;
    static_assert(LP * WAVES == LT, "whole loads per wave");
    __shared__ __align__(16) uint8_t ring[NS][STAGE];     // W parts, then A parts
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave >> 1, wm = wave & 1;
    const int tiles_n = (n + 64 * WT - 1) / (64 * WT), t = vk_xcd_tile(blockIdx.x, gridDim.x);
    const int mt = t / tiles_n, m0 = mt * 64 * WT, nt0 = (t - mt * tiles_n) * FR;  // first row, first 32-channel tile
    const int n_ot = n / 32, n_st = 3 * A.cbs;
    const size_t w_part = (size_t)n_ot * n_st * 512;  // halves

    // this wave's loads: fragment q = wave + 4 i of the stage
    const uint16_t* src[LP];
    uint32_t dst[LP];
    const uint32_t base = __builtin_amdgcn_readfirstlane(vk_lds_addr(&ring[0][0]));
#pragma unroll
    for (int i = 0; i < LP; ++i) {
        const int q = wave + WAVES * i, f = q % FR;
        dst[i] = base + q * 1024;
        if (q < 3 * FR) {
            src[i] = wp + (q / FR) * w_part + (size_t)min(nt0 + f, n_ot - 1) * n_st * 512 + lane * 8;
        } else {
            const int r = min(m0 + 32 * f + (lane & 31), A.m - 1), clip = r / A.rpc;
            src[i] = A.a + (q / FR - 3) * A.part + clip * A.clip + (size_t)(r - clip * A.rpc) * 16 + 8 * (lane >> 5);
        }
    }
    // requests the next stage; past the last one the last again, into a buffer that is not read
    int is = 0, icb = 0;
    size_t ioff = 0, itap = 0;
    auto issue = [&](int buf) {
#pragma unroll
        for (int i = 0; i < LP; ++i) {
            const bool w = wave + WAVES * i < 3 * FR;  // uniform
            vk_dma_b128(src[i] + (w ? (size_t)is * 512 : ioff), dst[i] + buf * STAGE);
        }
        if (is + 1 < n_st) {
            ++is;
            ++icb;
            ioff += A.block;
            if (icb == A.cbs) {
                icb = 0;
                itap = is == A.cbs ? A.tap1 : A.tap2;
                ioff = itap;
            }
        }
    };
    // p0 q0 apart from the smaller products: the large sums round once per 16 k
    vk_f32x16s top[WT][WT], low[WT][WT];
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) top[i][j][r] = low[i][j][r] = 0.0f;
    auto compute = [&](int buf, int nbuf) {
        const vk_bf16x8* st = reinterpret_cast<const vk_bf16x8*>(&ring[buf][0]) + lane;
        vk_bf16x8 w[3][WT], a[3][WT];
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int i = 0; i < WT; ++i) {
                w[p][i] = st[(p * FR + wn * WT + i) * 64];
                a[p][i] = st[((3 + p) * FR + wm * WT + i) * 64];
            }
        issue(nbuf);  // behind the reads: their wait does not take these addresses' time (390 -> 380 us, four clips)
        constexpr int PW[6] = {2, 0, 0, 1, 1, 0}, PA[6] = {0, 0, 2, 1, 0, 1};
#pragma unroll
        for (int u = 0; u < 6; ++u)
#pragma unroll
            for (int i = 0; i < WT; ++i)
#pragma unroll
                for (int j = 0; j < WT; ++j) {
                    vk_f32x16s& to = u == 1 ? top[i][j] : low[i][j];
                    to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[PW[u]][i], a[PA[u]][j], to, 0, 0, 0);
                }
    };
    issue(0);
    issue(1);
    int buf = 0, nbuf = 2;
#pragma unroll 1
    for (int s = 0; s < n_st; ++s) {
        // stage s has landed everywhere, and every wave has read stage s - 1
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LP) : "memory");
        compute(buf, nbuf);
        buf = buf == NS - 1 ? 0 : buf + 1;
        nbuf = nbuf == NS - 1 ? 0 : nbuf + 1;
    }
    vk_wait_vm<0>();  // nothing may land in LDS after the workgroup has ended

#pragma unroll
    for (int j = 0; j < WT; ++j) {
        const int row = m0 + (wm * WT + j) * 32 + (lane & 31), row_ld = min(row, A.m - 1);
        const int clip = row_ld / A.rpc, fr = row_ld - clip * A.rpc;
#pragma unroll
        for (int i = 0; i < WT; ++i) {
            const int ot = nt0 + wn * WT + i;
            if (ot >= n_ot) continue;  // uniform
            vk_f32x16s y;
            bool bad = false;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                y[r] = top[i][j][r] + low[i][j][r];
                bad |= !__builtin_isfinite(y[r]);
            }
            if (__any(bad)) {  // f32 products, for the outputs that are not finite
                vk_f32x16s f;
#pragma unroll
                for (int r = 0; r < 16; ++r) f[r] = 0.0f;
                const uint16_t* wsrc = wp + (size_t)ot * n_st * 512 + lane * 8;
                const uint16_t* asrc = A.a + clip * A.clip + (size_t)fr * 16 + 8 * (lane >> 5);
#pragma unroll 1
                for (int s = 0; s < n_st; ++s) {
                    const int tap = s / A.cbs;
                    const uint16_t* as = asrc + (size_t)(s - tap * A.cbs) * A.block + (tap == 0 ? 0 : tap == 1 ? A.tap1 : A.tap2);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float wv = stem_f(wsrc[e]) + stem_f(wsrc[w_part + e]) + stem_f(wsrc[2 * w_part + e]);
                        const float av = stem_f(as[e]) + stem_f(as[A.part + e]) + stem_f(as[2 * A.part + e]);
                        f = __builtin_amdgcn_mfma_f32_32x32x2f32(wv, av, f, 0, 0, 0);
                    }
                    wsrc += 512;
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) y[r] = __builtin_isfinite(y[r]) ? y[r] : f[r];
            }
            if (row >= A.m) continue;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int ch = 32 * ot + 8 * q + 4 * (lane >> 5);  // four consecutive output channels
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = vk_gelu_as(bias[ch + e] + y[4 * q + e]);
                if (SPLIT) {
                    uint16_t p[4][3];
#pragma unroll
                    for (int e = 0; e < 4; ++e) stem_split(v[e], p[e]);
                    const int pr = fr + 1;  // padded row
                    const size_t o = ((((size_t)clip * (n / 16) + (ch >> 4)) * 2 + (pr & 1)) * op_half + (pr >> 1)) * 16 + (ch & 15);
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        *reinterpret_cast<uint2*>(op + k * op_part + o) =
                            make_uint2(p[0][k] | ((uint32_t)p[1][k] << 16), p[2][k] | ((uint32_t)p[3][k] << 16));
                } else {
                    float* o = out + (size_t)row * n + ch;
                    const float4 ps = *reinterpret_cast<const float4*>(pos + (size_t)fr * n + ch);
                    const float z[4] = {v[0] + ps.x, v[1] + ps.y, v[2] + ps.z, v[3] + ps.w};
                    if ((reinterpret_cast<uintptr_t>(out) & 15) == 0) {
                        *reinterpret_cast<float4*>(o) = make_float4(z[0], z[1], z[2], z[3]);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[e] = z[e];
                    }
                }
            }
        }
    }
}

size_t stem_weight_halves(int out, int c) { return (size_t)3 * out * 3 * ((c + 15) / 16 * 16); }
size_t stem_mel_halves(size_t batch, int nm, int nf) { return 3 * batch * ((nm + 15) / 16) * (nf + 2) * 16; }
size_t stem_hidden_halves(size_t batch, int d, int nf) { return 3 * batch * (d / 16) * 2 * ((nf + 3) / 2) * 16; }

hipError_t launch_stem_pack(hipStream_t s, const float* w, int out, int c, void* wp) {
    if (out < 32 || out % 32 != 0 || c < 1) return hipErrorInvalidValue;
    const size_t n = (size_t)(out / 32) * 3 * ((c + 15) / 16) * 64;
    hipLaunchKernelGGL(vk_stem_pack, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, w, out, c, (uint16_t*)wp);
    return hipGetLastError();
}

// 128 x 128 tiles from about three quarters of a workgroup per CU on, else 64 x 64. Stem,
// us, 64 / 128: first convolution of 144 tiles (1 clip, d 768) 79 / 86, of 192 (1 x 1024) 101 /
// 107; second of 240 (2 x 1280) 245 / 211, of 216 (3 x 768) 165 / 150.
template <bool SPLIT>
static hipError_t go_stem(hipStream_t s, const StemRows& a, const void* wp, int n, const float* bias, float* out,
                          const float* pos, void* op, size_t op_part, int op_half) {
    const size_t big = (size_t)((a.m + 127) / 128) * ((n + 127) / 128), small = (size_t)((a.m + 63) / 64) * ((n + 63) / 64);
    if (small > (size_t)INT32_MAX) return hipErrorInvalidValue;
    if (big >= 200)
        hipLaunchKernelGGL((vk_stem_gemm<2, SPLIT>), dim3((unsigned)big), dim3(256), 0, s, a, (const uint16_t*)wp, n,
                           bias, out, pos, (uint16_t*)op, op_part, op_half);
    else
        hipLaunchKernelGGL((vk_stem_gemm<1, SPLIT>), dim3((unsigned)small), dim3(256), 0, s, a, (const uint16_t*)wp, n,
                           bias, out, pos, (uint16_t*)op, op_part, op_half);
    return hipGetLastError();
}

hipError_t launch_stem(hipStream_t s, const float* mel, size_t batch, int nm, int nf, int nc, int d, const StemW& w,
                       void* mel_parts, void* hidden_parts, float* out) {
    if (batch == 0) return hipSuccess;
    if (batch * nf > (size_t)INT32_MAX || d % 32 != 0) return hipErrorInvalidValue;
    const int rows = nf + 2, cbs = (nm + 15) / 16, hcb = d / 16, hp = (nf + 3) / 2;
    const size_t threads = batch * cbs * rows + batch * hcb * 2, wgs = (threads + 255) / 256;
    if (wgs > (size_t)INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(vk_stem_mel, dim3((unsigned)wgs), dim3(256), 0, s, mel, batch, nm, nf, (uint16_t*)mel_parts, d,
                       (uint16_t*)hidden_parts);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const size_t h_part = stem_hidden_halves(batch, d, nf) / 3;
    const StemRows a1 = {(const uint16_t*)mel_parts, stem_mel_halves(batch, nm, nf) / 3, (size_t)cbs * rows * 16,
                         (size_t)rows * 16, 16, 32, (int)(batch * nf), nf, cbs};
    e = go_stem<true>(s, a1, w.w1, d, w.b1, nullptr, nullptr, hidden_parts, h_part, hp);
    if (e != hipSuccess) return e;
    // stride 2: taps 0 and 2 lie in the even rows, tap 1 in the odd ones
    const StemRows a2 = {(const uint16_t*)hidden_parts, h_part, (size_t)hcb * 2 * hp * 16, (size_t)2 * hp * 16,
                         (size_t)hp * 16, 16, (int)(batch * nc), nc, hcb};
    return go_stem<false>(s, a2, w.w2, d, w.b2, out, w.pos, nullptr, 0, 0);
}

}  // namespace vk
