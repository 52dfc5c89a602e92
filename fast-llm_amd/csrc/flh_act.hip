// flh_act.hip -- ACT_Q8 (activation quantisation) and bit-exact dequant.
//
// ACT_Q8 writes, per column, the q8_1 appendix (per 32: f16 d, f16 s, i8 qs)
// and the q8_K appendix (per 256: f32 d, i16 bsums[16], i8 qs) with the same
// bytes as the reference's fl_quantize_q8_1_block / fl_quantize_q8_K_block
// (src/runtime/quants.h:360-416): amax is a max (order free), d = amax/127
// and id = 127/amax are correctly rounded IEEE divisions, q = roundf(x*id)
// clamped to +-127, sums are exact integers, halves are RNE.
//
// One wave per 256-element chunk of one column: lane i owns elements
// 4i..4i+3 (one 16-B load, one packed dword store per appendix); 8-lane
// groups form the q8_1 blocks, 4-lane groups the q8_K 16-sums.
#include "flh_kstream.h"
#include "flh_internal.h"
#include "flh_status.h"

namespace flh {

__global__ __launch_bounds__(64) void k_act_q8(float * x, uint8_t * yq, uint32_t cols,
                                               uint32_t xstride) {
    const uint32_t lane = threadIdx.x, chunk = blockIdx.x, col = blockIdx.y;
    float * xc = x + (size_t)col * xstride;
    uint8_t * q81 = yq ? yq + (size_t)col * xstride * 4 : (uint8_t *)xc + xq_off(cols);
    uint8_t * q8k = (uint8_t *)xc + xqk_off(cols);
    const uint32_t e0 = chunk * 256 + lane * 4;
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (e0 + j < cols) ? xc[e0 + j] : 0.f;
    act_q8_lanes(v, lane, chunk, q81, q8k, cols);
}

// SILU_MUL fused with the ACT_Q8 of its output (the MoE / FFN down input):
// lane i of the wave for chunk `chunk` of column c computes h = silu(g) * u
// for elements 4i..4i+3 with k_silu_mul's expression, stores h, and quantises
// the same register values -- the bytes of k_silu_mul followed by k_act_q8.
__global__ __launch_bounds__(64) void k_silu_act_q8(const float * gate, const float * up, float * h, uint32_t n,
                                                    uint32_t gstride, uint32_t hstride) {
    const uint32_t lane = threadIdx.x, chunk = blockIdx.x, col = blockIdx.y;
    const float * gc = gate + (size_t)col * gstride;
    const float * uc = up + (size_t)col * gstride;
    float * hc = h + (size_t)col * hstride;
    const uint32_t e0 = chunk * 256 + lane * 4;
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = 0.f;
        if (e0 + j < n) {
            const float g = gc[e0 + j];
            v[j] = (g / (1.0f + expf(-g))) * uc[e0 + j];
            hc[e0 + j] = v[j];
        }
    }
    act_q8_lanes(v, lane, chunk, (uint8_t *)hc + xq_off(n), (uint8_t *)hc + xqk_off(n), n);
}

// RMSNORM of one column with (write_app) the ACT_Q8 of its output, one
// workgroup of 16 waves: the sum of squares as thread partials (elements
// 4t..4t+3, 4t+4096.. in order) -> a wave butterfly (xor_lane exchanges;
// every lane ends with the same sum) -> the 16 wave sums in wave order; s = 1 / sqrtf(ss / n + eps)
// (correctly rounded sqrt and division, as the reference's libm); then wave w
// quantises chunks w, w + 16, ... with y = (x * s) * wnorm computed in the
// registers it quantises, so the appendices hold ACT_Q8's bytes for the
// stored y.
__global__ __launch_bounds__(1024) void k_rmsnorm_act_q8(const float * x, const float * wn, float * y, uint32_t n,
                                                         float eps, int write_app) {
    __shared__ float part[16];
    __shared__ float sh_s;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float ss = 0.f;
    for (uint32_t e0 = 4 * tid; e0 < n; e0 += 4096)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (e0 + j < n) ss += x[e0 + j] * x[e0 + j];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) ss += xor_lane(ss, o, lane);
    if (lane == 0) part[wave] = ss;
    __syncthreads();
    if (tid == 0) {
        float t = 0.f;
        for (int w = 0; w < 16; ++w) t += part[w];
        sh_s = 1.0f / sqrtf(t / (float)n + eps);
    }
    __syncthreads();
    const float s = sh_s;
    uint8_t * q81 = (uint8_t *)y + xq_off(n);
    uint8_t * q8k = (uint8_t *)y + xqk_off(n);
    for (uint32_t c = wave; c * 256 < n; c += 16) {
        const uint32_t e0 = c * 256 + 4 * lane;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = 0.f;
            if (e0 + j < n) {
                v[j] = x[e0 + j] * s * wn[e0 + j];
                y[e0 + j] = v[j];
            }
        }
        if (write_app) act_q8_lanes(v, lane, c, q81, q8k, n);
    }
}
// The same for n <= 16384, n % 4 == 0: thread t's elements (4t..4t+3,
// 4t+4096.., the chunks wave, wave + 16, ... of the loop above) and their
// norm weights come in as 16-B loads issued together, stay in registers
// through the reduction, and every thread sums the 16 wave partials itself
// (same order, so all hold the same s): one load round trip and one barrier.
__global__ __launch_bounds__(1024) void k_rmsnorm_act_q8_reg(const float * x, const float * wn, float * y, uint32_t n,
                                                             float eps, int write_app) {
    __shared__ float part[16];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float4 xv[4], wv[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t e0 = 4 * tid + 4096 * k;
        if (e0 < n) {
            xv[k] = *(const float4 *)(x + e0);
            wv[k] = *(const float4 *)(wn + e0);
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (4 * tid + 4096 * k < n) {
            ss += xv[k].x * xv[k].x;
            ss += xv[k].y * xv[k].y;
            ss += xv[k].z * xv[k].z;
            ss += xv[k].w * xv[k].w;
        }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) ss += xor_lane(ss, o, lane);
    if (lane == 0) part[wave] = ss;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < 16; ++w) t += part[w];
    const float s = 1.0f / sqrtf(t / (float)n + eps);
    uint8_t * q81 = (uint8_t *)y + xq_off(n);
    uint8_t * q8k = (uint8_t *)y + xqk_off(n);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t c = wave + 16 * k, e0 = c * 256 + 4 * lane;
        if (c * 256 >= n) break;
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        if (e0 < n) {
            v[0] = xv[k].x * s * wv[k].x;
            v[1] = xv[k].y * s * wv[k].y;
            v[2] = xv[k].z * s * wv[k].z;
            v[3] = xv[k].w * s * wv[k].w;
            *(float4 *)(y + e0) = make_float4(v[0], v[1], v[2], v[3]);
        }
        if (write_app) act_q8_lanes(v, lane, c, q81, q8k, n);
    }
}
int launch_rmsnorm_act_q8(const float * x, const float * wnorm, float * y, uint32_t n, float eps, bool app,
                          hipStream_t s) {
    if (n == 0) return FLH_OK;
    const bool reg = n <= 16384 && n % 4 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)wnorm & 15) == 0 &&
                     ((uintptr_t)y & 15) == 0;
    if (reg)
        hipLaunchKernelGGL(k_rmsnorm_act_q8_reg, dim3(1), dim3(1024), 0, s, x, wnorm, y, n, eps, app ? 1 : 0);
    else
        hipLaunchKernelGGL(k_rmsnorm_act_q8, dim3(1), dim3(1024), 0, s, x, wnorm, y, n, eps, app ? 1 : 0);
    return hip_check(hipGetLastError(), "k_rmsnorm_act_q8 launch");
}
int launch_silu_act_q8(const float * gate, const float * up, float * h, uint32_t n, uint32_t ncol,
                       uint32_t gstride, uint32_t hstride, hipStream_t s) {
    if (n == 0 || ncol == 0) return FLH_OK;
    hipLaunchKernelGGL(k_silu_act_q8, dim3((n + 255) / 256, ncol), dim3(64), 0, s, gate, up, h, n, gstride, hstride);
    return hip_check(hipGetLastError(), "k_silu_act_q8 launch");
}

int launch_act_q8(float * x, void * y_q81, uint32_t cols, uint32_t nx,
                  uint32_t xstride, hipStream_t s) {
    if (cols == 0 || nx == 0) return FLH_OK;
    const uint32_t chunks = (cols + 255) / 256;
    hipLaunchKernelGGL(k_act_q8, dim3(chunks, nx), dim3(64), 0, s, x, (uint8_t *)y_q81,
                       cols, xstride);
    return hip_check(hipGetLastError(), "k_act_q8 launch");
}

// ---------------------------------------------------------------- dequant --
// Bit-exact restatement of dequant_chunk's value formulas.  A matrix is one
// array of blocks (rows are whole blocks), so the work is split flat: a unit
// is 256 outputs (a superblock, or eight 32-weight blocks), lane i of a wave
// makes outputs 4i..4i+3 of it from one 4-byte read of the quants, so a wave
// stores 1 KiB in one piece and its reads of a block fall in one or two lines
// (one thread per 32 outputs stored 4 bytes every 128: 14336 x 4096 of Q4_K
// took 100 us, 2.7 TB/s).  Bound by the output's 4 bytes per weight: the
// stores are nontemporal (the output is far larger than an L2; ordinary ones
// take 64 us, these 40-43 us, 6.3-7.0 TB/s in every format), and a wave makes
// DEQ_UN = 2 units at once (1: 40-48 us, 4: 42, 8: 46; 1000 x 2048: 3.6 / 3.7
// / 4.5 / 6.6 us for 1 / 2 / 4 / 8).  Blocks are 2-byte aligned at best, and a
// caller's address may be odd: the reads are unaligned ones (memcpy), which
// gfx950 does in one instruction.
constexpr uint32_t DEQ_UN = 2;

__device__ __forceinline__ uint32_t ldu32(const uint8_t * p) {
    uint32_t v;
    __builtin_memcpy(&v, p, 4);
    return v;
}
__device__ __forceinline__ uint32_t ldu16(const uint8_t * p) {
    uint16_t v;
    __builtin_memcpy(&v, p, 2);
    return v;
}
// what lane `lane` reads of unit u (e: the lane's first element in its block or superblock)
struct DeqIn { uint32_t q, a, b, c; };

template <int FMT>
__device__ __forceinline__ DeqIn deq_load(const uint8_t * w, uint64_t u, uint32_t lane) {
    DeqIn in{0, 0, 0, 0};
    const uint32_t e = 4 * lane;
    if constexpr (FMT == FMT_Q8_0 || FMT == FMT_Q5_0) {
        constexpr uint32_t BB = FMT == FMT_Q8_0 ? 34 : 22;
        const uint8_t * b = w + (u * 8 + (lane >> 3)) * BB;
        const uint32_t i = e & 31;
        in.a = ldu16(b);
        if constexpr (FMT == FMT_Q8_0) in.q = ldu32(b + 2 + i);
        else { in.q = ldu32(b + 6 + (i & 15)); in.b = ldu32(b + 2); }
    } else if constexpr (FMT == FMT_Q4_K) {
        const uint8_t * b = w + u * 144;
        const uint32_t g = lane >> 3;                             // group of 32
        in.a = ldu32(b);                                          // d | dmin
        in.q = ldu32(b + 16 + 32 * (g >> 1) + (e & 31));
        in.b = ldu32(b + 4 + (g & 4 ? 8 : 0));                    // g < 4: scales 0..3, else bytes 8..11
        in.c = g & 4 ? (b[4 + (g & 3)] | ((uint32_t)b[8 + (g & 3)] << 8)) : b[8 + (g & 3)];
    } else if constexpr (FMT == FMT_Q6_K) {
        const uint8_t * b = w + u * 210;
        const uint32_t h = lane >> 5, gg = (lane >> 3) & 3, l = e & 31;
        in.q = ldu32(b + 64 * h + l + 32 * (gg & 1));
        in.b = ldu32(b + 128 + 32 * h + l);
        in.a = ldu16(b + 208);
        in.c = b[192 + 8 * h + l / 16 + 2 * gg];
    } else {
        const uint8_t * b = w + u * iq_block_bytes(FMT);
        const uint32_t ib = lane >> 3, l = (e & 31) >> 3;         // group, 8-element run
        in.a = ldu16(b);
        if constexpr (FMT == FMT_IQ2_XXS) {
            in.b = ldu32(b + 2 + 8 * ib + 4);
            in.q = (uint32_t)(k_iq2_grid[b[2 + 8 * ib + l]] >> (8 * (e & 4)));
        } else {
            in.b = ldu32(b + 66 + 4 * ib);
            in.q = k_iq3_grid[b[2 + 8 * ib + 2 * l + ((e >> 2) & 1)]];
        }
    }
    return in;
}
template <int FMT>
__device__ __forceinline__ float4 deq_vals(const DeqIn & in, uint32_t lane) {
    float v[4];
    const uint32_t e = 4 * lane;
    if constexpr (FMT == FMT_Q8_0) {
        const float d = h2f(in.a);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = d * (float)(int8_t)(in.q >> (8 * i));
    } else if constexpr (FMT == FMT_Q5_0) {
        const float d = h2f(in.a);
        const uint32_t s = e & 31, nib = (in.q >> (s & 16 ? 4 : 0)) & 0x0F0F0F0Fu, hb = in.b >> s;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t q5 = ((nib >> (8 * i)) & 0xFu) | (((hb >> i) & 1u) << 4);
            v[i] = d * (float)((int)q5 - 16);
        }
    } else if constexpr (FMT == FMT_Q4_K) {
        const float d = h2f(in.a & 0xFFFFu), dmin = h2f(in.a >> 16);
        const uint32_t g = lane >> 3, k = g & 3, s8 = (in.b >> (8 * k)) & 0xFFu;
        // the 6-bit scale and min of group g from bytes g, g + 4 (g < 4) or g + 4, g - 4, g
        uint32_t sc, mn;
        if (g < 4) { sc = s8 & 63u; mn = in.c & 63u; }
        else { sc = (s8 & 0xFu) | (((in.c & 0xFFu) >> 6) << 4); mn = (s8 >> 4) | ((in.c >> 14) << 4); }
        const float d1 = d * (float)sc, m1 = dmin * (float)mn;
        const uint32_t nib = (g & 1) ? (in.q >> 4) & 0x0F0F0F0Fu : in.q & 0x0F0F0F0Fu;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = d1 * (float)((nib >> (8 * i)) & 0xFFu) - m1;
    } else if constexpr (FMT == FMT_Q6_K) {
        const float d = h2f(in.a);
        const uint32_t gg = (lane >> 3) & 3;
        const uint32_t lo = gg < 2 ? in.q & 0x0F0F0F0Fu : (in.q >> 4) & 0x0F0F0F0Fu;
        const uint32_t q6 = lo | (((in.b >> (2 * gg)) & 0x03030303u) << 4);
        const float ds = d * (float)(int8_t)in.c;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = ds * (float)((int)((q6 >> (8 * i)) & 0xFFu) - 32);
    } else {
        // db * (+-grid magnitude), the factor the reference's canonical IQ dots
        // multiply x by (quants.h:252-254, 280-283); its dequant_chunk has no
        // IQ case (kernels.h:215-221)
        const float db = iq_db(FMT, h2f(in.a), in.b);
        const uint32_t sg = iq_sign8(in.b >> (7 * ((e & 31) >> 3))) >> (e & 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = (int)((in.q >> (8 * i)) & 0xFFu);
            v[i] = db * (float)((sg >> i) & 1u ? -m : m);
        }
    }
    return make_float4(v[0], v[1], v[2], v[3]);
}
// units of 256 outputs; n32: 32-weight blocks in the matrix (the last unit of
// a 32-weight-block format may be partial: its lanes past the end stop)
template <int FMT>
__global__ __launch_bounds__(256) void k_dequant(const uint8_t * __restrict__ w, uint64_t n32, float * __restrict__ out) {
    typedef float f4a __attribute__((ext_vector_type(4), aligned(4)));
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t u0 = ((uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * DEQ_UN;
    DeqIn in[DEQ_UN];
#pragma unroll
    for (uint32_t k = 0; k < DEQ_UN; ++k)
        if ((u0 + k) * 8 + (lane >> 3) < n32) in[k] = deq_load<FMT>(w, u0 + k, lane);
#pragma unroll
    for (uint32_t k = 0; k < DEQ_UN; ++k)
        if ((u0 + k) * 8 + (lane >> 3) < n32) {
            const float4 v = deq_vals<FMT>(in[k], lane);
            __builtin_nontemporal_store((f4a{v.x, v.y, v.z, v.w}), reinterpret_cast<f4a *>(out + (u0 + k) * 256 + 4 * lane));
        }
}

// A launch holds fewer than 2^32 threads, so 2^24 workgroups (2^35 outputs) and
// more go in several.
template <int FMT>
static int deq_go(const uint8_t * w, uint64_t n32, float * out, hipStream_t s) {
    constexpr uint64_t B32 = 8 * 4 * DEQ_UN, MOST = (1ull << 24) - 1;   // 32-weight blocks per workgroup; workgroups
    constexpr uint64_t BB = FMT == FMT_Q8_0 ? 34 : FMT == FMT_Q5_0 ? 22 : 0;   // bytes of a block
    constexpr uint64_t UB = BB ? 8 * BB : FMT == FMT_Q4_K ? 144 : FMT == FMT_Q6_K ? 210 : iq_block_bytes(FMT);   // of a unit
    while (n32) {
        const uint64_t nwg = min((n32 + B32 - 1) / B32, MOST), n = min(n32, nwg * B32);
        hipLaunchKernelGGL(k_dequant<FMT>, dim3((uint32_t)nwg), dim3(256), 0, s, w, n, out);
        if (int rc = hip_check(hipGetLastError(), "k_dequant launch")) return rc;
        n32 -= n;
        w += n / 8 * UB;                                          // (n is a multiple of 8 unless it is the last)
        out += n * 32;
    }
    return FLH_OK;
}

int launch_dequant(int fmt, const uint8_t * w, uint32_t rows, uint32_t cols,
                   float * out, hipStream_t s) {
    const uint64_t n32 = (uint64_t)rows * (cols / 32);
    switch (fmt) {
        case FMT_Q8_0: return deq_go<FMT_Q8_0>(w, n32, out, s);
        case FMT_Q5_0: return deq_go<FMT_Q5_0>(w, n32, out, s);
        case FMT_Q4_K: return deq_go<FMT_Q4_K>(w, n32, out, s);
        case FMT_Q6_K: return deq_go<FMT_Q6_K>(w, n32, out, s);
        case FMT_IQ2_XXS: return deq_go<FMT_IQ2_XXS>(w, n32, out, s);
        case FMT_IQ3_XXS: return deq_go<FMT_IQ3_XXS>(w, n32, out, s);
        default: return set_error(FLH_ERR_UNSUPPORTED, "dequant: format not supported");
    }
}

}  // namespace flh
