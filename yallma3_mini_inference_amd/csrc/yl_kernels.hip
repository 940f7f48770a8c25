// yl_kernels.hip -- standalone op kernels of the forward path (the per-op C
// ABI entry points and the embedding lookup).  The decode/prefill pipeline's
// fused kernels live in yl_gemv.hip, yl_attn.hip and yl_logits.hip.
//
// Each kernel reproduces the f32 operation order of the reference CPU path
// (paths relative to the reference repository):
//   quantize            quantization.rs:29-52, weight_type.rs:52-74
//   rmsnorm             util.rs:389-426
//   rope_gguf           util.rs:653-718
//   SwiGLU              forward.rs:220-237
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "yl_blocks.h"
#include "yl_device.h"
#include "yl_internal.h"

namespace yl {

constexpr int kThreads = 256;

// Vectors at any element address (callers' rows need not be aligned).
typedef float vf4u __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned int vu1u __attribute__((aligned(1)));
typedef unsigned int vu2u __attribute__((ext_vector_type(2), aligned(1)));

// RMSNorm (+ quantize) of `batch` rows, one workgroup per row; thread i owns
// 8-element chunks i + nt p (p < MP; nt threads: as many wavefronts as the
// row has chunks for, 4 at most), in registers throughout.  Bound: one
// memory round trip, then the reference's 8 serial lane sums (dim / 8
// dependent adds): their squares go to LDS lane by lane, and lanes 0-7 of
// wavefront 0 add them (lds_serial_sum).  Each thread normalizes and
// quantizes its chunks; 4 threads share a 32-group's maximum by DPP.
// Against an element per thread and pass, the row in LDS and a division per
// element: 500 rows of 2048 8.7 -> 4.5 us, 2048 rows of 8192 104 -> 36.6 us.
// (Always 256 threads: 2000 rows of 576 6.3 us, now 4.6.)
template <int QF, int MP>
__global__ __launch_bounds__(kThreads) void k_rmsnorm(const float* __restrict__ x, const float* __restrict__ w,
                                                      int dim, float eps, int nt, float* xn, int8_t* xq, float* xs) {
    extern __shared__ __align__(16) float sq[];   // [8][rowq_stride(dim)] squares
    __shared__ float ss_sh;
    const int t = blockIdx.x, tid = threadIdx.x, n8 = dim / 8, S = rowq_stride(dim);
    const float* xr = x + (size_t)t * dim;
    float v[MP][8];
#pragma unroll
    for (int p = 0; p < MP; p++) {
        const float* c = xr + 8 * (size_t)max(min(tid + p * nt, n8 - 1), 0);
        const vf4u a = n8 ? *reinterpret_cast<const vf4u*>(c) : vf4u{}, b = n8 ? *reinterpret_cast<const vf4u*>(c + 4) : vf4u{};
#pragma unroll
        for (int k = 0; k < 4; k++) { v[p][k] = a[k]; v[p][4 + k] = b[k]; }
    }
    float wv[MP][8];
#pragma unroll
    for (int p = 0; p < MP; p++) {
        const float* c = w + 8 * (size_t)max(min(tid + p * nt, n8 - 1), 0);
        const vf4u a = n8 ? *reinterpret_cast<const vf4u*>(c) : vf4u{}, b = n8 ? *reinterpret_cast<const vf4u*>(c + 4) : vf4u{};
#pragma unroll
        for (int k = 0; k < 4; k++) { wv[p][k] = a[k]; wv[p][4 + k] = b[k]; }
    }
#pragma unroll
    for (int p = 0; p < MP; p++) {
        const int i = tid + p * nt;
        if (i < n8)
#pragma unroll
            for (int k = 0; k < 8; k++) sq[k * S + i] = fmul(v[p][k], v[p][k]);
    }
    const int pad = rowq_chain_len(dim) - n8;
    for (int i = tid; i < 8 * pad; i += nt) sq[(i / pad) * S + n8 + i % pad] = 0.0f;
    __syncthreads();
    if (tid < 64) {
        const float ss = rowq_chain(dim, eps, sq);
        if (tid == 0) ss_sh = ss;
    }
    __syncthreads();
    const float ss = ss_sh;
#pragma unroll
    for (int p = 0; p < MP; p++) {
        const int i = tid + p * nt;
        float am = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            v[p][k] = fmul(wv[p][k], fmul(ss, v[p][k]));
            am = fmaxf(am, fabsf(v[p][k]));
        }
        if (xn && i < n8) {
            float* o = xn + (size_t)t * dim + 8 * i;
            *reinterpret_cast<vf4u*>(o) = vf4u{v[p][0], v[p][1], v[p][2], v[p][3]};
            *reinterpret_cast<vf4u*>(o + 4) = vf4u{v[p][4], v[p][5], v[p][6], v[p][7]};
        }
        if constexpr (QF >= 0) {
            // (dim % 32 == 0: a group's 4 threads are live or idle together)
            const float sc = group_scale<QF>(group_max(am, 4));
            int q[8];
            quant8<QF>(v[p], sc, q);
            if (i < n8) {
                *reinterpret_cast<vu2u*>(xq + (size_t)t * dim + 8 * i) =
                    vu2u{pack4(q[0], q[1], q[2], q[3]), pack4(q[4], q[5], q[6], q[7])};
                if ((i & 3) == 0) xs[(size_t)t * (dim / kGroup) + (i >> 2)] = sc;
            }
        }
    }
    // elements past the last whole chunk take no part and come out zero
    if (xn && tid < dim - 8 * n8) xn[(size_t)t * dim + 8 * n8 + tid] = 0.0f;
}

// Embedding lookup (base_transformer.rs:143-161: out-of-range ids give
// zeros; the row is the f32 dequantization q*scale of the Q8_0 table,
// transformer_llama_gguf.rs:459-473), written to x.
__global__ __launch_bounds__(kThreads) void k_embed(EmbQ8 e, const uint32_t* __restrict__ tokens,
                                                    float* __restrict__ x) {
    const int t = blockIdx.x;
    const int dim = e.dim;
    const uint32_t tok = tokens[t];
    const int lane = (int)(tok & 63u);
    const size_t tile = tok >> 6;
    // 8 elements per thread and pass, computed (loads issued) before any is stored
    for (int i0 = threadIdx.x; i0 < dim; i0 += 8 * (int)blockDim.x) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int i = min(i0 + k * (int)blockDim.x, dim - 1);
            v[k] = 0.0f;
            if (tok < (uint32_t)e.vocab) {
                const size_t off = emb_q_off(e.tiles, tile, i >> 4, lane) + (i & 15);
                if (e.fmt == 3) {
                    v[k] = fmul((float)e.q[off], e.d32[((size_t)(i / e.gs) * e.tiles + tile) * 64 + lane]);
                } else if (e.fmt == 1) {
                    v[k] = f16_to_f32(reinterpret_cast<const uint16_t*>(e.q)[off]);
                } else {
                    const int q = (int)(uint8_t)e.q[off] - 128;
                    v[k] = fmul((float)q, f16_to_f32(e.d[emb_d_idx(e.tiles, tile, i >> 5, lane)]));
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (i0 + k * (int)blockDim.x < dim) x[(size_t)t * dim + i0 + k * (int)blockDim.x] = v[k];
    }
}

// Activation quantization over a flat array: 4 threads per 32-group, 8
// consecutive elements each: 16-byte loads of whole lines.  One thread per
// group read 128 bytes apart: 4 M elements 7.6 us, now 5.1 (21 MB); a row of
// 2048 stays at the launch, 3.9 us.
template <int QF>
__global__ __launch_bounds__(kThreads) void k_quantize(int8_t* __restrict__ q, float* __restrict__ s,
                                                       const float* __restrict__ x, size_t groups) {
    const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x, n = 4 * groups;
    const size_t c = i < n ? i : n - 1;   // (idle threads repeat the last chunk: the maxima need every lane)
    const vf4u a = *reinterpret_cast<const vf4u*>(x + 8 * c), b = *reinterpret_cast<const vf4u*>(x + 8 * c + 4);
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    float am = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) am = fmaxf(am, fabsf(v[k]));
    const float sc = group_scale<QF>(group_max(am, 4));
    int qv[8];
    quant8<QF>(v, sc, qv);
    if (i < n) {
        *reinterpret_cast<vu2u*>(q + 8 * i) = vu2u{pack4(qv[0], qv[1], qv[2], qv[3]), pack4(qv[4], qv[5], qv[6], qv[7])};
        if ((i & 3) == 0) s[i >> 2] = sc;
    }
}

// out[c * out_ld + r] = in[r][c], 32x32 tiles through LDS.
__global__ __launch_bounds__(kThreads) void k_transpose(const float* __restrict__ in, float* __restrict__ out, int rows,
                                                        int cols, int out_ld) {
    __shared__ float tile[32][33];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    for (int i = threadIdx.x; i < 32 * 32; i += kThreads) {
        const int r = r0 + i / 32, c = c0 + i % 32;
        if (r < rows && c < cols) tile[i / 32][i % 32] = in[(size_t)r * cols + c];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 32 * 32; i += kThreads) {
        const int c = c0 + i / 32, r = r0 + i % 32;
        if (r < rows && c < cols) out[(size_t)c * out_ld + r] = tile[i % 32][i / 32];
    }
}

// RoPE on q [batch][n_heads*hd] and k [batch][n_kv_heads*hd] at positions
// pos+t, one thread per (head, pair).
__global__ void k_rope(const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                       const StepState* __restrict__ st, float* __restrict__ q, float* __restrict__ k,
                       int n_heads, int n_kv_heads, int hd) {
    const int t = blockIdx.y;
    const int half = hd / 2;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int nq = n_heads * half, nk = n_kv_heads * half;
    if (i >= nq + nk) return;
    const int pos = st->pos + t;
    const int pair = (i < nq ? i : i - nq) % half;
    const float c = cos_t[(size_t)pos * half + pair], s = sin_t[(size_t)pos * half + pair];
    float* v = i < nq ? q + (size_t)t * n_heads * hd + 2 * (size_t)i
                      : k + (size_t)t * n_kv_heads * hd + 2 * (size_t)(i - nq);
    const float v0 = v[0], v1 = v[1];
    v[0] = fmul(v0, c) - fmul(v1, s);
    v[1] = fadd(fmul(v0, s), fmul(v1, c));
}

// SwiGLU + group quantization: 8 threads per 32-group of hidden, 4
// consecutive elements each (16-byte loads, one division-free quantization
// per thread; bound by the exponentials' f64 steps and one round trip).
// Against an element per thread: 1000 rows of 8192 28.7 -> 16.5 us.
template <int QF>
__global__ __launch_bounds__(kThreads) void k_swiglu_quant(const float* __restrict__ gate, const float* __restrict__ up,
                                                           int hidden, int nt, float* __restrict__ h_f32,
                                                           int8_t* __restrict__ hq, float* __restrict__ hs) {
    const int t = blockIdx.y;
    const int i = 4 * (blockIdx.x * nt + threadIdx.x);
    const size_t off = (size_t)t * hidden + i;
    float g[4] = {}, u[4] = {}, h[4];
    if (i + 4 <= hidden) {
        const vf4u a = *reinterpret_cast<const vf4u*>(gate + off), b = *reinterpret_cast<const vf4u*>(up + off);
#pragma unroll
        for (int k = 0; k < 4; k++) { g[k] = a[k]; u[k] = b[k]; }
    } else {
        for (int k = 0; k < 4; k++)
            if (i + k < hidden) { g[k] = gate[off + k]; u[k] = up[off + k]; }
    }
    float am = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const float den = fadd(1.0f, expf_rn(-g[k]));
        h[k] = fmul(g[k] / den, u[k]);
        am = fmaxf(am, fabsf(h[k]));
    }
    if (h_f32) {
        if (i + 4 <= hidden) *reinterpret_cast<vf4u*>(h_f32 + off) = vf4u{h[0], h[1], h[2], h[3]};
        else
            for (int k = 0; k < 4; k++)
                if (i + k < hidden) h_f32[off + k] = h[k];
    }
    if constexpr (QF >= 0) {
        // (hidden % 32 == 0: a group's 8 threads are live or idle together)
        const float sc = group_scale<QF>(group_max(am, 8));
        int q[4];
        quant8<QF, 4>(h, sc, q);
        if (i < hidden) {
            *reinterpret_cast<vu1u*>(hq + off) = (unsigned)pack4(q[0], q[1], q[2], q[3]);
            if ((i & 31) == 0) hs[(size_t)t * (hidden / kGroup) + i / kGroup] = sc;
        }
    }
}

// Elementwise probes of the device arithmetic the forward path depends on:
// exp (expf_rn), correctly rounded sqrt and division, f16 widening.
__global__ void k_math_selftest(const float* __restrict__ x, int n, float* exp_out, float* sqrt_out,
                                float* div_out, float* f16_out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float v = x[i];
    exp_out[i] = expf_rn(v);
    sqrt_out[i] = sqrtf(fabsf(v));
    div_out[i] = 1.0f / v;
    f16_out[i] = f16_to_f32((uint16_t)(i & 0xffff));
}

// One wavefront per case: the serial sum of v[offs[c] .. offs[c+1]), in one
// call (seg 0) or in consecutive segments of seg values, each continuing
// from the previous segment's sum.
__global__ __launch_bounds__(64) void k_serial_sum_selftest(const float* __restrict__ v,
                                                            const uint32_t* __restrict__ offs, int seg, float* out) {
    const int c = blockIdx.x;
    const uint32_t a = offs[c], b = offs[c + 1];
    const int n = (int)(b - a);
    float s;
    if (seg <= 0) {
        s = wave_serial_sum(v + a, n);
    } else {
        s = 0.0f;
        for (int i = 0; i < n; i += seg) s = wave_serial_sum(v + a + i, min(seg, n - i), s);
    }
    if (threadIdx.x == 0) out[c] = s;
}

// seg_serial_sum (the decode attention's softmax denominator) over one case
// per workgroup of 4 wavefronts: the values staged into LDS with +0 up to
// the next multiple of 64, as the attention's exponential row holds them.
constexpr int kSegSumWaves = 4;
__global__ __launch_bounds__(64 * kSegSumWaves) void k_seg_sum_selftest(const float* __restrict__ v,
                                                                        const uint32_t* __restrict__ offs,
                                                                        float* out, unsigned* fault) {
    extern __shared__ __align__(16) float lds[];
    const int c = blockIdx.x;
    const uint32_t a = offs[c], b = offs[c + 1];
    const int n = (int)(b - a), pad = (n + 63) & ~63;
    float* sx = lds + pad;
    double* segsum = reinterpret_cast<double*>(sx + 2 * kSegSumWaves * 65);
    int* ctr = reinterpret_cast<int*>(segsum + 2 * kSegSumWaves);
    for (int i = threadIdx.x; i < pad; i += blockDim.x) lds[i] = i < n ? v[a + i] : 0.0f;
    if (threadIdx.x == 0) *ctr = 0;
    __syncthreads();
    seg_sums_f64<kSegSumWaves>(lds, n, segsum);
    __syncthreads();
    const float s = seg_serial_sum<kSegSumWaves>(lds, n, segsum, sx, ctr, 0, fault);
    if (threadIdx.x == 0) out[c] = s;
}

// seg_serial_sum_wide (the long-context softmax denominator) over one case
// per workgroup of 8 wavefronts, the values staged as the softmax kernel
// stages them (+0 up to the next multiple of 64).
constexpr int kSegSumWideWaves = 8;
__global__ __launch_bounds__(64 * kSegSumWideWaves) void k_seg_sum_wide_selftest(const float* __restrict__ v,
                                                                                 const uint32_t* __restrict__ offs,
                                                                                 float* out, unsigned* fault) {
    extern __shared__ __align__(16) float lds[];
    const int c = blockIdx.x;
    const uint32_t a = offs[c], b = offs[c + 1];
    const int n = (int)(b - a), pad = (n + 63) & ~63;
    float* sx = lds + pad + 64;
    double* segsum = reinterpret_cast<double*>(sx + 16 * 64 + 8);
    int* ctr = reinterpret_cast<int*>(segsum + kSegSumWideWaves);
    for (int i = threadIdx.x; i < pad + 64; i += blockDim.x) lds[i] = i < n ? v[a + i] : 0.0f;
    if (threadIdx.x == 0) *ctr = 0;
    __syncthreads();
    seg_sums_f64_wide<kSegSumWideWaves>(lds, n, segsum);
    __syncthreads();
    const float s = seg_serial_sum_wide<kSegSumWideWaves>(lds, n, segsum, sx, ctr, 0, fault);
    if (threadIdx.x == 0) out[c] = s;
}

// The step state of an op call: its first position (and token).
__global__ void k_set_state(StepState* st, int32_t pos, uint32_t token) {
    if (threadIdx.x == 0) {
        st->pos = pos;
        st->token = token;
        st->n_out = 0;
        st->logits_done = 0;
        st->argmax = 0ull;
    }
}

// A plain stream of two byte ranges (a GEMV class's weights and scales): each
// workgroup reads its contiguous slice of each with 16-byte non-temporal
// loads (as the GEMV), every lane issuing up to 16 loads before it uses any;
// the loaded words reach memory only through a comparison that is never
// true in practice, so no load is dropped.  Measurement only.
typedef unsigned int stream_u4 __attribute__((ext_vector_type(4)));
constexpr int kStreamAhead = 16;
__global__ __launch_bounds__(1024) void k_stream(const stream_u4* __restrict__ a, size_t na,
                                                 const stream_u4* __restrict__ b, size_t nb, unsigned* __restrict__ sink) {
    uint32_t x = 0;
    for (int part = 0; part < 2; part++) {
        const stream_u4* p = part ? b : a;
        const size_t n = part ? nb : na;
        const size_t per = (n + gridDim.x - 1) / gridDim.x;
        const size_t lo = (size_t)blockIdx.x * per, hi = lo + per < n ? lo + per : n;
        for (size_t i0 = lo + threadIdx.x; i0 < hi; i0 += (size_t)kStreamAhead * blockDim.x) {
            stream_u4 v[kStreamAhead];
#pragma unroll
            for (int k = 0; k < kStreamAhead; k++) {
                const size_t i = i0 + (size_t)k * blockDim.x;
                v[k] = __builtin_nontemporal_load(p + (i < hi ? i : i0));
            }
#pragma unroll
            for (int k = 0; k < kStreamAhead; k++)
                if (i0 + (size_t)k * blockDim.x < hi) x ^= v[k].x ^ v[k].y ^ v[k].z ^ v[k].w;
        }
    }
    if (x == 0x9e3779b9u) sink[blockIdx.x] = x;
}

// ------------------------------------------------------------- launchers --

hipError_t launch_stream(const void* a, size_t abytes, const void* b, size_t bbytes, int grid, int threads,
                         unsigned* sink, hipStream_t s) {
    if (grid <= 0 || threads <= 0 || threads > 1024 || threads % 64 || (size_t)grid > abytes / 16) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_stream, dim3(grid), dim3(threads), 0, s, reinterpret_cast<const stream_u4*>(a), abytes / 16,
                       reinterpret_cast<const stream_u4*>(b), bbytes / 16, sink);
    return hipGetLastError();
}

hipError_t launch_set_state(StepState* st, int32_t pos, uint32_t token, hipStream_t s) {
    hipLaunchKernelGGL(k_set_state, dim3(1), dim3(64), 0, s, st, pos, token);
    return hipGetLastError();
}

hipError_t launch_quantize(int fmt, int8_t* q, float* scale, const float* x, size_t n, hipStream_t s) {
    const size_t groups = n / kGroup;
    if (groups == 0) return hipSuccess;
    const dim3 grid((unsigned)((4 * groups + kThreads - 1) / kThreads));
    if (fmt == kQ8) hipLaunchKernelGGL((k_quantize<kQ8>), grid, dim3(kThreads), 0, s, q, scale, x, groups);
    else if (fmt == kQ4) hipLaunchKernelGGL((k_quantize<kQ4>), grid, dim3(kThreads), 0, s, q, scale, x, groups);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

template <int QF>
static void launch_rmsnorm_q(const float* x, const float* w, int dim, float eps, int batch, float* xn, int8_t* xq,
                             float* xs, hipStream_t s) {
    const size_t smem = 8 * (size_t)rowq_stride(dim) * sizeof(float);
    auto k = dim <= 8 * kThreads ? k_rmsnorm<QF, 1> : dim <= 16 * kThreads ? k_rmsnorm<QF, 2> : k_rmsnorm<QF, 4>;
    const int nt = std::min(kThreads, std::max(64, (dim / 8 + 63) & ~63));
    hipLaunchKernelGGL(k, dim3(batch), dim3(nt), smem, s, x, w, dim, eps, nt, xn, xq, xs);
}

hipError_t launch_rmsnorm(int qfmt, const float* x, const float* w, int dim, float eps, int batch, float* xn,
                          int8_t* xq, float* xs, hipStream_t s) {
    if (dim > 8192) return hipErrorInvalidValue;
    if (qfmt == kQ8) launch_rmsnorm_q<kQ8>(x, w, dim, eps, batch, xn, xq, xs, s);
    else if (qfmt == kQ4) launch_rmsnorm_q<kQ4>(x, w, dim, eps, batch, xn, xq, xs, s);
    else launch_rmsnorm_q<-1>(x, w, dim, eps, batch, xn, xq, xs, s);
    return hipGetLastError();
}

hipError_t launch_transpose(const float* in, float* out, int rows, int cols, int out_ld, hipStream_t s) {
    if (rows <= 0 || cols <= 0) return hipSuccess;
    if (out_ld < rows) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_transpose, dim3((cols + 31) / 32, (rows + 31) / 32), dim3(kThreads), 0, s, in, out, rows, cols,
                       out_ld);
    return hipGetLastError();
}

hipError_t launch_embed(const EmbQ8& e, const uint32_t* tokens, int batch, float* x, hipStream_t s) {
    hipLaunchKernelGGL(k_embed, dim3(batch), dim3(kThreads), 0, s, e, tokens, x);
    return hipGetLastError();
}

hipError_t launch_rope(const float* cos_t, const float* sin_t, const StepState* st, int batch, float* q, float* k,
                       int n_heads, int n_kv_heads, int head_size, hipStream_t s) {
    const int items = (n_heads + n_kv_heads) * (head_size / 2);
    const dim3 grid((items + kThreads - 1) / kThreads, batch);
    hipLaunchKernelGGL(k_rope, grid, dim3(kThreads), 0, s, cos_t, sin_t, st, q, k, n_heads, n_kv_heads, head_size);
    return hipGetLastError();
}

hipError_t launch_swiglu_quant(int qfmt, const float* gate, const float* up, int hidden, int batch, float* h_f32,
                               int8_t* hq, float* hs, hipStream_t s) {
    // workgroups of equal width, a row of 576 on 192 threads (256: 2000 rows
    // 5.0 us, f32 output only, against 4.5)
    const int chunks = (hidden + 3) / 4, nb = (chunks + kThreads - 1) / kThreads;
    const int nt = ((chunks + nb - 1) / nb + 63) & ~63;
    const dim3 grid(nb, batch), block(nt);
    if (qfmt == kQ8)
        hipLaunchKernelGGL((k_swiglu_quant<kQ8>), grid, block, 0, s, gate, up, hidden, nt, h_f32, hq, hs);
    else if (qfmt == kQ4)
        hipLaunchKernelGGL((k_swiglu_quant<kQ4>), grid, block, 0, s, gate, up, hidden, nt, h_f32, hq, hs);
    else
        hipLaunchKernelGGL((k_swiglu_quant<-1>), grid, block, 0, s, gate, up, hidden, nt, h_f32, hq, hs);
    return hipGetLastError();
}

hipError_t launch_math_selftest(const float* x, int n, float* exp_out, float* sqrt_out, float* div_out,
                                float* f16_out, hipStream_t s) {
    hipLaunchKernelGGL(k_math_selftest, dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0, s, x, n, exp_out,
                       sqrt_out, div_out, f16_out);
    return hipGetLastError();
}

// what a bounded wait that gives up does to the fault word
__global__ void k_raise_fault(unsigned* fault) {
    if (threadIdx.x == 0) __hip_atomic_store(fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
hipError_t launch_raise_fault(unsigned* fault, hipStream_t s) {
    hipLaunchKernelGGL(k_raise_fault, dim3(1), dim3(64), 0, s, fault);
    return hipGetLastError();
}

hipError_t launch_serial_sum_selftest(const float* v, const uint32_t* offs, int cases, int seg, float* out,
                                      hipStream_t s) {
    if (cases <= 0) return hipSuccess;
    if (seg == -2) {
        // the wide segmented sum: LDS for the longest case
        std::vector<uint32_t> h((size_t)cases + 1);
        hipError_t e = hipMemcpy(h.data(), offs, h.size() * sizeof(uint32_t), hipMemcpyDeviceToHost);
        if (e != hipSuccess) return e;
        uint32_t mx = 0;
        for (int c = 0; c < cases; c++) mx = std::max(mx, h[c + 1] - h[c]);
        const size_t smem = ((((size_t)mx + 63) & ~(size_t)63) + 64 + 16 * 64 + 8 + 2 * kSegSumWideWaves + 4) * 4;
        if (smem > 150 * 1024) return hipErrorInvalidValue;
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_seg_sum_wide_selftest),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_seg_sum_wide_selftest, dim3(cases), dim3(64 * kSegSumWideWaves), smem, s, v, offs, out,
                           wait_fault_word(false));
        return hipGetLastError();
    }
    if (seg < 0) {
        // the segmented sum: LDS for the longest case
        std::vector<uint32_t> h((size_t)cases + 1);
        hipError_t e = hipMemcpy(h.data(), offs, h.size() * sizeof(uint32_t), hipMemcpyDeviceToHost);
        if (e != hipSuccess) return e;
        uint32_t mx = 0;
        for (int c = 0; c < cases; c++) mx = std::max(mx, h[c + 1] - h[c]);
        const size_t smem = (((size_t)mx + 63) & ~(size_t)63) * 4 + (2 * kSegSumWaves * 65 + 4 * kSegSumWaves + 4) * 4;
        if (smem > 150 * 1024) return hipErrorInvalidValue;
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_seg_sum_selftest),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_seg_sum_selftest, dim3(cases), dim3(64 * kSegSumWaves), smem, s, v, offs, out,
                           wait_fault_word(false));
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_serial_sum_selftest, dim3(cases), dim3(64), 0, s, v, offs, seg, out);
    return hipGetLastError();
}

}  // namespace yl
