// The layer's output epilogue, RMSNorm(o) x SiLU(gate) over the value head
// dim (linear_attention.py:814-825, norm_layer.py:15-24), as one HBM pass.
//
// Rows of dv elements (one per (token, head)) are cut into 16-byte units; a
// group of LPR = dv / VE consecutive lanes owns one row, so a wavefront covers
// 64 / LPR rows and every global access is one coalesced 16-byte load or
// store.  The sum of squares is reduced across the group with xor shuffles.
// The decode step applies the same epilogue inside recurrent_kernel, where a
// workgroup holds a whole row; the chunk kernels tile dv across workgroups,
// so prefill runs this pass after the scan.
#include "gdr_common.hpp"
#include "gdr_kernels.hpp"

namespace vgdr {

__device__ __forceinline__ float silu_(float x) { return x * sigmoidf_(x); }

template <typename E, int LPR>
__global__ void __launch_bounds__(256) norm_gate_kernel(const E *o, const E *__restrict__ gate,
                                                        const void *__restrict__ gamma, int gamma_f32, float eps,
                                                        E *out, int64_t n_rows) {
    constexpr int VE = 16 / (int)sizeof(E), DV = LPR * VE;
    typedef E V __attribute__((ext_vector_type(VE)));
    const int64_t gt = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = gt / LPR;
    const int part = (int)(gt % LPR);
    const bool live = row < n_rows;
    const int64_t off = (live ? row : n_rows - 1) * DV + part * VE;      // groups past the end re-read the last row
    // o and the gate stream through once: nontemporal
    const V xv = __builtin_nontemporal_load(reinterpret_cast<const V *>(o + off));
    const V gv = __builtin_nontemporal_load(reinterpret_cast<const V *>(gate + off));
    float x[VE], w[VE];
    float ss = 0.f;
    if (gamma_f32) {
        // VE fp32 values: one or two 16-byte loads (gamma is 16-byte aligned)
        const f32x4 *gp = reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(gamma) + part * VE);
#pragma unroll
        for (int q = 0; q < VE / 4; ++q) {
            const f32x4 g4 = gp[q];
#pragma unroll
            for (int e = 0; e < 4; ++e) w[4 * q + e] = g4[e];
        }
    } else {
        const V g = *reinterpret_cast<const V *>(reinterpret_cast<const E *>(gamma) + part * VE);
#pragma unroll
        for (int e = 0; e < VE; ++e) w[e] = (float)g[e];
    }
#pragma unroll
    for (int e = 0; e < VE; ++e) {
        x[e] = (float)xv[e];
        ss += x[e] * x[e];
    }
#pragma unroll
    for (int m = 1; m < LPR; m <<= 1) ss += __shfl_xor(ss, m);
    const float r = rsqrtf(ss * (1.f / DV) + eps);
    V y;
#pragma unroll
    for (int e = 0; e < VE; ++e) y[e] = (E)(x[e] * r * w[e] * silu_((float)gv[e]));
    if (live) __builtin_nontemporal_store(y, reinterpret_cast<V *>(out + off));
}

template <typename E>
static hipError_t norm_gate_t(const void *o, const Epilogue &ep, void *out, int64_t n_rows, int dv,
                              hipStream_t stream) {
    constexpr int VE = 16 / (int)sizeof(E);
    const int lpr = dv / VE;
    const int64_t blocks = (n_rows * lpr + 255) / 256;
    if (blocks == 0) return hipSuccess;
    const E *x = reinterpret_cast<const E *>(o), *g = reinterpret_cast<const E *>(ep.gate);
    E *y = reinterpret_cast<E *>(out);
#define VGDR_NG(L)                                                                                             \
    case L:                                                                                                     \
        hipLaunchKernelGGL((norm_gate_kernel<E, L>), dim3((unsigned)blocks), dim3(256), 0, stream, x, g, ep.gamma, \
                           ep.gamma_f32, ep.eps, y, n_rows);                                                    \
        break;
    switch (lpr) {
        VGDR_NG(1) VGDR_NG(2) VGDR_NG(4) VGDR_NG(8) VGDR_NG(16) VGDR_NG(32) VGDR_NG(64)
        default: return hipErrorInvalidValue;
    }
#undef VGDR_NG
    return hipGetLastError();
}

hipError_t norm_gate(int dtype, const void *o, const Epilogue &ep, void *out, int64_t n_rows, int dv,
                     hipStream_t stream) {
    if (dtype == 1) return norm_gate_t<__bf16>(o, ep, out, n_rows, dv, stream);
    if (dtype == 2) return norm_gate_t<_Float16>(o, ep, out, n_rows, dv, stream);
    return norm_gate_t<float>(o, ep, out, n_rows, dv, stream);
}

// The epilogue's gradients: with r = rsqrt(mean o^2 + eps), n = o r and s = SiLU(gate),
// from dy
//     do = r (m - n mean(m n)),  m = dy gamma s
//     dgate = dy n gamma SiLU'(gate),  dgamma = sum over rows of dy n s
// in one pass that reads o, gate and dy and writes do and dgate: bound by HBM.  The
// lane layout is the forward's; a workgroup walks over rows (its threads keep the
// channels they sum dgamma for), writes one partial dgamma row, and row_sums_kernel adds
// the workgroups' rows in a fixed order.  Measured at 131,072 rows of 256, bf16: 59 us
// (5.7 TB/s of the five tensors), where torch's expression and its autograd took 0.9 ms.
template <typename E, int LPR>
__global__ void __launch_bounds__(256) norm_gate_bwd_kernel(const E *__restrict__ o, const E *__restrict__ gate,
                                                            const E *__restrict__ gamma, float eps,
                                                            const E *__restrict__ dy, E *__restrict__ d_o,
                                                            E *__restrict__ dgate, float *__restrict__ part,
                                                            int64_t n_rows) {
    constexpr int VE = 16 / (int)sizeof(E), DV = LPR * VE, RPB = 256 / LPR;
    typedef E V __attribute__((ext_vector_type(VE)));
    const int tid = threadIdx.x, lane = tid % LPR;
    const V wv = reinterpret_cast<const V *>(gamma)[lane];
    float dw[VE];
#pragma unroll
    for (int e = 0; e < VE; ++e) dw[e] = 0.f;
    for (int64_t row0 = (int64_t)blockIdx.x * RPB; row0 < n_rows; row0 += (int64_t)gridDim.x * RPB) {
        const int64_t row = row0 + tid / LPR;
        const bool live = row < n_rows;
        const int64_t off = (live ? row : n_rows - 1) * DV + lane * VE;      // groups past the end re-read the last row
        const V ov = __builtin_nontemporal_load(reinterpret_cast<const V *>(o + off));
        const V gv = __builtin_nontemporal_load(reinterpret_cast<const V *>(gate + off));
        const V dv = __builtin_nontemporal_load(reinterpret_cast<const V *>(dy + off));
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < VE; ++e) ss += (float)ov[e] * (float)ov[e];
#pragma unroll
        for (int k = 1; k < LPR; k <<= 1) ss += __shfl_xor(ss, k);
        const float r = rsqrtf(ss * (1.f / DV) + eps);
        float n[VE], m[VE], mn = 0.f;
        V dg;
#pragma unroll
        for (int e = 0; e < VE; ++e) {
            const float w = (float)wv[e], x = (float)gv[e], d = (float)dv[e], sg = sigmoidf_(x), s = x * sg;
            n[e] = (float)ov[e] * r;
            m[e] = d * w * s;
            mn += m[e] * n[e];
            dg[e] = (E)(d * n[e] * w * (sg * (1.f + x * (1.f - sg))));
            dw[e] += live ? d * n[e] * s : 0.f;
        }
#pragma unroll
        for (int k = 1; k < LPR; k <<= 1) mn += __shfl_xor(mn, k);
        mn *= 1.f / DV;
        V dx;
#pragma unroll
        for (int e = 0; e < VE; ++e) dx[e] = (E)(r * (m[e] - n[e] * mn));
        if (live) {
            __builtin_nontemporal_store(dx, reinterpret_cast<V *>(d_o + off));
            __builtin_nontemporal_store(dg, reinterpret_cast<V *>(dgate + off));
        }
    }
    __shared__ float red[256][VE + 1];
#pragma unroll
    for (int e = 0; e < VE; ++e) red[tid][e] = dw[e];
    __syncthreads();
    for (int c = tid; c < DV; c += 256) {
        float s = 0.f;
        for (int k = 0; k < RPB; ++k) s += red[k * LPR + c / VE][c % VE];
        part[(int64_t)blockIdx.x * DV + c] = s;
    }
}

// out[i] = the sum over the rows of part [rows, n] in a fixed order: 64 columns per
// workgroup, its 16 waves take every 16th row (with four waves, 64 to 128 rows of
// 2,048 to 4,096 columns took 17 us of dependent loads)
template <typename E>
__global__ void __launch_bounds__(1024) row_sums_kernel(const float *__restrict__ part, E *__restrict__ out, int64_t n,
                                                        int64_t rows) {
    __shared__ float red[16][64];
    const int c = threadIdx.x % 64, w = threadIdx.x / 64;
    const int64_t i = (int64_t)blockIdx.x * 64 + c;
    float s = 0.f;
    if (i < n) {
#pragma unroll 4
        for (int64_t r = w; r < rows; r += 16) s += part[r * n + i];
    }
    red[w][c] = s;
    __syncthreads();
    if (w == 0 && i < n) {
#pragma unroll
        for (int k = 1; k < 16; ++k) s += red[k][c];
        out[i] = (E)s;
    }
}

hipError_t row_sums(int dtype, const float *part, void *out, int64_t n, int64_t rows, hipStream_t stream) {
    const int64_t groups = (n + 63) / 64;
    if (groups > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 grid((unsigned)groups), block(1024);
    if (dtype == 1) hipLaunchKernelGGL((row_sums_kernel<__bf16>), grid, block, 0, stream, part, (__bf16 *)out, n, rows);
    else if (dtype == 2) hipLaunchKernelGGL((row_sums_kernel<_Float16>), grid, block, 0, stream, part, (_Float16 *)out, n, rows);
    else hipLaunchKernelGGL((row_sums_kernel<float>), grid, block, 0, stream, part, (float *)out, n, rows);
    return hipGetLastError();
}

// workgroups of the epilogue's backward, one partial dgamma row each: four per CU keep
// HBM busy, and more only lengthen the sum over the partial rows
int norm_gate_bwd_blocks(int dtype, int64_t n_rows, int dv) {
    const int64_t rpb = 256 / (dv / (dtype == 0 ? 4 : 8)), need = (n_rows + rpb - 1) / rpb;
    return (int)(need < 1024 ? need : 1024);
}

template <typename E>
static hipError_t norm_gate_bwd_t(int dtype, const NormGateBwd &p, hipStream_t stream) {
    const int lpr = p.dv / (16 / (int)sizeof(E));
    const int blocks = norm_gate_bwd_blocks(dtype, p.n_rows, p.dv);
#define VGDR_NGB(L)                                                                                              \
    case L:                                                                                                       \
        hipLaunchKernelGGL((norm_gate_bwd_kernel<E, L>), dim3((unsigned)blocks), dim3(256), 0, stream,            \
                           reinterpret_cast<const E *>(p.o), reinterpret_cast<const E *>(p.gate),                 \
                           reinterpret_cast<const E *>(p.gamma), p.eps, reinterpret_cast<const E *>(p.dy),        \
                           reinterpret_cast<E *>(p.d_o), reinterpret_cast<E *>(p.dgate), p.part, p.n_rows);       \
        break;
    switch (lpr) {
        VGDR_NGB(1) VGDR_NGB(2) VGDR_NGB(4) VGDR_NGB(8) VGDR_NGB(16) VGDR_NGB(32) VGDR_NGB(64)
        default: return hipErrorInvalidValue;
    }
#undef VGDR_NGB
    const hipError_t rc = hipGetLastError();
    return rc != hipSuccess ? rc : row_sums(dtype, p.part, p.dgamma, p.dv, blocks, stream);
}

hipError_t norm_gate_bwd(int dtype, const NormGateBwd &p, hipStream_t stream) {
    if (dtype == 1) return norm_gate_bwd_t<__bf16>(dtype, p, stream);
    if (dtype == 2) return norm_gate_bwd_t<_Float16>(dtype, p, stream);
    return norm_gate_bwd_t<float>(dtype, p, stream);
}

// y = x rsqrt(sum x^2 + eps) over rows of LPR 16-byte units (the q, k producer,
// linear_attention.py:703-706), and its gradient dx = r (dy - y <y, dy>) with r formed
// again from x: one pass each, bound by HBM, the epilogue's lane layout.
template <typename E, int LPR, bool BWD>
__global__ void __launch_bounds__(256) l2norm_kernel(const E *__restrict__ x, const E *__restrict__ dy,
                                                     E *__restrict__ out, float eps, int64_t n_rows) {
    constexpr int VE = 16 / (int)sizeof(E), D = LPR * VE;
    typedef E V __attribute__((ext_vector_type(VE)));
    const int64_t gt = (int64_t)blockIdx.x * 256 + threadIdx.x, row = gt / LPR;
    const bool live = row < n_rows;
    const int64_t off = (live ? row : n_rows - 1) * D + gt % LPR * VE;       // groups past the end re-read the last row
    const V xv = *reinterpret_cast<const V *>(x + off);
    V dv{};
    if constexpr (BWD) dv = __builtin_nontemporal_load(reinterpret_cast<const V *>(dy + off));
    float ss = 0.f, xd = 0.f;
#pragma unroll
    for (int e = 0; e < VE; ++e) {
        ss += (float)xv[e] * (float)xv[e];
        if constexpr (BWD) xd += (float)xv[e] * (float)dv[e];
    }
#pragma unroll
    for (int k = 1; k < LPR; k <<= 1) {
        ss += __shfl_xor(ss, k);
        if constexpr (BWD) xd += __shfl_xor(xd, k);
    }
    const float r = rsqrtf(ss + eps);
    V o;
#pragma unroll
    for (int e = 0; e < VE; ++e)
        o[e] = BWD ? (E)(r * ((float)dv[e] - r * r * xd * (float)xv[e])) : (E)((float)xv[e] * r);
    if (live) *reinterpret_cast<V *>(out + off) = o;
}

template <typename E>
static hipError_t l2norm_t(const void *x, const void *dy, void *out, float eps, int64_t n_rows, int d,
                           hipStream_t stream) {
    const int lpr = d / (16 / (int)sizeof(E));
    const dim3 grid((unsigned)((n_rows * lpr + 255) / 256));
    const E *xp = reinterpret_cast<const E *>(x), *dp = reinterpret_cast<const E *>(dy);
    E *op = reinterpret_cast<E *>(out);
#define VGDR_L2(L)                                                                                                \
    case L:                                                                                                       \
        if (dy) hipLaunchKernelGGL((l2norm_kernel<E, L, true>), grid, dim3(256), 0, stream, xp, dp, op, eps, n_rows); \
        else hipLaunchKernelGGL((l2norm_kernel<E, L, false>), grid, dim3(256), 0, stream, xp, dp, op, eps, n_rows);   \
        break;
    switch (lpr) {
        VGDR_L2(1) VGDR_L2(2) VGDR_L2(4) VGDR_L2(8) VGDR_L2(16) VGDR_L2(32) VGDR_L2(64)
        default: return hipErrorInvalidValue;
    }
#undef VGDR_L2
    return hipGetLastError();
}

hipError_t l2norm(int dtype, const void *x, const void *dy, void *out, float eps, int64_t n_rows, int d,
                  hipStream_t stream) {
    if (dtype == 1) return l2norm_t<__bf16>(x, dy, out, eps, n_rows, d, stream);
    if (dtype == 2) return l2norm_t<_Float16>(x, dy, out, eps, n_rows, d, stream);
    return l2norm_t<float>(x, dy, out, eps, n_rows, d, stream);
}

// The pre-norm blocks' RMSNorm (norm_layer.py:15-23) with the residual add in
// front of it (block.py:57-59, :85-87): h = x + res rounded to E (the stream's
// new value, stored to x_out), then y = E(E(h * rsqrt(mean(h^2) + eps)) * gamma),
// the module's order of roundings.  One workgroup per row; a thread holds up to U
// 16-byte units of the row in registers between the two passes.  Decode feeds
// a handful of rows of a few thousand elements, so one kernel here replaces the
// eight elementwise and reduction kernels of the module's expression.
template <typename E, int U>
// x_out may be x or res itself (the residual stream updated in place), so
// neither input is declared __restrict__.
__global__ void __launch_bounds__(256) rms_norm_kernel(const E *x, const E *res, E *x_out,
                                                       const E *__restrict__ gamma, float eps, E *y, int dim) {
    constexpr int VE = 16 / (int)sizeof(E);
    typedef E V __attribute__((ext_vector_type(VE)));
    __shared__ float part[4];
    const int tid = threadIdx.x, nu = dim / VE;
    const int64_t base = (int64_t)blockIdx.x * dim;
    float h[U][VE];
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = tid + 256 * u;
        if (i < nu) {
            V hv = *reinterpret_cast<const V *>(x + base + (int64_t)i * VE);
            if (res) {
                const V rv = *reinterpret_cast<const V *>(res + base + (int64_t)i * VE);
#pragma unroll
                for (int e = 0; e < VE; ++e) hv[e] = (E)((float)hv[e] + (float)rv[e]);
            }
            if (x_out) *reinterpret_cast<V *>(x_out + base + (int64_t)i * VE) = hv;
#pragma unroll
            for (int e = 0; e < VE; ++e) {
                h[u][e] = (float)hv[e];
                ss += h[u][e] * h[u][e];
            }
        }
    }
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) ss += __shfl_xor(ss, m);
    if ((tid & 63) == 0) part[tid >> 6] = ss;
    __syncthreads();
    const float r = rsqrtf((part[0] + part[1] + part[2] + part[3]) / (float)dim + eps);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = tid + 256 * u;
        if (i < nu) {
            const V gv = *reinterpret_cast<const V *>(gamma + (int64_t)i * VE);
            V o;
#pragma unroll
            for (int e = 0; e < VE; ++e) o[e] = (E)((float)(E)(h[u][e] * r) * (float)gv[e]);
            *reinterpret_cast<V *>(y + base + (int64_t)i * VE) = o;
        }
    }
}

template <typename E>
static hipError_t rms_norm_t(const void *x, const void *res, void *x_out, const void *gamma, void *y, int64_t rows,
                             int dim, float eps, hipStream_t stream) {
    constexpr int VE = 16 / (int)sizeof(E);
    const int units = dim / VE;
    const E *xe = reinterpret_cast<const E *>(x), *re = reinterpret_cast<const E *>(res),
            *ge = reinterpret_cast<const E *>(gamma);
    E *xo = reinterpret_cast<E *>(x_out), *ye = reinterpret_cast<E *>(y);
    const dim3 grid((unsigned)rows);
    if (units <= 256)
        hipLaunchKernelGGL((rms_norm_kernel<E, 1>), grid, dim3(256), 0, stream, xe, re, xo, ge, eps, ye, dim);
    else if (units <= 512)
        hipLaunchKernelGGL((rms_norm_kernel<E, 2>), grid, dim3(256), 0, stream, xe, re, xo, ge, eps, ye, dim);
    else if (units <= 1024)
        hipLaunchKernelGGL((rms_norm_kernel<E, 4>), grid, dim3(256), 0, stream, xe, re, xo, ge, eps, ye, dim);
    else
        hipLaunchKernelGGL((rms_norm_kernel<E, 8>), grid, dim3(256), 0, stream, xe, re, xo, ge, eps, ye, dim);
    return hipGetLastError();
}

hipError_t rms_norm(int dtype, const void *x, const void *res, void *x_out, const void *gamma, void *y, int64_t rows,
                    int dim, float eps, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    if (dtype == 1) return rms_norm_t<__bf16>(x, res, x_out, gamma, y, rows, dim, eps, stream);
    if (dtype == 2) return rms_norm_t<_Float16>(x, res, x_out, gamma, y, rows, dim, eps, stream);
    return rms_norm_t<float>(x, res, x_out, gamma, y, rows, dim, eps, stream);
}

}  // namespace vgdr
