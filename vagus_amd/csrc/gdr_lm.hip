// Small kernels of the language model's one-token decode step around the
// layer kernels, each replacing a run of library calls or elementwise kernels:
//
//  * project_rows_kernel: the projections of one token's layer inputs, y =
//    [W_0 x | W_1 x | ...] for a few rows x and up to PROJ_MAX weights.  One launch
//    for six, which reads the weights where the modules hold them: no stacked copy
//    that a change of a parameter would have to reach.
//
//  * scalar_gates_kernel: the scalar gate and the beta logits of one decode
//    token (GatedDeltaNet._gates, linear_attention.py:719-721 and :734-735):
//    the projections W_a x and W_b x (rounded to the element type, as the
//    module's nn.Linear returns them), then
//        g    = -exp(A_log) * softplus(W_a x + dt_bias)      (fp32)
//        beta = W_b x                                         (fp32, the logits)
//    -exp(A_log) comes in precomputed.  The projections are 2H dot products of
//    dim elements per token: a wavefront owns eight of them, its lanes split
//    the row, and a shuffle reduction closes each one.
//
//  * swiglu_kernel: the FFN's SiLU(x1) x xgate (infra/components/ffn.py:48-50)
//    over [rows, 2 h] -> [rows, h], with the module's two roundings: SiLU's
//    result in the element type, then the product.
//
// The last two use the accurate expf / log1pf, as torch's softplus and SiLU do.
#include <type_traits>

#include "gdr_common.hpp"
#include "gdr_kernels.hpp"

namespace vgdr {

namespace {

// torch's softplus at beta 1, threshold 20
__device__ __forceinline__ float softplus_t(float x) { return x > 20.f ? x : log1pf(expf(x)); }

}  // namespace

// One wavefront per (token, OPW outputs): every lane loads its slice of the
// row and of the OPW weight rows at once, so the call costs about one trip to
// memory rather than one per output.
constexpr int GATE_OPW = 8;

template <typename E>
__global__ void __launch_bounds__(64) scalar_gates_kernel(const E *__restrict__ x, const E *__restrict__ w,
                                                          const float *__restrict__ neg_a,
                                                          const float *__restrict__ dt_bias, float *g, float *beta,
                                                          int dim, int H, int n_out) {
    constexpr int VE = 16 / (int)sizeof(E);
    typedef E V __attribute__((ext_vector_type(VE)));
    const int lane = threadIdx.x;
    const int64_t row = blockIdx.x;
    const int n0 = blockIdx.y * GATE_OPW;
    const int nu = dim / VE;
    const E *xr = x + row * dim;
    float acc[GATE_OPW];
#pragma unroll
    for (int j = 0; j < GATE_OPW; ++j) acc[j] = 0.f;
#pragma unroll 2
    for (int u = lane; u < nu; u += 64) {
        const V xv = *reinterpret_cast<const V *>(xr + (int64_t)u * VE);
        V wv[GATE_OPW];
#pragma unroll
        for (int j = 0; j < GATE_OPW; ++j) {
            const int n = n0 + j < n_out ? n0 + j : n_out - 1;            // rows past the end: reread the last
            wv[j] = *reinterpret_cast<const V *>(w + (int64_t)n * dim + (int64_t)u * VE);
        }
#pragma unroll
        for (int j = 0; j < GATE_OPW; ++j)
#pragma unroll
            for (int e = 0; e < VE; ++e) acc[j] += (float)xv[e] * (float)wv[j][e];
    }
#pragma unroll
    for (int j = 0; j < GATE_OPW; ++j) {
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) acc[j] += __shfl_xor(acc[j], m);
    }
    if (lane < GATE_OPW && n0 + lane < n_out) {
        float a = acc[0];
#pragma unroll
        for (int j = 1; j < GATE_OPW; ++j) a = lane == j ? acc[j] : a;
        const int n = n0 + lane;
        const float p = (float)(E)a;                                      // nn.Linear's output in E
        if (n < H) g[row * H + n] = neg_a[n] * softplus_t(p + dt_bias[n]);
        else beta[row * H + (n - H)] = p;
    }
}

template <typename E>
__global__ void __launch_bounds__(256) swiglu_kernel(const E *__restrict__ x, E *__restrict__ y, int64_t rows,
                                                     int hidden) {
    constexpr int VE = 16 / (int)sizeof(E);
    typedef E V __attribute__((ext_vector_type(VE)));
    const int nu = hidden / VE;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= rows * nu) return;
    const int64_t row = i / nu;
    const int u = (int)(i - row * nu);
    const E *xr = x + row * 2 * (int64_t)hidden;
    const V a = *reinterpret_cast<const V *>(xr + (int64_t)u * VE);
    const V b = *reinterpret_cast<const V *>(xr + hidden + (int64_t)u * VE);
    V o;
#pragma unroll
    for (int e = 0; e < VE; ++e) {
        const float s = (float)a[e] / (1.f + expf(-(float)a[e]));
        o[e] = (E)((float)(E)s * (float)b[e]);
    }
    *reinterpret_cast<V *>(y + row * (int64_t)hidden + (int64_t)u * VE) = o;
}

// y[b][col0_i + n] = sum_k W_i[n][k] x[b][k], fp32 sums in a fixed order, rounded once.
// A workgroup owns 16 MT weight rows and 16 NB rows of x; its NWV waves take every
// NWV-th 128-byte unit of k and meet in LDS.  A wave stages its units' rows through an
// LDS region of its own, eight rows to a load, and needs no barrier for it: fragments
// loaded straight from global memory touch 16 rows an instruction, and the address unit then
// bounds the kernel (64 rows, dim 2048: 16.5 against 15.5 us, dim 1024: 7.4 against 6.3).
// Bound by the weights' read up to about 32 rows, above by every workgroup's own read
// of x.  us for W_q .. W_g of one layer, bf16, weights from memory; beside it one library GEMM over a
// stacked copy, and one GEMM per weight:
//   dim 1024, 4,096 columns: 4 rows 4.7 (6.2, 23), 64: 6.3 (8.8, 33), 128: 8.0 (9.4, 32), 256: 13 (9.1, 32)
//   dim 2048, 8,192 columns: 4 rows 10.8 (12.4, 42), 32: 11.2 (12.3, 43), 64: 15.5 (12.9, 45), 128: 20.5 (15.5, 43),
//   256: 34 (24, 46).
template <typename E, int MT, int NB, int NWV>
__global__ void __launch_bounds__(64 * NWV) project_rows_kernel(const ProjectParams p) {
    constexpr int VE = 16 / (int)sizeof(E), UNIT = 8 * VE;               // a lane's load; a unit of k: 128 bytes
    typedef E V __attribute__((ext_vector_type(VE)));
    constexpr int R = 2 * (MT + NB), PITCH = UNIT + VE;                  // rows staged, 8 at a time; 16 bytes of padding
    __shared__ __attribute__((aligned(16))) E stage[NWV][8 * R * PITCH];
    __shared__ f32x4 red[NWV / 2][MT][NB][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, r = lane & 15;
    int gi = 0;
    while (gi + 1 < p.n_mats && (int)blockIdx.x >= p.m[gi + 1].tile0) ++gi;
    const ProjectMat &m = p.m[gi];
    const int n0 = ((int)blockIdx.x - m.tile0) * 16 * MT, b0 = blockIdx.y * 16 * NB;
    // a lane loads 16 bytes (piece l % 8 of a unit) of rows l / 8 + 8 i of W, then of x; rows past the
    // end are the last one again (their products are not stored)
    const int lr = lane >> 3, lk = VE * (lane & 7);
    const E *src[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int wr = n0 + 8 * i + lr, xr = b0 + 8 * (i - 2 * MT) + lr;
        src[i] = i < 2 * MT ? reinterpret_cast<const E *>(m.w) + (int64_t)(wr < m.n ? wr : m.n - 1) * p.dim
                            : reinterpret_cast<const E *>(p.x) + (int64_t)(xr < p.rows ? xr : p.rows - 1) * p.ldx;
    }
    f32x4 acc[MT][NB];
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int units = (p.dim + UNIT - 1) / UNIT;
    V in[R];
    auto load = [&](int u) __attribute__((always_inline)) {                        // zeros past the row's end
        const int k = UNIT * u + lk;
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const V v = *reinterpret_cast<const V *>(src[i] + (k < p.dim ? k : 0));
            in[i] = k < p.dim ? v : V{};
        }
    };
    E *mine = stage[wave];
    if (wave < units) load(wave);
    for (int u = wave; u < units; u += NWV) {
#pragma unroll
        for (int i = 0; i < R; ++i) *reinterpret_cast<V *>(mine + (8 * i + lr) * PITCH + lk) = in[i];
        // the rows are this wave's alone: LDS operations of one wave are in order, and only the compiler
        // has to keep the order
        asm volatile("" ::: "memory");
        if (u + NWV < units) load(u + NWV);
        V f[MT + NB][2];
#pragma unroll
        for (int t = 0; t < MT + NB; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                f[t][h] = *reinterpret_cast<const V *>(mine + (16 * t + r) * PITCH + VE * (g + 4 * h));
        asm volatile("" ::: "memory");
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int a = 0; a < MT; ++a)
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    if constexpr (sizeof(E) == 2) acc[a][b] = mfma_pair(f[a][h], f[MT + b][h], acc[a][b]);
                    else acc[a][b] = mfma_kb1(f[a][h], f[MT + b][h], acc[a][b]);
                }
    }
    // the last products' results pass their wait states on every path to their readers
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) asm volatile("" : "+v"(acc[a][b]));
    asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");
    // the waves' sums, halves onto halves, in a fixed order
#pragma unroll
    for (int half = NWV / 2; half > 0; half /= 2) {
        if (wave >= half && wave < 2 * half) {
#pragma unroll
            for (int a = 0; a < MT; ++a)
#pragma unroll
                for (int b = 0; b < NB; ++b) red[wave - half][a][b][lane] = acc[a][b];
        }
        __syncthreads();
        if (wave < half) {
#pragma unroll
            for (int a = 0; a < MT; ++a)
#pragma unroll
                for (int b = 0; b < NB; ++b) acc[a][b] += red[wave][a][b][lane];
        }
        __syncthreads();
    }
    if (wave > 0) return;
    // lane (g, r) holds weight rows n0 + 16 a + 4 g .. + 3 of row b0 + 16 b + r of x
    typedef E E4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int row = b0 + 16 * b + r;
        if (row >= p.rows) continue;
#pragma unroll
        for (int a = 0; a < MT; ++a) {
            const int n = n0 + 16 * a + 4 * g;
            const f32x4 s = acc[a][b];
            if (gi == p.beta_mat) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (n + j < m.n) p.beta[(int64_t)row * m.n + n + j] = (float)(E)s[j];
                continue;
            }
            E *y = reinterpret_cast<E *>(p.y) + (int64_t)row * p.ldy + m.col0 + n;
            if (n + 4 <= m.n) {
                *reinterpret_cast<E4 *>(y) = E4{(E)s[0], (E)s[1], (E)s[2], (E)s[3]};
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (n + j < m.n) y[j] = (E)s[j];
            }
        }
    }
}

template <typename E, int MT, int NB, int NWV>
static hipError_t project_rows_go(ProjectParams p, hipStream_t stream) {
    int tiles = 0;
    for (int i = 0; i < p.n_mats; ++i) {
        p.m[i].tile0 = tiles;
        tiles += (p.m[i].n + 16 * MT - 1) / (16 * MT);
    }
    const dim3 grid((unsigned)tiles, (unsigned)((p.rows + 16 * NB - 1) / (16 * NB)));
    hipLaunchKernelGGL((project_rows_kernel<E, MT, NB, NWV>), grid, dim3(64 * NWV), 0, stream, p);
    return hipGetLastError();
}

template <typename E>
static hipError_t project_rows_t(const ProjectParams &p, hipStream_t stream) {
    // us at 4 / 16 rows: dim 1024, 4,096 columns 4.7 / 4.8; dim 2048, 8,192 columns 10.8 / 11.3 (4 waves: 12.2, 12.4)
    if (p.rows <= 16) return project_rows_go<E, 1, 1, 8>(p, stream);
    // then 32 x 32 tiles, of eight waves while the grid is about one workgroup a CU (dim 1024, 64 rows: 6.3, four
    // waves 7.4; dim 2048, 32 rows: 11.2, 14.6), of four up to two (dim 2048, 64 rows: 15.5, eight waves 18.1,
    // 32 x 64 tiles 18.4); 32 x 64 tiles above (dim 2048: 128 rows 20.5, 26.6 with the smaller ones; 256: 34, 38)
    const int64_t cus = device_cu_count();
    int64_t grid = 0;
    for (int i = 0; i < p.n_mats; ++i) grid += (p.m[i].n + 31) / 32;
    grid *= (p.rows + 31) / 32;
    if (2 * grid <= 3 * cus) return project_rows_go<E, 2, 2, 8>(p, stream);
    if (4 * grid <= 9 * cus) return project_rows_go<E, 2, 2, 4>(p, stream);
    return project_rows_go<E, 2, 4, 4>(p, stream);
}

hipError_t project_rows(int dtype, const ProjectParams &p, hipStream_t stream) {
    if (dtype == 1) return project_rows_t<__bf16>(p, stream);
    if (dtype == 2) return project_rows_t<_Float16>(p, stream);
    return project_rows_t<float>(p, stream);
}

template <typename E>
static hipError_t scalar_gates_t(const void *x, const void *w, const float *neg_a, const float *dt_bias, float *g,
                                 float *beta, int64_t rows, int dim, int H, bool with_beta, hipStream_t stream) {
    const int n_out = with_beta ? 2 * H : H;
    hipLaunchKernelGGL((scalar_gates_kernel<E>), dim3((unsigned)rows, (unsigned)((n_out + GATE_OPW - 1) / GATE_OPW)),
                       dim3(64), 0, stream,
                       reinterpret_cast<const E *>(x), reinterpret_cast<const E *>(w), neg_a, dt_bias, g, beta, dim,
                       H, n_out);
    return hipGetLastError();
}

hipError_t scalar_gates(int dtype, const void *x, const void *w, const float *neg_a, const float *dt_bias, float *g,
                        float *beta, int64_t rows, int dim, int H, bool with_beta, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    if (dtype == 1) return scalar_gates_t<__bf16>(x, w, neg_a, dt_bias, g, beta, rows, dim, H, with_beta, stream);
    if (dtype == 2) return scalar_gates_t<_Float16>(x, w, neg_a, dt_bias, g, beta, rows, dim, H, with_beta, stream);
    return scalar_gates_t<float>(x, w, neg_a, dt_bias, g, beta, rows, dim, H, with_beta, stream);
}

template <typename E>
static hipError_t swiglu_t(const void *x, void *y, int64_t rows, int hidden, hipStream_t stream) {
    constexpr int VE = 16 / (int)sizeof(E);
    const int64_t blocks = (rows * (hidden / VE) + 255) / 256;
    hipLaunchKernelGGL((swiglu_kernel<E>), dim3((unsigned)blocks), dim3(256), 0, stream,
                       reinterpret_cast<const E *>(x), reinterpret_cast<E *>(y), rows, hidden);
    return hipGetLastError();
}

hipError_t swiglu(int dtype, const void *x, void *y, int64_t rows, int hidden, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    if (dtype == 1) return swiglu_t<__bf16>(x, y, rows, hidden, stream);
    if (dtype == 2) return swiglu_t<_Float16>(x, y, rows, hidden, stream);
    return swiglu_t<float>(x, y, rows, hidden, stream);
}

}  // namespace vgdr
