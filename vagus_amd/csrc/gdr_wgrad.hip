// Weight gradients of a layer's projections: dW[n][c] = sum_t dy[t][n] x[t][c] for up
// to WGRAD_MAX matrices dy that share the input x.  The output is small (a thousand
// rows and columns) and the sum long (every token of the batch), so a library product
// without a split sum leaves most CUs idle; here the tokens are split until the chip is
// full (about two workgroups per CU) and the fp32 partial products are added in a
// fixed order by wgrad_sum_kernel.
//
// A workgroup owns 256 rows n x 128 columns c for a run of tokens, 32 at a time: four
// waves of 128 x 64, 32 16x16x32 MFMAs per wave and step.  Both operands lie token-major,
// i.e. with the contraction index in the rows, so their fragments are transpose reads
// (ds_read_b64_tr_b16) of row-major LDS tiles: 24 of 8 bytes per lane and step, 48 KB of
// LDS reads and 24 KB of writes per workgroup and step against 512 MFMA cycles: close to
// the LDS's 128 bytes per clock, which bounds the loop (a 128 x 128 tile reads twice as much
// per MFMA).  Tile rows are unpadded with 16-byte unit u of row t at u ^ 2 (t mod 8): the
// eight rows a half wave reads 32 bytes of fall on distinct banks.  The next step's rows are
// loaded into registers during this step's products and stored to the other LDS buffer
// after them.  Measured for the seven projections of a KDA layer (dim 1024, 4 heads of
// 128 / 256) over 32,768 tokens: 491 us and 71 us of sums, 600 TFLOP/s, where the
// library's products took 1,440 us.  Tiles of one run of tokens sit on one XCD as far as the counts allow, so that
// its L2 serves the x and dy rows they share.
#include "gdr_chunk_layout.hpp"

namespace vgdr {

namespace {

constexpr int MT = 256, NT = 128, KT = 32;

// element offset of (row t, column c) in a swizzled tile of W columns
template <int W>
__device__ __forceinline__ int wg_at(int t, int c) {
    return t * W + ((((c >> 3) ^ (2 * (t & 7))) << 3) | (c & 7));
}

}  // namespace

template <typename E>
__global__ void __launch_bounds__(256, 2) wgrad_kernel(const WgradParams p) {
    using F = typename Elem<E>::frag;
    typedef E V8 __attribute__((ext_vector_type(8)));
    __shared__ __attribute__((aligned(16))) E sa[2][KT * MT];
    __shared__ __attribute__((aligned(16))) E sb[2][KT * NT];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, r = lane & 15;
    // (split, tile): consecutive ones on one XCD
    const int per = gridDim.x / 8, order = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    const int tiles = p.tiles_m * p.tiles_n;
    if (order >= tiles * p.splits) return;
    const int split = order / tiles, tile = order % tiles;
    const int mt = tile / p.tiles_n, c0 = tile % p.tiles_n * NT;
    int gi = 0;
    while (gi + 1 < p.n_groups && mt >= p.g[gi + 1].tile0) ++gi;
    const WgradGroup &gr = p.g[gi];
    const int n0 = (mt - gr.tile0) * MT;
    const int64_t t0 = (int64_t)split * p.split_len;
    const int64_t t1 = t0 + p.split_len < p.T ? t0 + p.split_len : p.T;
    const int steps = (int)((t1 - t0 + KT - 1) / KT);
    // columns past the matrix read its first ones: their products are not stored
    const E *dy = reinterpret_cast<const E *>(gr.dy), *x = reinterpret_cast<const E *>(p.x);
    const int ua = tid % (MT / 8), ra = tid / (MT / 8), ub = tid % (NT / 8), rb = tid / (NT / 8);
    const E *ap = dy + (n0 + 8 * ua < gr.n ? n0 + 8 * ua : 0);
    const E *bp = x + (c0 + 8 * ub < p.dim ? c0 + 8 * ub : 0);
    V8 va[4], vb[2];
    auto load = [&](int s) __attribute__((always_inline)) {
        const int64_t t = t0 + (int64_t)s * KT;
        unroll<4>([&](auto i) __attribute__((always_inline)) {
            const int64_t row = t + ra + 8 * decltype(i)::value;
            va[i] = *reinterpret_cast<const V8 *>(ap + (row < t1 ? row : t1 - 1) * gr.ld);
        });
        unroll<2>([&](auto i) __attribute__((always_inline)) {
            const int64_t row = t + rb + 16 * decltype(i)::value;
            vb[i] = *reinterpret_cast<const V8 *>(bp + (row < t1 ? row : t1 - 1) * p.ldx);
        });
    };
    auto store = [&](int s) __attribute__((always_inline)) {
        const int64_t left = t1 - t0 - (int64_t)s * KT;             // rows past the end are zeros
        unroll<4>([&](auto i) __attribute__((always_inline)) {
            const int row = ra + 8 * decltype(i)::value;
            *reinterpret_cast<V8 *>(sa[s & 1] + wg_at<MT>(row, 8 * ua)) = row < left ? va[i] : V8{};
        });
        unroll<2>([&](auto i) __attribute__((always_inline)) {
            const int row = rb + 16 * decltype(i)::value;
            *reinterpret_cast<V8 *>(sb[s & 1] + wg_at<NT>(row, 8 * ub)) = row < left ? vb[i] : V8{};
        });
    };
    const int wm = (wave & 1) * 128, wn = (wave >> 1) * 64;
    const bool busy = n0 + wm < gr.n && c0 + wn < p.dim;            // this wave has outputs
    f32x4 acc[8][4];
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int trow = 4 * g + (r >> 2), tcol = 4 * (r & 3);          // transpose-read source of this lane
    load(0);
    store(0);
    __syncthreads();
    for (int s = 0; s < steps; ++s) {
        if (s + 1 < steps) load(s + 1);
        if (busy) {
            const E *A = sa[s & 1], *B = sb[s & 1];
            F fb[4][2];
            unroll<4>([&](auto b) __attribute__((always_inline)) {
                const int c = wn + 16 * decltype(b)::value + tcol;
                fb[b][0] = ld_tr<E>(B + wg_at<NT>(trow, c));
                fb[b][1] = ld_tr<E>(B + wg_at<NT>(trow, c) + 16 * NT);
            });
            unroll<8>([&](auto a) __attribute__((always_inline)) {
                const int c = wm + 16 * decltype(a)::value + tcol;
                const F f0 = ld_tr<E>(A + wg_at<MT>(trow, c)), f1 = ld_tr<E>(A + wg_at<MT>(trow, c) + 16 * MT);
                unroll<4>([&](auto b) __attribute__((always_inline)) {
                    acc[a][b] = mfma_kb2(fb[b][0], f0, fb[b][1], f1, acc[a][b]);
                });
            });
        }
        if (s + 1 < steps) store(s + 1);
        __syncthreads();
    }
    // the last products' results pass their wait states on every path to the stores
    asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");
    if (!busy) return;
    // lane (g, r) holds row n = .. + r, columns .. + 4 g .. + 3 of each 16 x 16 tile
    typedef E E4 __attribute__((ext_vector_type(4)));
    unroll<8>([&](auto a) __attribute__((always_inline)) {
        const int n = n0 + wm + 16 * decltype(a)::value + r;
        unroll<4>([&](auto b) __attribute__((always_inline)) {
            const int c = c0 + wn + 16 * decltype(b)::value + 4 * g;
            const f32x4 v = acc[a][b];
            if (n >= gr.n || c >= p.dim) return;
            if (p.splits == 1)
                *reinterpret_cast<E4 *>(reinterpret_cast<E *>(gr.dw) + (int64_t)n * p.dim + c) =
                    E4{(E)v[0], (E)v[1], (E)v[2], (E)v[3]};
            else
                __builtin_nontemporal_store(v, reinterpret_cast<f32x4 *>(
                    p.part + ((int64_t)split * p.rows + gr.row0 + n) * p.dim + c));
        });
    });
}

// dW = the sum over the splits, in order; four columns per thread
template <typename E>
__global__ void __launch_bounds__(256) wgrad_sum_kernel(const WgradParams p) {
    typedef E E4 __attribute__((ext_vector_type(4)));
    const int64_t n4 = (int64_t)p.rows * p.dim / 4, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    const f32x4 *src = reinterpret_cast<const f32x4 *>(p.part) + i;
    f32x4 s = src[0];
#pragma unroll 4
    for (int k = 1; k < p.splits; ++k) s += src[(int64_t)k * n4];
    const int row = (int)(4 * i / p.dim), c = (int)(4 * i % p.dim);
    int gi = 0;
    while (gi + 1 < p.n_groups && row >= p.g[gi + 1].row0) ++gi;
    *reinterpret_cast<E4 *>(reinterpret_cast<E *>(p.g[gi].dw) + (int64_t)(row - p.g[gi].row0) * p.dim + c) =
        E4{(E)s[0], (E)s[1], (E)s[2], (E)s[3]};
}

// tiles and splits: the split sum fills about two workgroups per CU, of at least four
// steps each (a shorter run does not pay its partial tile's trip through memory)
void wgrad_plan(WgradParams &p) {
    p.rows = p.tiles_m = 0;
    for (int i = 0; i < p.n_groups; ++i) {
        p.g[i].row0 = p.rows;
        p.g[i].tile0 = p.tiles_m;
        p.rows += p.g[i].n;
        p.tiles_m += (p.g[i].n + MT - 1) / MT;
    }
    p.tiles_n = (p.dim + NT - 1) / NT;
    const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n, most = (p.T + 4 * KT - 1) / (4 * KT);
    int64_t s = 2 * device_cu_count() / tiles;
    s = s < 1 ? 1 : (s > most ? most : s);
    p.split_len = ((p.T + s - 1) / s + KT - 1) / KT * KT;
    p.splits = (int)((p.T + p.split_len - 1) / p.split_len);
}

template <typename E>
static hipError_t wgrad_t(const WgradParams &p, hipStream_t stream) {
    const int64_t groups = ((int64_t)p.tiles_m * p.tiles_n * p.splits + 7) / 8 * 8;
    if (groups > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL((wgrad_kernel<E>), dim3((unsigned)groups), dim3(256), 0, stream, p);
    if (p.splits > 1)
        hipLaunchKernelGGL((wgrad_sum_kernel<E>), dim3((unsigned)(((int64_t)p.rows * p.dim / 4 + 255) / 256)), dim3(256),
                           0, stream, p);
    return hipGetLastError();
}

hipError_t wgrad(int dtype, const WgradParams &p, hipStream_t stream) {
    if (dtype == 1) return wgrad_t<__bf16>(p, stream);
    if (dtype == 2) return wgrad_t<_Float16>(p, stream);
    return hipErrorInvalidValue;
}

}  // namespace vgdr
