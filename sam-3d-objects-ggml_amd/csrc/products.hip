// products.hip -- the sparse conv of a nearest-upsampled level, computed on
// the coarse rows (spc_sparse_conv_products).
//
// A conv over the fine rows of an upsampled tensor (SparseResBlock3d with
// upsample: SP/spatial.py:75-105 then the 3x3x3 conv) reads coarse rows
// through the fine neighbour table, and the ~5 children of a coarse row
// multiply it by the same 27 tap matrices: (rows x taps) products repeat
// ~3x.  Here each product is formed once,
//     P[r][o] = W_o x[r]     (dense: [n_in, cin] x [cin, ntaps * cout], F32)
// and every output row adds its present taps' products in ascending tap
// order, y[t] = bias + sum_o P[idx(t, o)][o], before the conv's usual
// rounding and epilogue.  All partial sums stay F32, so the result differs
// from the implicit GEMM's by the order of F32 additions only.
//
// 12,516 coarse / 66,779 fine rows, C 2048 -> 128, bf16: the dense product
// does 177 GFLOP where the implicit GEMM runs 946 (padded tiles included):
// 1173 -> 215 us with the norm epilogue, 953 -> 204 without.
#include "common.h"

namespace spc {

namespace {

template <typename T>
struct Mma16;
template <>
struct Mma16<__bf16> {
    typedef bf16x8 frag;
    __device__ static floatx4 mma(frag a, frag b, floatx4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
    __device__ static uint32_t bits(float v) { return f32_to_bf16_bits(v); }
    __device__ static float val(uint32_t h) { return bf16_bits_to_f32((uint16_t)h); }
};
template <>
struct Mma16<_Float16> {
    typedef f16x8 frag;
    __device__ static floatx4 mma(frag a, frag b, floatx4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
    __device__ static uint32_t bits(float v) { return f32_to_f16_bits(v); }
    __device__ static float val(uint32_t h) { return f16_bits_to_f32((uint16_t)h); }
};

struct ProductArgs {
    const void* x;     // [m, cin]
    const void* w;     // packed 16-bit panels of ntaps taps
    float* p;          // [m, ntaps * cout]
    int64_t m;
    int32_t cin;
    int32_t cb_tap;    // 16-channel blocks per tap (cout / 16)
    int32_t cb_all;    // ntaps * cb_tap
    int32_t tiles_n;
    int64_t tiles;
    int64_t tiles_per_xcd;
};

// P = x W: 256 rows x 256 columns per workgroup of eight waves (two per
// SIMD, wave tiles of 128 rows x 64 columns), both operands staged 64
// channels at a time through two LDS buffers by LDS DMA (64 KB a stage,
// 128 KB in all), one barrier per stage: the next stage's sixty-four 1 KB
// DMA loads land behind the 2,048 matrix-core clocks of this one.
// Bounded by the matrix cores (1.28 PFLOP/s from 1024 to 2048 channels, 12,516
// rows x 3,456 columns); the fragment reads take 96 B/clk of LDS.
//   A stage  row r (128 bytes = eight 16-byte segments), segment s at unit
//            8 r + (s ^ (r & 7)): the 16-row fragment reads hit every bank.
//   B stage  the packed panels' 1 KB (16 channels x 32) fragments as they
//            are, flat 16-column blocks counted across taps, so narrow
//            convs fill the 256 columns with several taps.
constexpr int kPR = 256, kPC = 16;  // tile rows, 16-column blocks

template <typename T>
__global__ __launch_bounds__(512, 2) void products_kernel(ProductArgs a) {
    using M = Mma16<T>;
    __shared__ u32x4 As[2][kPR * 8];
    __shared__ u32x4 Bs[2][2 * kPC * 64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // XCD-major: each XCD takes a contiguous range of tiles, columns fastest
    const int64_t tile = (int64_t)(blockIdx.x & 7) * a.tiles_per_xcd + (blockIdx.x >> 3);
    if (tile >= a.tiles) return;
    const int64_t r0 = tile / a.tiles_n * kPR;
    const int cb0 = (int)(tile % a.tiles_n) * kPC;

    const uint32_t rowbytes = (uint32_t)a.cin * 2u;
    const int kch = a.cin / 32;          // 32-channel chunks (even)
    const int nst = kch / 2;             // stages
    const int64_t live = min<int64_t>(kPR, a.m - r0);
    const uint64_t xb = reinterpret_cast<uint64_t>(static_cast<const char*>(a.x) + r0 * rowbytes);
    const u32x4 xr = {(uint32_t)xb, (uint32_t)(xb >> 32) & 0xffffu, (uint32_t)(live * rowbytes), 0x00020000u};
    const uint64_t wb = reinterpret_cast<uint64_t>(a.w);
    const u32x4 wr = {(uint32_t)wb, (uint32_t)(wb >> 32) & 0xffffu,
                      (uint32_t)((int64_t)a.cb_all * kch * 1024), 0x00020000u};
    const uint32_t as0 = __builtin_amdgcn_readfirstlane(
        (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) u32x4*)&As[0][0]));
    const uint32_t bs0 = __builtin_amdgcn_readfirstlane(
        (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) u32x4*)&Bs[0][0]));
    // the wave's DMA blocks: A blocks wave + 8 j (8 rows each), B blocks
    // wave + 8 j (chunk (wave + 8 j) / 16 of the stage); out-of-range rows and
    // columns read zeros
    uint32_t av[4], bv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = (wave + 8 * j) * 8 + (lane >> 3);
        av[j] = row < live ? (uint32_t)row * rowbytes + (uint32_t)(((lane & 7) ^ (lane >> 3)) * 16)
                           : 0x80000000u;
        const int b = wave + 8 * j;
        const int cb = cb0 + (b & 15);
        bv[j] = 0x80000000u;
        if (cb < a.cb_all)
            bv[j] = (uint32_t)(((cb / a.cb_tap) * kch + (b >> 4)) * a.cb_tap + cb % a.cb_tap) * 1024u +
                    (uint32_t)lane * 16u;
    }
    auto stage = [&](int st, int buf) __attribute__((always_inline)) {
        const uint32_t ak = (uint32_t)st * 128u;
        const uint32_t bk = (uint32_t)st * 2u * (uint32_t)a.cb_tap * 1024u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t blk = (uint32_t)(wave + 8 * j) * 1024u;
            lds_dma_x4(xr, as0 + (uint32_t)buf * (kPR * 128u) + blk, av[j], ak);
            lds_dma_x4(wr, bs0 + (uint32_t)buf * (2u * kPC * 1024u) + blk, bv[j], bk);
        }
    };

    const int wrow = (wave >> 2) * 128, wcb = (wave & 3) * 4;
    floatx4 acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int arow = wrow + (lane & 15);

    stage(0, 0);
    dma_barrier<0>();
    for (int st = 0; st < nst; ++st) {
        const int buf = st & 1;
        if (st + 1 < nst) stage(st + 1, buf ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        typename M::frag af[2][8], bf[2][4];
        auto read = [&](int c) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                bf[c][j] = *reinterpret_cast<const typename M::frag*>(&Bs[buf][(c * kPC + wcb + j) * 64 + lane]);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                af[c][i] = *reinterpret_cast<const typename M::frag*>(
                    &As[buf][(arow + 16 * i) * 8 + ((4 * c + (lane >> 4)) ^ (lane & 7))]);
        };
        read(0);
        read(1);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = M::mma(bf[c][j], af[c][i], acc[i][j]);
        // the first chunk's reads, then the second's behind the first MFMAs
        __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
        for (int q = 0; q < 18; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 28, 0);
        dma_barrier<0>();
    }

    // lane: row lane % 16 of a block, columns 4 (lane / 16) .. + 3
    const int64_t ldp = (int64_t)a.cb_all * 16;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int row = arow + 16 * i;
        if (row >= live) continue;
        float* pr = a.p + (r0 + row) * ldp + (int64_t)(cb0 + wcb) * 16 + 4 * (lane >> 4);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (cb0 + wcb + j < a.cb_all) *reinterpret_cast<floatx4*>(pr + 16 * j) = acc[i][j];
    }
}

struct GatherArgs {
    const float* p;
    const void* bias;
    void* y;
    const int32_t* idx;            // token-major [n_out, ntaps] into P's rows
    int64_t n_out, n_in;
    int32_t ntaps, cout;
    int32_t epi_mode;
    float eps;
    const void* residual;
    const int32_t* residual_rows;
    int64_t n_residual;
    const float* scale;
    const float* shift;
    const int32_t* coords;
    int64_t n_batch;
};

// y[t] = epilogue(dt(bias + sum of the present taps' products)): G lanes a
// row, four channels each (4 G columns; grid.y walks wider rows), the row's
// indices spread over the group's lanes and shuffled out, nine taps' 16-byte
// loads in flight at once.  Bounded by the products it reads (66,779 rows x
// 21 taps x 512 B out of the caches: rows close in the table read the same
// products); blocks go XCD-major, so they find them in their own L2.
template <typename T, int G>
__global__ __launch_bounds__(256) void gather_products_kernel(GatherArgs a, int64_t blocks_per_xcd) {
    using M = Mma16<T>;
    constexpr int RPB = 256 / G;
    constexpr int NI = (32 + G - 1) / G;
    const int lane = threadIdx.x & 63;
    const int gl = threadIdx.x % G;
    const int64_t blk = (int64_t)(blockIdx.x & 7) * blocks_per_xcd + (blockIdx.x >> 3);
    const int64_t t = blk * RPB + threadIdx.x / G;
    const bool have = t < a.n_out;   // uniform per lane group; shuffles stay inside it
    const int c0 = blockIdx.y * (4 * G) + 4 * gl;
    int32_t id[NI];
#pragma unroll
    for (int k = 0; k < NI; ++k) {
        const int o = k * G + gl;
        id[k] = -1;
        if (have && o < a.ntaps) {
            const int32_t s = a.idx[t * a.ntaps + o];
            if (s >= 0 && s < a.n_in) id[k] = s;
        }
    }
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    if (a.bias) {  // element loads: the bias may lie at any element
        const uint16_t* b = static_cast<const uint16_t*>(a.bias) + c0;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = M::val(b[e]);
    }
    const int64_t ldp = (int64_t)a.ntaps * a.cout;
    const float* pc = a.p + c0;
    constexpr int B = 9;
#pragma unroll
    for (int o0 = 0; o0 < 27; o0 += B) {
        floatx4 v[B];
#pragma unroll
        for (int k = 0; k < B; ++k) {
            const int o = o0 + k;
            const int32_t s = __shfl(id[o / G], (lane & ~(G - 1)) | (o % G));
            v[k] = floatx4{0.f, 0.f, 0.f, 0.f};
            if (s >= 0) v[k] = *reinterpret_cast<const floatx4*>(pc + s * ldp + (int64_t)o * a.cout);
        }
#pragma unroll
        for (int k = 0; k < B; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] += v[k][e];
    }
    auto round = [](float v) __attribute__((always_inline)) { return M::val(M::bits(v)); };
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = round(acc[e]);
    if (a.epi_mode == SPC_EPI_NORM_MOD_SILU) {
        // the conv epilogue's steps (4 G == cout): LayerNorm without affine,
        // modulation and SiLU, each rounded to the feature dtype
        float s = (o[0] + o[1]) + (o[2] + o[3]);
#pragma unroll
        for (int off = G / 2; off > 0; off >>= 1) s += __shfl_xor(s, off);
        const float mean = s / (float)(4 * G);
        float q = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o[e] -= mean;
            q += o[e] * o[e];
        }
#pragma unroll
        for (int off = G / 2; off > 0; off >>= 1) q += __shfl_xor(q, off);
        if (!have) return;
        const float rstd = 1.0f / sqrtf(q / (float)(4 * G) + a.eps);
        const int64_t b = min(max((int64_t)a.coords[t * 4], (int64_t)0), a.n_batch - 1);
        const floatx4 sc = *reinterpret_cast<const floatx4*>(a.scale + b * a.cout + c0);
        const floatx4 sh = *reinterpret_cast<const floatx4*>(a.shift + b * a.cout + c0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float u = round(o[e] * rstd);
            o[e] = silu_f32(round(round(u * round(1.0f + sc[e])) + sh[e]));
        }
    } else if (a.epi_mode == SPC_EPI_RESIDUAL) {
        if (!have) return;
        int64_t rr = t;
        if (a.residual_rows) {
            const int32_t v = a.residual_rows[t];
            rr = (v >= 0 && v < a.n_residual) ? v : -1;
        }
        if (rr >= 0) {
            const u32x2 r = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(a.residual) +
                                                            rr * a.cout + c0);
            o[0] += M::val(r.x & 0xffffu);
            o[1] += M::val(r.x >> 16);
            o[2] += M::val(r.y & 0xffffu);
            o[3] += M::val(r.y >> 16);
        }
    }
    if (!have) return;
    __builtin_nontemporal_store(u32x2{M::bits(o[0]) | (M::bits(o[1]) << 16), M::bits(o[2]) | (M::bits(o[3]) << 16)},
                                reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.y) + t * a.cout + c0));
}

template <typename T>
hipError_t run_products(hipStream_t s, ProductArgs p, GatherArgs g) {
    p.tiles_n = (p.cb_all + kPC - 1) / kPC;
    p.tiles = ceil_div(p.m, kPR) * p.tiles_n;
    p.tiles_per_xcd = ceil_div(p.tiles, 8);
    if (p.tiles > 0) products_kernel<T><<<(unsigned)(p.tiles_per_xcd * 8), 512, 0, s>>>(p);
    const int w = g.cout % 128 == 0 ? 32 : g.cout % 64 == 0 ? 16 : 8;  // lanes a row
    const int64_t per = ceil_div(ceil_div(g.n_out, 256 / w), 8);
    const dim3 grid((unsigned)(per * 8), (unsigned)(g.cout / (4 * w)));
    if (w == 32) gather_products_kernel<T, 32><<<grid, 256, 0, s>>>(g, per);
    else if (w == 16) gather_products_kernel<T, 16><<<grid, 256, 0, s>>>(g, per);
    else gather_products_kernel<T, 8><<<grid, 256, 0, s>>>(g, per);
    return hipGetLastError();
}

}  // namespace
}  // namespace spc

using namespace spc;

extern "C" {

size_t spc_conv_products_workspace_bytes(int64_t n_in, int64_t cout) {
    if (n_in <= 0 || cout <= 0) return 0;
    return (size_t)n_in * 27u * (size_t)cout * sizeof(float);
}

int spc_sparse_conv_products(spc_stream_t stream, int dtype, const void* x, const void* w,
                             const void* bias, void* y, const int32_t* idx, int64_t n_out,
                             int64_t n_in, int64_t cin, int64_t cout, const spc_conv_epilogue* epi,
                             void* workspace, size_t workspace_bytes) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto bad16 = [](const void* q) { return ((uintptr_t)q & 15u) != 0; };
    if (dtype != SPC_BF16 && dtype != SPC_F16) {
        set_last_error("spc_sparse_conv_products: 16-bit features only");
        return SPC_BAD_ARG;
    }
    if (n_out < 0 || n_in < 0 || n_out > INT32_MAX || n_in > INT32_MAX || cin < 64 || cin % 64 != 0 ||
        cout < 32 || cout % 32 != 0 || cin > (1 << 20) || 27 * cin * cout * 2 >= ((int64_t)1 << 31)) {
        set_last_error("spc_sparse_conv_products: unsupported n_out=%lld n_in=%lld cin=%lld cout=%lld",
                       (long long)n_out, (long long)n_in, (long long)cin, (long long)cout);
        return SPC_BAD_SHAPE;
    }
    if (n_out == 0) return SPC_OK;
    if (!x || !w || !y || !idx || bad16(x) || bad16(w) || bad16(y)) {
        set_last_error("spc_sparse_conv_products: null / misaligned pointer");
        return SPC_BAD_ARG;
    }
    if (workspace_bytes < spc_conv_products_workspace_bytes(n_in, cout) ||
        (n_in > 0 && (!workspace || bad16(workspace)))) {
        set_last_error("spc_sparse_conv_products: workspace too small or misaligned");
        return SPC_OOM;
    }
    ProductArgs p{};
    p.x = x;
    p.w = w;
    p.p = static_cast<float*>(workspace);
    p.m = n_in;
    p.cin = (int32_t)cin;
    p.cb_tap = (int32_t)(cout / 16);
    p.cb_all = 27 * p.cb_tap;
    GatherArgs g{};
    g.p = p.p;
    g.bias = bias;
    g.y = y;
    g.idx = idx;
    g.n_out = n_out;
    g.n_in = n_in;
    g.ntaps = 27;
    g.cout = (int32_t)cout;
    if (epi) {
        g.epi_mode = epi->mode;
        g.eps = epi->eps;
        g.residual = epi->residual;
        g.residual_rows = epi->residual_rows;
        g.n_residual = epi->n_residual;
        g.scale = epi->scale;
        g.shift = epi->shift;
        g.coords = epi->coords;
        g.n_batch = epi->n_batch;
        if (g.epi_mode == SPC_EPI_NORM_MOD_SILU && cout != 32 && cout != 64 && cout != 128) {
            set_last_error("spc_sparse_conv_products: the norm epilogue needs cout 32, 64 or 128 "
                           "(got %lld)", (long long)cout);
            return SPC_BAD_SHAPE;
        }
        // (the conv's own checks)
        if ((g.epi_mode == SPC_EPI_RESIDUAL &&
             (!g.residual || bad16(g.residual) ||
              (g.residual_rows && (g.n_residual < 1 || g.n_residual > INT32_MAX)))) ||
            (g.epi_mode == SPC_EPI_NORM_MOD_SILU &&
             (!g.scale || !g.shift || !g.coords || bad16(g.scale) || bad16(g.shift) || g.n_batch < 1 ||
              !(g.eps >= 0.0f))) ||
            g.epi_mode < SPC_EPI_NONE || g.epi_mode > SPC_EPI_NORM_MOD_SILU) {
            set_last_error("spc_sparse_conv_products: a residual needs a 16-byte aligned pointer and "
                           "with residual_rows 1 <= n_residual <= INT32_MAX, the norm epilogue 16-byte "
                           "aligned scale and shift, coords, n_batch >= 1 and eps >= 0");
            return SPC_BAD_ARG;
        }
    }
    const hipError_t e = dtype == SPC_BF16 ? run_products<__bf16>(s, p, g) : run_products<_Float16>(s, p, g);
    SPC_HIP(e);
    return SPC_OK;
}

}  // extern "C"
