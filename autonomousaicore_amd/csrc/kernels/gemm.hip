// GEMM for the Linear layers: C = alpha * op(A) op(B) + beta * C + R.
//
// Replaces the reference's GEMM backend (src/cuda/cuda_gemm.cu:241-398, called from
// src/ops/matmul.cpp:25-52): one launch per product instead of one per batch slice, no
// weight transpose copy (op() reads either layout), fp32 accumulation, and the residual add
// of TransformerBlock (include/nn/transformer_block.hpp:26-36) fused into the epilogue.
//
// This file holds the dispatch (tile shape, split-K, grouped and expert-ragged launches), the
// split-K reduction and the SIMT kernel; the bf16 MFMA kernels are in gemm_kernels.inc,
// instantiated per operand layout and output type by gemm_{nt,nn,tn,tt}_{bf16,f32}.hip.
// fp32 products run gemm_f32.hip, most of up to 64 rows of x W^T gemm_skinny.hip; fp32 operands with bf16
// output and bf16 operands whose layout the matrix kernels do not take, a plain SIMT tiled kernel.
#include "gemm.hpp"

#include <algorithm>
#include <vector>
#include <type_traits>

#include "common.hpp"
#include "gemm_launch.hpp"
#include "kernels.hpp"
#include "../runtime/memory_pool.hpp"

namespace aic::hip {

namespace {

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The 256-thread block's sum of every thread's (acc, nf) into *out / *out_nf: a fixed butterfly
// within each wave, then the four waves in order.  Every thread of the block must call it.
__device__ __forceinline__ void sq_block256(double acc, int nf, double* out, int* out_nf) {
    __shared__ double sd[4];
    __shared__ int sn[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        acc += __shfl_xor(acc, o);
        nf |= __shfl_xor(nf, o);
    }
    if ((threadIdx.x & 63) == 0) {
        sd[threadIdx.x >> 6] = acc;
        sn[threadIdx.x >> 6] = nf;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        *out = ((sd[0] + sd[1]) + sd[2]) + sd[3];
        *out_nf = sn[0] | sn[1] | sn[2] | sn[3];
    }
}

__device__ __forceinline__ void sq_add1(double& acc, int& nf, float v) {
    acc += static_cast<double>(v * v);
    nf |= (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u;
}

// V partials of consecutive elements, summed over the K parts in part order.
template <int V>
struct alignas(4 * V) Partials {
    float v[V];
    __device__ __forceinline__ void add(const Partials& p) {
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] += p.v[e];
    }
};
template <int V>
__device__ __forceinline__ Partials<V> sum_parts(const float* P, int splits, int64_t pz) {
    auto part = [&](int z) { return *reinterpret_cast<const Partials<V>*>(P + z * pz); };
    Partials<V> acc = part(0);
    int z = 1;
    // eight loads in flight, added in z order
    for (; z + 8 <= splits; z += 8) {
        Partials<V> p[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) p[u] = part(z + u);
#pragma unroll
        for (int u = 0; u < 8; ++u) acc.add(p[u]);
    }
    Partials<V> rest[7];
#pragma unroll
    for (int u = 0; u < 7; ++u)
        if (z + u < splits) rest[u] = part(z + u);
#pragma unroll
    for (int u = 0; u < 7; ++u)
        if (z + u < splits) acc.add(rest[u]);
    return acc;
}

// C = alpha * sum_z P[z] + beta * C + R over the split-K partials P [splits][M][N] (fp32,
// summed in z order: deterministic); with sq, each block also writes the sum of squares of
// the values it stored (one slot per block).  V elements of a row per thread: 4 (16-byte loads) where
// rows and bases allow it, else 1.  Block (x, y) takes every gridDim.y-th stripe of 256 V elements of
// the tile that the product's block x formed (tile x tile, in its order), so that where the tile
// count is a multiple of 8 the partials are read on the XCD, from the L2, that wrote them:
// 256x2048 in four parts of K 512, product and reduction, 12.3 us, 15.0 with 16-byte loads in row
// order; 256x2304 14.0 (17.1 with 4-byte loads in row order), 1000x768 in four of 512 14.6 (17.4).
template <typename CT, int V>
__global__ __launch_bounds__(256) void splitk_reduce_k(const float* __restrict__ P, int splits, int64_t pz, int M, int N,
                                                       int tile, int tiles_m, int tiles_n, float alpha, float beta,
                                                       CT* C, int64_t ldc, const CT* R, int64_t ldr, double* sq,
                                                       int* sq_nf) {
    struct alignas(sizeof(CT) * V) CV {
        CT v[V];
    };
    int tm, tn;
    tile_of(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn);
    const int rows = 256 * V / tile, n = tn * tile + static_cast<int>(threadIdx.x) * V % tile;
    const int end = n < N ? min((tm + 1) * tile, M) : 0;
    double sqa = 0.0;
    int sqf = 0;
    for (int m = tm * tile + static_cast<int>(blockIdx.y) * rows + static_cast<int>(threadIdx.x) * V / tile; m < end;
         m += rows * static_cast<int>(gridDim.y)) {
        const Partials<V> acc = sum_parts<V>(P + static_cast<int64_t>(m) * N + n, splits, pz);
        CT* c = C + static_cast<int64_t>(m) * ldc + n;
        CV old{}, res{}, out;
        if (beta != 0.0f) old = *reinterpret_cast<const CV*>(c);
        if (R) res = *reinterpret_cast<const CV*>(R + static_cast<int64_t>(m) * ldr + n);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            float v = alpha * acc.v[e];
            if (beta != 0.0f) v += beta * ld(old.v, e);
            if (R) v += ld(res.v, e);
            st(out.v, e, v);
            if (sq) sq_add1(sqa, sqf, v);  // fp32 C: the stored value
        }
        *reinterpret_cast<CV*>(c) = out;
    }
    if (sq) {
        const unsigned slot = blockIdx.y * gridDim.x + blockIdx.x;
        sq_block256(sqa, sqf, sq + slot, sq_nf + slot);
    }
}

// The same for at most kFewResults elements, one per thread in row order: finding the tile costs more than
// their sums, and a tile's stripes leave most lanes of narrow rows idle.  Product and reduction, in tile
// order and here: 65x16 over K 5632 12.1 and 11.0 us, 128x16 over 2048 11.4 and 10.5, 65x768 over 2048
// 10.8 and 10.1, 8192x16 over 1536 12.8 and 11.9, 1024x64 over 2048 14.6 and 14.3; from 131072 elements up
// the order of the tiles pays.
constexpr int64_t kFewResults = 131072;
template <typename CT>
__global__ __launch_bounds__(256) void splitk_reduce_few_k(const float* __restrict__ P, int splits, int M, int N,
                                                           float alpha, float beta, CT* C, int64_t ldc, const CT* R,
                                                           int64_t ldr, double* sq, int* sq_nf) {
    const int i = static_cast<int>(blockIdx.x * 256 + threadIdx.x);
    double sqa = 0.0;
    int sqf = 0;
    if (i < M * N) {
        const int m = i / N, n = i % N;
        const int64_t at = static_cast<int64_t>(m) * ldc + n;
        float v = alpha * sum_parts<1>(P + i, splits, static_cast<int64_t>(M) * N).v[0];
        if (beta != 0.0f) v += beta * ld(C, at);
        if (R) v += ld(R, static_cast<int64_t>(m) * ldr + n);
        st(C, at, v);
        if (sq) sq_add1(sqa, sqf, v);
    }
    if (sq) sq_block256(sqa, sqf, sq + blockIdx.x, sq_nf + blockIdx.x);
}

// Sums of squares of the fp32 matrix C [M, N] (leading dimension ldc), one slot per block: the
// products whose path has no such epilogue.
__global__ __launch_bounds__(256) void sq_matrix_k(const float* __restrict__ C, int64_t ldc, int M, int N, double* sq,
                                                   int* sq_nf) {
    const int64_t total = static_cast<int64_t>(M) * N;
    double sqa = 0.0;
    int sqf = 0;
    for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < total; i += static_cast<int64_t>(gridDim.x) * 256)
        sq_add1(sqa, sqf, C[(i / N) * ldc + i % N]);
    sq_block256(sqa, sqf, sq + blockIdx.x, sq_nf + blockIdx.x);
}

// ---------------------------------------------------------------------------------------
// SIMT tiled GEMM (odd shapes).  64x64 tile, 256 threads, 4x4 each.
// ---------------------------------------------------------------------------------------
template <typename T, typename CT>
__global__ __launch_bounds__(256) void gemm_simt(const T* __restrict__ A, const T* __restrict__ B, CT* C,
                                                  const CT* R, int64_t lda, int64_t ldb, int64_t ldc, int64_t ldr,
                                                  int M, int N, int K, int ta, int tb, float alpha, float beta) {
    constexpr int TS = 64, TK = 16;
    __shared__ float As[TK][TS + 4];
    __shared__ float Bs[TK][TS + 4];
    const int m0 = blockIdx.y * TS, n0 = blockIdx.x * TS;
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += TK) {
        for (int e = threadIdx.x; e < TS * TK; e += 256) {
            const int r = e / TK, kk = e % TK;
            const int m = m0 + r, k = k0 + kk;
            float a = 0.0f;
            if (m < M && k < K) a = ld(A, ta ? static_cast<int64_t>(k) * lda + m : static_cast<int64_t>(m) * lda + k);
            As[kk][r] = a;
            const int n = n0 + r;
            float b = 0.0f;
            if (n < N && k < K) b = ld(B, tb ? static_cast<int64_t>(n) * ldb + k : static_cast<int64_t>(k) * ldb + n);
            Bs[kk][r] = b;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < TK; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= N) continue;
            const int64_t ci = static_cast<int64_t>(m) * ldc + n;
            float v = alpha * acc[i][j];
            if (beta != 0.0f) v += beta * ld(C, ci);
            if (R) v += ld(R, static_cast<int64_t>(m) * ldr + n);
            st(C, ci, v);
        }
    }
}

template <int BM, int BN, int BK, int S, typename CT>
void dispatch_ragged(const RaggedArgs& r, hipStream_t s) {
    if (r.ragged_k) gemm_impl::launch_dma_ragged<BM, BN, BK, S, true, false, CT>(r, s);
    else if (r.g.transB) gemm_impl::launch_dma_ragged<BM, BN, BK, S, false, true, CT>(r, s);
    else gemm_impl::launch_dma_ragged<BM, BN, BK, S, false, false, CT>(r, s);
}

template <int BM, int BN, int BK, int S, typename CT>
void dispatch_grouped(const GemmArgs* a, int n, hipStream_t s) {
    if (!a[0].transA && a[0].transB) gemm_impl::launch_dma_grouped<BM, BN, BK, S, false, true, CT>(a, n, s);
    else if (!a[0].transA && !a[0].transB) gemm_impl::launch_dma_grouped<BM, BN, BK, S, false, false, CT>(a, n, s);
    else if (a[0].transA && !a[0].transB) gemm_impl::launch_dma_grouped<BM, BN, BK, S, true, false, CT>(a, n, s);
    else gemm_impl::launch_dma_grouped<BM, BN, BK, S, true, true, CT>(a, n, s);
}

template <int BM, int BN, int BK, int S, typename CT>
void dispatch_dma(const GemmArgs& a, hipStream_t s, int splits = 1, float* part = nullptr) {
    if (!a.transA && a.transB) gemm_impl::launch_dma<BM, BN, BK, S, false, true, CT>(a, s, splits, part);
    else if (!a.transA && !a.transB) gemm_impl::launch_dma<BM, BN, BK, S, false, false, CT>(a, s, splits, part);
    else if (a.transA && !a.transB) gemm_impl::launch_dma<BM, BN, BK, S, true, false, CT>(a, s, splits, part);
    else gemm_impl::launch_dma<BM, BN, BK, S, true, true, CT>(a, s, splits, part);
}

template <int BM, int BN, typename CT>
void dispatch_trans(const GemmArgs& a, hipStream_t s) {
    if (!a.transA && a.transB) gemm_impl::launch_mfma<BM, BN, false, true, CT>(a, s);
    else if (!a.transA && !a.transB) gemm_impl::launch_mfma<BM, BN, false, false, CT>(a, s);
    else if (a.transA && !a.transB) gemm_impl::launch_mfma<BM, BN, true, false, CT>(a, s);
    else gemm_impl::launch_mfma<BM, BN, true, true, CT>(a, s);
}

template <typename T, typename CT>
void launch_simt(const GemmArgs& a, hipStream_t s) {
    dim3 grid(static_cast<unsigned>((a.N + 63) / 64), static_cast<unsigned>((a.M + 63) / 64));
    hipLaunchKernelGGL((gemm_simt<T, CT>), grid, dim3(256), 0, s, static_cast<const T*>(a.A),
                       static_cast<const T*>(a.B), static_cast<CT*>(a.C), static_cast<const CT*>(a.R), a.lda, a.ldb,
                       a.ldc, a.ldr, static_cast<int>(a.M), static_cast<int>(a.N), static_cast<int>(a.K), a.transA,
                       a.transB, a.alpha, a.beta);
    AIC_LAUNCH_CHECK("gemm_simt");
}

}  // namespace

bool gemm_mfma_eligible(const GemmArgs& a) {
    if (a.ab != DType::BFloat16) return false;
    // K in 16-byte pieces where an operand is contiguous along it (a weight gradient's are not)
    if (((!a.transA || a.transB) && a.K % 8) || a.lda % 8 || a.ldb % 8 || !aligned16(a.A) || !aligned16(a.B)) return false;
    if (a.transA && a.M % 8) return false;
    if (!a.transB && a.N % 8) return false;
    return true;
}

bool gemm_q4_eligible(const GemmArgs& a) {
    if (!a.Bq || !a.Bscale || a.ab != DType::BFloat16 || a.transA) return false;
    if (a.K <= 0 || a.K % 64 || a.M < 1 || a.N < 1 || a.lda % 8 || !aligned16(a.A) || !aligned16(a.Bq)) return false;
    if (a.scale_t != DType::Float16 || reinterpret_cast<uintptr_t>(a.Bscale) % 4) return false;
    if (a.group <= 0 || a.group % 64 || a.group >= (int64_t{1} << 31) || a.ldb % 64) return false;
    if (!a.transB && (a.N % 64 || a.ldb < a.N)) return false;
    if (a.transB && a.ldb < a.K) return false;
    const int64_t rows = a.transB ? a.N : a.K;
    return rows * a.ldb / 64 < (int64_t{1} << 32);
}

bool gemm_dma_eligible(const GemmArgs& a) {
    if (!gemm_mfma_eligible(a)) return false;
    // (row copies clamp to the last row; a row-contiguous operand has at least 8 columns by then)
    if (((!a.transA || a.transB) && a.K % 64) || a.M < 1 || a.N < 1) return false;
    if (a.lda >= (int64_t{1} << 23) || a.ldb >= (int64_t{1} << 23)) return false;  // 32-bit copy offsets
    return true;
}

namespace {

size_t partial_bytes(const GemmArgs& a, int parts) { return sizeof(float) * parts * a.M * a.N; }

// C = alpha * (sum of the split-K partials) + beta * C + R, in the product's tile x tile tiles (and
// the sums of squares of C when a.sq_part is set: at most 1024 slots).
void splitk_reduce(const float* part, int splits, int tile, const GemmArgs& a, hipStream_t s) {
    const int64_t total = a.M * a.N, es = static_cast<int64_t>(dtype_size(a.c));
    const bool vec = a.N % 4 == 0 && a.ldc % 4 == 0 && reinterpret_cast<uintptr_t>(a.C) % (4 * es) == 0 &&
                     (!a.R || (a.ldr % 4 == 0 && reinterpret_cast<uintptr_t>(a.R) % (4 * es) == 0)) &&
                     reinterpret_cast<uintptr_t>(part) % 16 == 0;
    const bool few = total <= kFewResults, f32 = a.c == DType::Float32;
    const int64_t tm = (a.M + tile - 1) / tile, tn = (a.N + tile - 1) / tile;
    const int64_t gx = few ? (total + 255) / 256 : tm * tn, stripes = int64_t{tile} * tile / (vec ? 1024 : 256);
    const int64_t gy = few ? 1 : std::max<int64_t>(1, std::min<int64_t>(stripes, (a.sq_part ? 1024 : 4096) / gx));
    AIC_CHECK(gx * gy < (int64_t{1} << 31), InvalidArgument, "split-K reduction: too many tiles");
    AIC_CHECK(!f32 || !a.sq_part || (a.sq_nf && gx * gy <= a.sq_cap), InvalidArgument, "GEMM sums of squares: ", gx * gy,
              " slots needed, ", a.sq_cap, " given");
    const dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(gy));
    const int M = static_cast<int>(a.M), N = static_cast<int>(a.N);
    auto launch = [&](auto tag) {
        using CT = decltype(tag);
        CT* C = static_cast<CT*>(a.C);
        const CT* R = static_cast<const CT*>(a.R);
        double* sq = f32 ? a.sq_part : nullptr;
        int* nf = f32 ? a.sq_nf : nullptr;
        if (few) {
            hipLaunchKernelGGL(splitk_reduce_few_k<CT>, grid, dim3(256), 0, s, part, splits, M, N, a.alpha, a.beta, C, a.ldc,
                               R, a.ldr, sq, nf);
            return;
        }
        void (*kernel)(const float*, int, int64_t, int, int, int, int, int, float, float, CT*, int64_t, const CT*, int64_t,
                       double*, int*) = vec ? splitk_reduce_k<CT, 4> : splitk_reduce_k<CT, 1>;
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, part, splits, total, M, N, tile, static_cast<int>(tm),
                           static_cast<int>(tn), a.alpha, a.beta, C, a.ldc, R, a.ldr, sq, nf);
    };
    if (f32) launch(float{});
    else launch(bf16{});
    AIC_LAUNCH_CHECK("splitk_reduce_k");
}

// K parts of a product on 128x128 tiles of which one block fits a CU: few tiles over a long K fill
// the chip with parts of it (the partials summed in a fixed order afterwards), at most one round of
// blocks.  The part count with the least of: the chain along K, 6 ns a step of one column (measured
// from K 768 to 8192), and, with parts, the reduction's launch and fill (4 us, 2.8 for few results)
// and its traffic (0.35 us per MB of partials).  2304x768 over K 1024 in one part 12.1 us (two parts,
// which any product of fewer than 128 tiles was cut into, 18.4); 65x8 over 1024 in two 9.9 (one 10.4);
// 768x768 over K 8192 in four parts 22.6 (eight, more than a round, 30.8; one 53.7); 1000x768 over
// K 3072 in four 16.4 (one 23.0).
double dma_us(const GemmArgs& a, int parts) {
    const int64_t total = a.M * a.N;
    return 6e-3 * a.K / parts + (parts > 1 ? (total <= kFewResults ? 2.8 : 4.0) + 1.4e-6 * parts * total : 0.0);
}
int dma_splits(int64_t t128, const GemmArgs& a) {
    int best = 1;
    for (int n = 2; n <= std::min<int64_t>({a.K / 512, 256 / t128, 16}); ++n)
        if (a.K / 64 % n == 0 && dma_us(a, n) < dma_us(a, best)) best = n;
    return best;
}

// The sums of squares of the product already in C, for the paths without them in an epilogue.
void sq_matrix(const GemmArgs& a, hipStream_t s) {
    const unsigned grid = static_cast<unsigned>(std::min<int64_t>({(a.M * a.N + 1023) / 1024, 256, a.sq_cap}));
    AIC_CHECK(a.sq_nf && grid >= 1, InvalidArgument, "GEMM sums of squares: no slots given");
    hipLaunchKernelGGL(sq_matrix_k, dim3(grid), dim3(256), 0, s, static_cast<const float*>(a.C), a.ldc,
                       static_cast<int>(a.M), static_cast<int>(a.N), a.sq_part, a.sq_nf);
    AIC_LAUNCH_CHECK("sq_matrix_k");
}

// Whether the rank term alpha X2 Y2^T fits the k-loop tail of the DMA kernels with BN-wide tiles.
bool rank_tail_ok(const GemmArgs& a, int64_t bn) {
    return a.r2 % 8 == 0 && a.ldx2 % 8 == 0 && aligned16(a.X2) && (a.y2_kmajor || (a.ldy2 % 8 == 0 && aligned16(a.Y2))) &&
           (a.seg_n == 0 || a.seg_n % bn == 0);
}

// C = alpha X2 Y2^T + C, per segment, as ordinary GEMMs (the shapes the kernel tail cannot take).
void rank_term_separately(const GemmArgs& a, hipStream_t s) {
    const size_t es = dtype_size(a.ab), ec = dtype_size(a.c);
    const int64_t nseg = a.seg_n > 0 ? a.N / a.seg_n : 1, nn = a.seg_n > 0 ? a.seg_n : a.N;
    for (int64_t g = 0; g < nseg; ++g) {
        GemmArgs t;
        t.transA = 0;
        t.transB = a.y2_kmajor ? 0 : 1;
        t.M = a.M;
        t.N = nn;
        t.K = a.r2;
        t.alpha = a.alpha;
        t.beta = 1.0f;
        t.A = static_cast<const char*>(a.X2) + es * g * a.r2;
        t.lda = a.ldx2;
        t.B = a.y2_kmajor ? static_cast<const char*>(a.Y2) + es * g * nn
                          : static_cast<const char*>(a.Y2) + es * g * nn * a.ldy2;
        t.ldb = a.ldy2;
        t.C = static_cast<char*>(a.C) + ec * g * nn;
        t.ldc = a.ldc;
        t.ab = a.ab;
        t.c = a.c;
        gemm(t, s);
    }
}

}  // namespace

namespace {
// The product with an INT4 B operand; tile size as for the bf16 operands (two stages on both), and
// as there K split where few 128x128 tiles have a long one (5632 -> 2048 on 200 tokens, 32 tiles
// over K 5632: 62 -> 20 us; 11264 -> 2048 on 64 114 -> 18).
void gemm_q4(const GemmArgs& a, hipStream_t s) {
    AIC_CHECK(gemm_q4_eligible(a), InvalidArgument,
              "INT4 GEMM: unsupported shape or layout (bf16 A, K % 64, group % 64, ldb % 64, N % 64 for dy W)");
    const int64_t t256 = ((a.M + 255) / 256) * ((a.N + 255) / 256);
    const bool big = t256 >= 128;
    if (a.r2 > 0) {
        const int64_t bn = big ? 256 : 128;
        if (!rank_tail_ok(a, bn)) {
            GemmArgs b = a;
            b.r2 = 0;
            gemm_q4(b, s);
            rank_term_separately(a, s);
            return;
        }
    }
    const int64_t t128 = ((a.M + 127) / 128) * ((a.N + 127) / 128);
    int splits = 1;
    if (!big && t128 < 128 && a.K >= 1024) {
        splits = static_cast<int>(std::min<int64_t>({a.K / 512, (256 + t128 - 1) / t128, 16}));
        while (splits > 1 && a.K / 64 % splits) --splits;
    } else if (!big && t128 <= 256 && a.K >= 4096 && a.K % 128 == 0) {
        splits = 2;  // two of these blocks fit a CU
    }
    if (splits > 1 && stream_scratch_ready(s)) {
        const StreamScratchUse use(s);
        float* part = static_cast<float*>(stream_scratch(partial_bytes(a, splits), s, 7));
        a.transB ? gemm_impl::launch_dma_q4<128, 128, 64, 2, true, float>(a, s, splits, part)
                 : gemm_impl::launch_dma_q4<128, 128, 64, 2, false, float>(a, s, splits, part);
        splitk_reduce(part, splits, 128, a, s);
        return;
    }
    if (a.c == DType::Float32) {
        if (big) a.transB ? gemm_impl::launch_dma_q4<256, 256, 64, 2, true, float>(a, s)
                          : gemm_impl::launch_dma_q4<256, 256, 64, 2, false, float>(a, s);
        else a.transB ? gemm_impl::launch_dma_q4<128, 128, 64, 2, true, float>(a, s)
                      : gemm_impl::launch_dma_q4<128, 128, 64, 2, false, float>(a, s);
    } else {
        if (big) a.transB ? gemm_impl::launch_dma_q4<256, 256, 64, 2, true, bf16>(a, s)
                          : gemm_impl::launch_dma_q4<256, 256, 64, 2, false, bf16>(a, s);
        else a.transB ? gemm_impl::launch_dma_q4<128, 128, 64, 2, true, bf16>(a, s)
                      : gemm_impl::launch_dma_q4<128, 128, 64, 2, false, bf16>(a, s);
    }
}

// Rows that the fused RoPE / SwiGLU epilogues take: whole 256-row tiles, or any where the product
// runs the persistent kernel (launch_dma, which checks), whose ragged form ends inside a tile: RoPE and
// SwiGLU on x W^T, SwiGLU's backward on dy W.
bool rows_fuse(const GemmArgs& a) {
    return a.M % 256 == 0 || (!a.Bq && a.r2 == 0 && !a.transA && (a.transB != 0) == !a.dglu_gu && a.K % 128 == 0 &&
                              a.K >= 256);
}

void run_f32(const GemmArgs& a, hipStream_t s) {
    const int parts = gemm_f32_parts(a);
    if (parts == 1 || !stream_scratch_ready(s)) {
        gemm_f32(a, s);
        return;
    }
    const StreamScratchUse use(s);
    float* partial = static_cast<float*>(stream_scratch(partial_bytes(a, parts), s, 7));
    gemm_f32(a, s, parts, partial);
    splitk_reduce(partial, parts, 64, a, s);
}

// Few rows of x W^T: the kernel of gemm_skinny.hip (its low-rank term separately where the kernel
// cannot take it).  False: not its shape.
bool try_skinny(const GemmArgs& a, hipStream_t s) {
    // From 17 rows on the tiles' padding shrinks and the skinny kernel's blocks read x again and
    // again: a dense bf16 product stays on it only up to 4 M weights (64 rows: 2048x2048 11.5 us
    // against 14.2 on split tiles, 768x2048 11.4 against 14.7, 6144x2048 20.4 against 18.4, 32 rows:
    // 2048x5632 16.7 against 12.5, 11264x2048 18.7 against 15.8).
    // INT4 alike: 64 rows, 5632->2048 23 us against 14 on split tiles.
    if (a.M > 16 && a.ab == DType::BFloat16 && a.N * a.K > (int64_t{1} << 22) && (!a.Bq || gemm_q4_eligible(a)))
        return false;
    if (a.r2 == 0 && !a.Bq && gemm_dma_eligible(a)) {
        // A block's eight waves walk all of K, 1 ns a column and 0.045 more for each row, so a long K is
        // better cut among tile blocks, by more than the tiles' own fill and an epilogue's pass (64
        // rows: 16 columns over K 5632 25 us here, 11 there; 16 over 32768 147 and 21; eight rows: 2048 over
        // 5632 9.9 and 11.7, 256 over 8192 13.2 and 13.1, 64 over 16384 24.4 and 15.6).
        const bool fused = a.rope_cos || a.glu_f > 0;
        const double us = a.K * (1e-3 + 4.5e-5 * a.M) - (fused ? 6.5 : 2.5);
        if (us > 2.8 && stream_scratch_ready(s) && us > dma_us(a, dma_splits((a.N + 127) / 128, a))) return false;
        // Past 2^25 weights the tile copies read W faster (32000x2048: eight rows 27.1 us here and 20.9
        // there, 16 rows 27.7 and 21.1); not where their epilogue would round the bf16 product before it
        // adds R or C, and for fewer rows not by enough to keep other streams off the CUs (four
        // rows 26.9 and 20.9, a decoding step 283 and 279 us, with three models at a time 308 and 310).
        const bool adds = a.c == DType::BFloat16 && (a.R || a.beta != 0.0f);
        if (!fused && !adds && a.M >= 8 && a.N * a.K > (int64_t{1} << 25)) return false;
    }
    SkinnyArgs q;
    q.g = a;
    if (gemm_skinny_eligible(q)) {
        gemm_skinny(q, s);
        return true;
    }
    if (a.r2 == 0 || a.rope_cos || a.glu_f > 0) return false;
    q.g.r2 = 0;
    if (!gemm_skinny_eligible(q)) return false;
    gemm_skinny(q, s);
    rank_term_separately(a, s);
    return true;
}
}  // namespace

void gemm(const GemmArgs& a, hipStream_t s) {
    AIC_CHECK(a.M >= 0 && a.N >= 0 && a.K >= 0, InvalidArgument, "negative GEMM size");
    AIC_CHECK(a.M < (1LL << 31) && a.N < (1LL << 31) && a.K < (1LL << 31), InvalidArgument, "GEMM size too large");
    AIC_CHECK(a.A && (a.B || a.Bq) && a.C, InvalidArgument, "null GEMM operand");
    AIC_CHECK(a.ab == DType::Float32 || a.ab == DType::BFloat16, DTypeMismatch, "GEMM inputs must be f32 or bf16");
    AIC_CHECK(a.c == DType::Float32 || a.c == DType::BFloat16, DTypeMismatch, "GEMM output must be f32 or bf16");
    const int64_t amin = a.transA ? a.M : a.K, bmin = a.transB ? a.K : a.N;
    AIC_CHECK(a.lda >= (amin > 0 ? amin : 1) && a.ldb >= (bmin > 0 ? bmin : 1) && a.ldc >= (a.N > 0 ? a.N : 1),
              InvalidArgument, "leading dimension smaller than the row length");
    if (a.r2 > 0) {
        AIC_CHECK(a.X2 && a.Y2, InvalidArgument, "low-rank GEMM term without X2 / Y2");
        AIC_CHECK(a.seg_n >= 0 && (a.seg_n == 0 || a.N % a.seg_n == 0), InvalidArgument,
                  "low-rank segments must tile N");
        const int64_t segs = a.seg_n > 0 ? a.N / a.seg_n : 1;
        AIC_CHECK(a.ldx2 >= segs * a.r2 && a.ldy2 >= (a.y2_kmajor ? a.N : a.r2), InvalidArgument,
                  "low-rank term: leading dimension smaller than the row length");
    }
    if (a.M == 0 || a.N == 0) return;
    if (a.sq_part) {
        AIC_CHECK(a.c == DType::Float32 && a.sq_nf && a.sq_cap > 0 && !a.rope_cos && a.glu_f == 0 && !a.dglu_gu,
                  InvalidArgument, "GEMM sums of squares: fp32 output only, without the RoPE / SwiGLU epilogues");
        // in the epilogue of the DMA tile kernels and of gemm_f32, or in the reduction of K parts; the
        // other paths (INT4 B, a low-rank term, the non-DMA kernels) read the product back
        if (gemm_f32_has_sq(a)) {
            run_f32(a, s);
            return;
        }
        if (a.Bq || a.r2 > 0 || !gemm_dma_eligible(a)) {
            GemmArgs b = a;
            b.sq_part = nullptr;
            b.sq_nf = nullptr;
            b.sq_cap = 0;
            gemm(b, s);
            sq_matrix(a, s);
            return;
        }
    }
    if (a.rope_cos) {
        AIC_CHECK(a.rope_sin && a.rope_hd > 0 && a.rope_hd % 2 == 0 && a.rope_cols % a.rope_hd == 0 &&
                      a.rope_cols <= a.N && a.rope_seq > 0 && a.M % a.rope_seq == 0 && a.beta == 0.0f && !a.R,
                  InvalidArgument, "GEMM rotary epilogue: bad rope arguments");
        if (try_skinny(a, s)) return;
        // in the epilogue: bf16 output on full 256x256 tiles, for the eight-wave plain path heads of
        // 128 (split in halves by the 64-column wave sub-tiles, exchanged through LDS) or 64 (one
        // per wave sub-tile), for the four-wave INT4 path heads of 128 (one per wave sub-tile,
        // after the kernel's low-rank term)
        const bool tiles = a.c == DType::BFloat16 && rows_fuse(a) && a.N % 256 == 0 && a.rope_cols % 256 == 0 &&
                           a.ldc % 8 == 0 && aligned16(a.C) && (((a.M + 255) / 256) * (a.N / 256) >= 128);
        const bool fused = tiles && (a.Bq ? a.rope_hd == 128 && a.transB && gemm_q4_eligible(a) &&
                                                (a.r2 == 0 || rank_tail_ok(a, 256))
                                          : (a.rope_hd == 128 || a.rope_hd == 64) && gemm_impl::kDmaWaves256 == 8 &&
                                                gemm_dma_eligible(a) && a.r2 == 0);
        if (!fused) {
            const StreamScratchUse use(s);  // w, until the product is launched
            GemmArgs b = a;
            b.rope_cos = b.rope_sin = nullptr;
            if (a.Bq && !gemm_q4_eligible(a)) {
                // an INT4 weight the operand-load dequantization cannot take (group or row length
                // not a multiple of 64, misaligned scales): dequantized into a scratch copy first
                const int64_t nw = a.N * a.K;
                AIC_CHECK(a.transB && a.ldb == a.K && a.Bscale, InvalidArgument,
                          "INT4 GEMM: the weight must be [N][K] with ld K");
                void* w = stream_scratch(dtype_size(a.ab) * static_cast<size_t>(nw), s, 5);
                int4_dequant(a.Bq, a.Bscale, a.scale_t, nw, a.group, w, a.ab, s);
                b.B = w;
                b.Bq = nullptr;
                b.Bscale = nullptr;
            }
            gemm(b, s);
            rope(a.C, a.ldc, a.M / a.rope_seq, a.rope_seq, a.rope_cols / a.rope_hd, a.rope_hd, a.rope_start,
                 a.rope_cos, a.rope_sin, false, a.c, s);
            return;
        }
    }
    if (a.glu_f > 0) {
        AIC_CHECK(a.N == 2 * a.glu_f && a.glu_out && a.ld_glu >= a.glu_f && a.beta == 0.0f && !a.R && !a.rope_cos,
                  InvalidArgument, "GEMM SwiGLU epilogue: bad arguments");
        if (try_skinny(a, s)) return;
        // in the epilogue: bf16 x W^T on full 256x256 tiles of the eight-wave plain path, or of the
        // four-wave INT4 path (also after its low-rank term, whose segments follow the pairing)
        const bool tiles = a.transB && !a.transA && a.c == DType::BFloat16 && rows_fuse(a) && a.glu_f % 128 == 0 &&
                           a.ldc % 8 == 0 && aligned16(a.C) && a.ld_glu % 8 == 0 && aligned16(a.glu_out) &&
                           (((a.M + 255) / 256) * (a.N / 256) >= 128);
        const bool fused = tiles && (a.Bq ? gemm_q4_eligible(a) && (a.r2 == 0 || rank_tail_ok(a, 256))
                                          : gemm_impl::kDmaWaves256 == 8 && gemm_dma_eligible(a) && a.r2 == 0);
        if (!fused) {
            GemmArgs b = a;
            b.glu_f = 0;
            b.glu_out = nullptr;
            gemm(b, s);
            swiglu_fwd(a.C, static_cast<const char*>(a.C) + dtype_size(a.c) * a.glu_f, a.ldc, a.glu_out, a.ld_glu,
                       a.M, a.glu_f, a.c, s);
            return;
        }
        if (a.Bq) gemm_q4(a, s);
        else dispatch_dma<256, 256, 64, 2, bf16>(a, s);
        return;
    }
    if (a.dglu_gu) {
        AIC_CHECK(a.dglu_out && a.dglu_ld >= 2 * a.N && a.beta == 0.0f && !a.R && !a.rope_cos && a.glu_f == 0,
                  InvalidArgument, "GEMM SwiGLU-backward epilogue: bad arguments");
        // in the epilogue of the full-tile paths without K split (at least 128 tiles of 256x256)
        const int64_t es = static_cast<int64_t>(dtype_size(a.c));
        const bool fused = a.c == DType::BFloat16 && (a.Bq ? gemm_q4_eligible(a) : gemm_dma_eligible(a)) &&
                           rows_fuse(a) && (a.M % 256 == 0 || !a.dglu_whole) && a.N % 256 == 0 &&
                           ((a.M + 255) / 256) * (a.N / 256) >= 128 && a.ldc % 8 == 0 && aligned16(a.C) &&
                           a.dglu_ld % 8 == 0 && aligned16(a.dglu_gu) && aligned16(a.dglu_out) &&
                           (a.r2 == 0 || rank_tail_ok(a, 256));  // C is not written: no rank term added later
        if (!fused) {
            GemmArgs b = a;
            b.dglu_gu = nullptr;
            b.dglu_out = nullptr;
            gemm(b, s);
            swiglu_bwd(a.dglu_gu, static_cast<const char*>(a.dglu_gu) + es * a.N, a.dglu_ld, a.C, a.ldc, a.dglu_out,
                       static_cast<char*>(a.dglu_out) + es * a.N, a.dglu_ld, a.M, a.N, a.c, s);
            return;
        }
    }
    if (try_skinny(a, s)) return;
    if (a.Bq) {
        gemm_q4(a, s);
        return;
    }
    if (gemm_dma_eligible(a)) {
        // 256x256 tiles from half a round of tiles up (measured on the 1B shapes: 176 tiles of
        // 256x256 beat 704 of 128x128 by 24%); between 32 and 128 of them over a long K, 256x256
        // tiles with K split so that about one full round runs (the 2048x2048x8192 weight
        // gradient: 80 us against 93 us on 128x128 tiles)
        const int64_t t256 = ((a.M + 255) / 256) * ((a.N + 255) / 256);
        const int64_t t128 = ((a.M + 127) / 128) * ((a.N + 127) / 128);
        const int64_t tw = ((a.M + 127) / 128) * ((a.N + 255) / 256);  // 128x256 tiles
        const bool big = t256 >= 128;
        // under a round of 256x256 tiles over a long K (a 1024-wide head's input gradient: 128
        // tiles, K 32000): split K until about one round runs (682 -> 444 us there)
        int splits256 = 1;
        const bool plain = a.r2 == 0 && !a.rope_cos && !a.dglu_gu;  // forms that the K splits' reduction has
        if (plain && t256 < 256 && t256 >= 32 && a.K >= 4096) {
            splits256 = static_cast<int>(std::min<int64_t>(4, 256 / t256));
            while (splits256 > 1 && a.K / 64 % splits256) --splits256;
        }
        if (a.r2 > 0) {
            const int64_t bn = big ? 256 : 128;
            if (!rank_tail_ok(a, bn)) {
                GemmArgs b = a;
                b.r2 = 0;
                gemm(b, s);
                rank_term_separately(a, s);
                return;
            }
        }
        if (splits256 > 1 && stream_scratch_ready(s)) {
            const StreamScratchUse use(s);
            float* part = static_cast<float*>(stream_scratch(partial_bytes(a, splits256), s, 7));
            dispatch_dma<256, 256, 64, 2, float>(a, s, splits256, part);
            splitk_reduce(part, splits256, 256, a, s);
            return;
        }
        const int splits = plain && !big ? dma_splits(t128, a) : 1;
        if (splits > 1 && stream_scratch_ready(s)) {
            const StreamScratchUse use(s);
            float* part = static_cast<float*>(stream_scratch(partial_bytes(a, splits), s, 7));
            dispatch_dma<128, 128, 64, 4, float>(a, s, splits, part);
            splitk_reduce(part, splits, 128, a, s);
            return;
        }
        // under a round of 256x256 tiles where 128x256 tiles fill between half the chip and one
        // round (768- and 1024-wide products over 8192 rows): one round of the four-wave 128x256
        // kernel beats a partial round of 256x256 tiles and two rounds of 128x128 ones (measured
        // 3-9% on those shapes); with a residual and at least half a round of 256x256 tiles the
        // persistent kernel stays ahead (its epilogue overlaps the next tile's copies)
        if (plain && t256 < 256 && tw >= 128 && tw <= 256 && !(a.R && big)) {
            if (a.c == DType::Float32) dispatch_dma<128, 256, 64, 3, float>(a, s);
            else dispatch_dma<128, 256, 64, 3, bf16>(a, s);
            return;
        }
        if (a.c == DType::Float32) {
            if (big) dispatch_dma<256, 256, 64, 2, float>(a, s);
            else dispatch_dma<128, 128, 64, 4, float>(a, s);
        } else {
            if (big) dispatch_dma<256, 256, 64, 2, bf16>(a, s);
            else dispatch_dma<128, 128, 64, 4, bf16>(a, s);
        }
        return;
    }
    if (a.r2 > 0) {
        GemmArgs b = a;
        b.r2 = 0;
        gemm(b, s);
        rank_term_separately(a, s);
        return;
    }
    if (gemm_mfma_eligible(a)) {
        const bool big = a.M >= 2048 && a.N >= 2048 && ((a.M / 256) * (a.N / 256) >= 256);
        if (a.c == DType::Float32) {
            if (big) dispatch_trans<256, 256, float>(a, s);
            else dispatch_trans<128, 128, float>(a, s);
        } else {
            if (big) dispatch_trans<256, 256, bf16>(a, s);
            else dispatch_trans<128, 128, bf16>(a, s);
        }
        return;
    }
    if (gemm_f32_eligible(a)) {
        run_f32(a, s);
        return;
    }
    if (a.ab == DType::Float32) {
        launch_simt<float, bf16>(a, s);
    } else {
        if (a.c == DType::Float32) launch_simt<bf16, float>(a, s);
        else launch_simt<bf16, bf16>(a, s);
    }
}

void gemm_grouped(const GemmArgs* a, int n, hipStream_t s) {
    AIC_CHECK(a && n >= 0, InvalidArgument, "gemm_grouped: bad arguments");
    bool one_launch = n >= 2 && n <= gemm_impl::kMaxGroups;
    int64_t t256 = 0;
    for (int i = 0; i < n && one_launch; ++i) {
        const GemmArgs& x = a[i];
        one_launch = gemm_dma_eligible(x) && x.transA == a[0].transA && x.transB == a[0].transB &&
                     x.ab == a[0].ab && x.c == a[0].c && !x.R && x.r2 == 0 && x.alpha == a[0].alpha &&
                     x.beta == a[0].beta && x.M > 0 && x.N > 0 && x.ldc >= x.N &&
                     x.lda >= (x.transA ? x.M : x.K) && x.ldb >= (x.transB ? x.K : x.N);
        t256 += ((x.M + 255) / 256) * ((x.N + 255) / 256);
    }
    if (!one_launch) {
        for (int i = 0; i < n; ++i) {
            GemmArgs b = a[i];
            if (a[0].sq_part) {  // the launch's slot region in equal shares
                const int64_t share = a[0].sq_cap / n;
                b.sq_part = a[0].sq_part + i * share;
                b.sq_nf = a[0].sq_nf + i * share;
                b.sq_cap = share;
            } else {
                b.sq_part = nullptr;
            }
            gemm(b, s);
        }
        return;
    }
    if (t256 > 256 && t256 % 256 != 0 && t256 % 256 <= 64) {
        // A few tiles past whole rounds of the chip (the 1B layer's four weight gradients: 784
        // tiles of 256x256, 3 rounds + 16) would cost most of a fourth round.  One product gives
        // up whole tile-columns (or tile-rows) making up the excess; they run after the launch
        // as their own GEMM, which splits them along K over the chip (834 -> 745 us at that
        // shape).  Taken only when the remaining tiles fall evenly on the 8 XCDs (block b runs
        // on XCD b % 8; each product's blocks start at a multiple of 8).
        const int64_t excess = t256 % 256, rounds = t256 / 256;
        for (int i = n - 1; i >= 0; --i) {
            const GemmArgs& x = a[i];
            const int64_t tm = (x.M + 255) / 256, tn = (x.N + 255) / 256;
            GemmArgs keep = x, cut = x;
            const size_t es = dtype_size(x.ab), ec = dtype_size(x.c);
            if (excess % tm == 0 && excess / tm < tn) {  // the rightmost tile-columns
                const int64_t n0 = 256 * (tn - excess / tm);
                keep.N = n0;
                cut.N = x.N - n0;
                cut.B = static_cast<const char*>(x.B) + es * (x.transB ? n0 * x.ldb : n0);
                cut.C = static_cast<char*>(x.C) + ec * n0;
            } else if (excess % tn == 0 && excess / tn < tm) {  // the bottom tile-rows
                const int64_t m0 = 256 * (tm - excess / tn);
                keep.M = m0;
                cut.M = x.M - m0;
                cut.A = static_cast<const char*>(x.A) + es * (x.transA ? m0 : m0 * x.lda);
                cut.C = static_cast<char*>(x.C) + ec * m0 * x.ldc;
            } else {
                continue;
            }
            std::vector<GemmArgs> g(a, a + n);
            g[i] = keep;
            int64_t per_xcd[8] = {};
            for (const GemmArgs& y : g) {
                const int64_t t = ((y.M + 255) / 256) * ((y.N + 255) / 256);
                for (int xcd = 0; xcd < 8; ++xcd) per_xcd[xcd] += t / 8 + (xcd < t % 8 ? 1 : 0);
            }
            if (*std::max_element(per_xcd, per_xcd + 8) > 32 * rounds) continue;
            if (g[0].c == DType::Float32) dispatch_grouped<256, 256, 64, 2, float>(g.data(), n, s);
            else dispatch_grouped<256, 256, 64, 2, bf16>(g.data(), n, s);
            cut.sq_part = nullptr;
            if (a[0].sq_part) {  // the launch's blocks (8-aligned per product), then the cut's slots
                int64_t blocks = 0;
                for (const GemmArgs& y : g) blocks += (((y.M + 255) / 256) * ((y.N + 255) / 256) + 7) / 8 * 8;
                AIC_CHECK(blocks < a[0].sq_cap, InvalidArgument, "grouped GEMM sums of squares: region too small");
                cut.sq_part = a[0].sq_part + blocks;
                cut.sq_nf = a[0].sq_nf + blocks;
                cut.sq_cap = a[0].sq_cap - blocks;
            }
            gemm(cut, s);
            return;
        }
    }
    // under half a round of 256x256 tiles: 128x128 tiles, or 128x256 ones where those fill one
    // round and 128x128 tiles would need more (the 125M layer's four weight gradients: 216 tiles
    // of 128x256 against 432 of 128x128)
    int64_t t128 = 0, tw = 0;
    for (int i = 0; i < n; ++i) {
        t128 += ((a[i].M + 127) / 128) * ((a[i].N + 127) / 128);
        tw += ((a[i].M + 127) / 128) * ((a[i].N + 255) / 256);
    }
    const bool wide = t256 < 128 && t128 > 256 && tw <= 256;
    if (a[0].c == DType::Float32) {
        if (t256 >= 128) dispatch_grouped<256, 256, 64, 2, float>(a, n, s);
        else if (wide) dispatch_grouped<128, 256, 64, 3, float>(a, n, s);
        else dispatch_grouped<128, 128, 64, 4, float>(a, n, s);
    } else {
        if (t256 >= 128) dispatch_grouped<256, 256, 64, 2, bf16>(a, n, s);
        else if (wide) dispatch_grouped<128, 256, 64, 3, bf16>(a, n, s);
        else dispatch_grouped<128, 128, 64, 4, bf16>(a, n, s);
    }
}

// One product: the tile kernels write one slot per block (at most its 128x128 tile count,
// rounded up to a multiple of 8 for the grouped launch's per-product padding), the split-K
// reduction at most 1024 and the read-back pass at most 256.  Several products: the grouped
// launch's blocks, or the blocks of all but a cut product plus the cut's own launch, or equal
// shares of the region per product (one gemm() each) -- all within n + 1 times the largest
// single bound.
int64_t gemm_sq_slots(const GemmArgs* a, int n) {
    AIC_CHECK(a && n >= 1, InvalidArgument, "gemm_sq_slots: no products");
    int64_t most = 0;
    for (int i = 0; i < n; ++i) {
        const int64_t t128 = ((a[i].M + 127) / 128) * ((a[i].N + 127) / 128);
        most = std::max(most, (std::max<int64_t>(t128, 1024) + 7) / 8 * 8);
    }
    return n == 1 ? most : (n + 1) * most;
}

// The ragged-K launch writes one slot per block: E experts of its tile count rounded up to a
// multiple of 8 (256x256 or 128x128 tiles); the fallback (one product per expert, in grouped
// launches of up to 8 sharing the region equally) needs its launches' bounds.
int64_t gemm_ragged_sq_slots(int64_t M, int64_t N, int E) {
    AIC_CHECK(M > 0 && N > 0 && E >= 1, InvalidArgument, "gemm_ragged_sq_slots: bad shape");
    const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
    GemmArgs g;
    g.M = M;
    g.N = N;
    std::vector<GemmArgs> eight(8, g);
    const int64_t launches = (E + 7) / 8;
    return std::max(E * ((t128 + 7) / 8 * 8), launches * gemm_sq_slots(eight.data(), std::min(E, 8)));
}

bool gemm_ragged_eligible(const RaggedArgs& r) {
    const GemmArgs& a = r.g;
    if (!r.offsets || r.E < 1 || r.E > 64 || a.R || a.r2 || a.ab != DType::BFloat16) return false;
    if (a.M < 8 || a.N < 8 || a.lda % 8 || a.ldb % 8 || !aligned16(a.A) || !aligned16(a.B)) return false;
    if (a.M > (int64_t{1} << 30) || a.N > (int64_t{1} << 30)) return false;
    if (r.ragged_k) {
        // A [rows][M], B [rows][N]: row offsets move both by whole rows
        return a.transA && !a.transB && a.M % 8 == 0 && a.N % 8 == 0 && a.lda >= a.M && a.ldb >= a.N &&
               a.ldc >= a.N && r.b_stride == 0 && r.c_stride >= a.M * a.ldc;
    }
    return !a.transA && a.K > 0 && a.K % 64 == 0 && a.lda >= a.K && a.ldc >= a.N && (a.transB || a.N % 8 == 0) &&
           a.ldb >= (a.transB ? a.K : a.N) && r.b_stride % 8 == 0;
}

void gemm_ragged(const RaggedArgs& r, hipStream_t s) {
    AIC_CHECK(gemm_ragged_eligible(r), InvalidArgument, "gemm_ragged: unsupported shape, layout or dtype");
    const GemmArgs& a = r.g;
    bool force256 = false;
    if (a.glu_f > 0 || a.dglu_gu) {
        // SwiGLU (forward or backward) of an expert-ragged product: in the epilogue on bf16 outputs
        // whose columns are whole 256-wide tiles (the forward on 256x256 tiles, whose columns pair
        // 128 gate with 128 up columns); otherwise the product, then the pass over all rows
        AIC_CHECK(!r.ragged_k && a.beta == 0.0f && !a.R && !(a.glu_f > 0 && a.dglu_gu), InvalidArgument,
                  "gemm_ragged: SwiGLU epilogue arguments");
        const bool cols = a.c == DType::BFloat16 && a.N % 256 == 0 && a.ldc % 8 == 0 && aligned16(a.C);
        const bool glu = a.glu_f > 0 && cols && a.transB && !a.transA && gemm_impl::kDmaWaves256 == 8 &&
                         a.N == 2 * a.glu_f && a.glu_f % 128 == 0 && a.ld_glu >= a.glu_f && a.ld_glu % 8 == 0 &&
                         aligned16(a.glu_out);
        const bool dglu = a.dglu_gu && cols && a.dglu_ld >= 2 * a.N && a.dglu_ld % 8 == 0 && aligned16(a.dglu_gu) &&
                          aligned16(a.dglu_out);
        if (!glu && !dglu) {
            RaggedArgs b = r;
            b.g.glu_f = 0;
            b.g.glu_out = nullptr;
            b.g.dglu_gu = nullptr;
            b.g.dglu_out = nullptr;
            gemm_ragged(b, s);
            const int64_t es = static_cast<int64_t>(dtype_size(a.c));
            if (a.glu_f > 0)
                swiglu_fwd(a.C, static_cast<const char*>(a.C) + es * a.glu_f, a.ldc, a.glu_out, a.ld_glu, a.M, a.glu_f,
                           a.c, s);
            else
                swiglu_bwd(a.dglu_gu, static_cast<const char*>(a.dglu_gu) + es * a.N, a.dglu_ld, a.C, a.ldc,
                           a.dglu_out, static_cast<char*>(a.dglu_out) + es * a.N, a.dglu_ld, a.M, a.N, a.c, s);
            return;
        }
        force256 = glu;
    }
    // Tile shape: the grid's tiles (a bound for ragged M) in rounds of 256 CUs; the 256x256
    // tile unless its last round leaves so many CUs idle that 128x128 tiles (0.8 of its rate, 2/3
    // where both operands are read transposed: ragged K) fill the rounds better.  Weight gradients of
    // 8 experts with 2048 rows each, 128x128 and 256x256: 1024x2816 156 and 133 us (1408 and 352
    // tiles), 5632x1024 278 and 198; with 1024 rows each 768x2048 52 and 39; 4 experts with 1500
    // rows, 512x1408 (72 tiles of 256x256) 20 and 37.
    auto tiles = [&](int64_t t) {
        const int64_t tn = (a.N + t - 1) / t;
        return r.ragged_k ? r.E * ((a.M + t - 1) / t) * tn : ((a.M + t - 1) / t + r.E) * tn;
    };
    auto fill = [](int64_t n) { return static_cast<double>(n) / (256.0 * static_cast<double>((n + 255) / 256)); };
    // bf16 rows on whole 256-column tiles run the persistent kernel (gemm_kernels.inc,
    // launch_dma_ragged), whose blocks take tile after tile: a round of 256 tiles is enough
    const bool pers = a.c == DType::BFloat16 && !r.ragged_k && r.E <= 63 && a.N % 256 == 0 && a.K % 128 == 0 &&
                      a.K >= 256 && a.beta == 0.0f;
    const bool big = force256 || (pers && tiles(256) >= 256) ||
                     (tiles(256) >= 128 && fill(tiles(256)) >= (r.ragged_k ? 2.0 / 3 : 0.8) * fill(tiles(128)));
    if (a.c == DType::Float32) {
        if (big) dispatch_ragged<256, 256, 64, 2, float>(r, s);
        else dispatch_ragged<128, 128, 64, 4, float>(r, s);
    } else {
        if (big) dispatch_ragged<256, 256, 64, 2, bf16>(r, s);
        else dispatch_ragged<128, 128, 64, 4, bf16>(r, s);
    }
}

}  // namespace aic::hip
