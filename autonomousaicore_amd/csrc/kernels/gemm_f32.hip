// fp32 products (the fp32 reference configuration; cuda_gemm.cuh:11-14, functions.cpp:254-273) on
// v_mfma_f32_16x16x4_f32: C = alpha op(A) op(B) + beta C + R, fp32 operands and sums.
//
// The fp32 matrix pipe takes 512 cycles for the sixteen MFMAs of a 32x32 tile's 16-deep step and
// that step needs 4 KB of operands, so the fragments come straight from global memory (L1 and L2
// hold the panels): no LDS staging and no barrier in the loop.  A wave owns a tile of 32x32 (64x64
// where those alone fill the chip: half the loads per product); where there are few tiles, `split`
// waves of a block share one, taking the 16-deep K steps in turn and adding their parts through LDS
// in wave order (deterministic, one launch).  K runs in the order of each operand's own layout: a
// lane holds four consecutive k of row lane % 16, one 16-byte load where K is contiguous, four
// 4-byte loads (64 bytes across lanes) where the rows are.
//
// Before (64x64 SIMT tiles, no K split) and now: 512x128x352 42 -> 8 us, 128x352 over 512 rows 64 ->
// 7 us, 1000^3 178 -> 30 us, 4096x4096x1024 576 -> 300 us (114 TFLOP/s of the 157 the pipe has); the
// two-layer d 128 training step of 8 x 64 tokens 1.95 -> 0.53 ms.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "gemm.hpp"

namespace aic::hip {

namespace {

struct F32Params {
    const float* A;
    const float* B;
    float* C;
    const float* R;
    int64_t lda, ldb, ldc, ldr;
    int M, N, K;
    float alpha, beta;
    int tiles_m, tiles_n, split;
    int parts, kpart;  // K in `parts` runs of kpart, part z written to C + z * cz
    int64_t cz;
    int vec;  // C and R rows take 16-byte vectors
    double* sq;
    int* sq_nf;
};

constexpr int kWaves = 8;

// Four consecutive k of row `row`; KC: K contiguous.  VEC: 16-byte aligned rows, K % 4 == 0.
template <bool KC, bool VEC, bool GUARD>
__device__ __forceinline__ float4 frag(const float* p, int64_t ld, int row, int k, int K) {
    if constexpr (KC) {
        const float* q = p + row * ld + k;
        if constexpr (VEC) {
            if (GUARD && k >= K) return make_float4(0, 0, 0, 0);
            return *reinterpret_cast<const float4*>(q);
        } else {
            return make_float4(!GUARD || k < K ? q[0] : 0.0f, !GUARD || k + 1 < K ? q[1] : 0.0f,
                               !GUARD || k + 2 < K ? q[2] : 0.0f, !GUARD || k + 3 < K ? q[3] : 0.0f);
        }
    } else {
        const float* q = p + k * ld + row;
        return make_float4(!GUARD || k < K ? q[0] : 0.0f, !GUARD || k + 1 < K ? q[ld] : 0.0f,
                           !GUARD || k + 2 < K ? q[2 * ld] : 0.0f, !GUARD || k + 3 < K ? q[3 * ld] : 0.0f);
    }
}

// NT x NT 16x16 tiles per wave.
template <bool TA, bool TB, bool VEC, int NT>
__global__ __launch_bounds__(64 * kWaves) void gemm_f32_k(const F32Params p) {
    extern __shared__ __attribute__((aligned(16))) char f32_lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    const int part = wave % p.split;
    // block b takes K part b % parts: with 8 parts an XCD (b % 8) reads only its eighth of the panels
    const int kz = static_cast<int>(blockIdx.x) % p.parts;
    const int tile = static_cast<int>(blockIdx.x) / p.parts * (kWaves / p.split) + wave / p.split;
    const int64_t k0 = static_cast<int64_t>(kz) * p.kpart;
    const int K = static_cast<int>(min(static_cast<int64_t>(p.kpart), p.K - k0));
    const float* A = p.A + (TA ? k0 * p.lda : k0);
    const float* B = p.B + (TB ? k0 : k0 * p.ldb);
    const bool live = tile < p.tiles_m * p.tiles_n;
    const int m0 = tile / p.tiles_n * 16 * NT, n0 = tile % p.tiles_n * 16 * NT;
    f32x4 acc[NT][NT] = {};  // [m][n]: rows n = 4 g + i, column m = lane % 16
    if (live) {
        int am[NT], bn[NT];
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            am[i] = min(m0 + 16 * i + c, p.M - 1);
            bn[i] = min(n0 + 16 * i + c, p.N - 1);
        }
        struct Step {
            float4 a[NT], b[NT];
        };
        auto load = [&](int step, Step& f, auto guard) {
            constexpr bool G = decltype(guard)::value;
            const int k = 16 * step + 4 * g;
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                f.a[i] = frag<!TA, VEC, G>(A, p.lda, am[i], k, K);
                f.b[i] = frag<TB, VEC, G>(B, p.ldb, bn[i], k, K);
            }
        };
        auto mma = [&](const Step& f) {
#pragma unroll
            for (int m = 0; m < NT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.b[n].x, f.a[m].x, acc[m][n], 0, 0, 0);
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.b[n].y, f.a[m].y, acc[m][n], 0, 0, 0);
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.b[n].z, f.a[m].z, acc[m][n], 0, 0, 0);
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.b[n].w, f.a[m].w, acc[m][n], 0, 0, 0);
                }
        };
        const int full = K / 16;
        int s = part;
        Step nxt;
        if (s < full) load(s, nxt, std::false_type{});
        for (; s < full; s += p.split) {
            const Step cur = nxt;
            if (s + p.split < full) load(s + p.split, nxt, std::false_type{});
            mma(cur);
        }
        if (16 * full < K && s == full) {  // the wave whose turn it is takes the rest
            Step f;
            load(full, f, std::true_type{});
            mma(f);
        }
    }
    double sqa = 0.0;
    int sqf = 0;
    if (p.split > 1) {
        f32x4* red = reinterpret_cast<f32x4*>(f32_lds);  // [kWaves][NT * NT][64]
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) red[(wave * NT * NT + m * NT + n) * 64 + lane] = acc[m][n];
        __syncthreads();
    }
    if (live) {
        const int w0 = wave - part;
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                f32x4 t = acc[m][n];
                if (p.split > 1) {  // the group's waves finish its 16x16 tiles in turn
                    if ((m * NT + n) % p.split != part) continue;
                    const f32x4* red = reinterpret_cast<const f32x4*>(f32_lds) + (w0 * NT * NT + m * NT + n) * 64 + lane;
                    t = red[0];
                    for (int w = 1; w < p.split; ++w) t += red[w * NT * NT * 64];
                }
                const int row = m0 + 16 * m + c, col = n0 + 16 * n + 4 * g;
                if (row >= p.M || col >= p.N) continue;
                float* C = p.C + kz * p.cz + row * p.ldc + col;
                const float* R = p.R ? p.R + row * p.ldr + col : nullptr;
                float v[4] = {p.alpha * t[0], p.alpha * t[1], p.alpha * t[2], p.alpha * t[3]};
                if (p.vec && col + 4 <= p.N) {
                    if (p.beta != 0.0f) {
                        const float4 o = *reinterpret_cast<const float4*>(C);
                        v[0] += p.beta * o.x; v[1] += p.beta * o.y; v[2] += p.beta * o.z; v[3] += p.beta * o.w;
                    }
                    if (R) {
                        const float4 o = *reinterpret_cast<const float4*>(R);
                        v[0] += o.x; v[1] += o.y; v[2] += o.z; v[3] += o.w;
                    }
                    *reinterpret_cast<float4*>(C) = make_float4(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (col + i >= p.N) {
                            v[i] = 0.0f;
                            continue;
                        }
                        if (p.beta != 0.0f) v[i] += p.beta * C[i];
                        if (R) v[i] += R[i];
                        C[i] = v[i];
                    }
                }
                if (p.sq) {
                    sqa += static_cast<double>(v[0] * v[0] + v[1] * v[1]) + static_cast<double>(v[2] * v[2] + v[3] * v[3]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) sqf |= (__float_as_uint(v[i]) & 0x7f800000u) == 0x7f800000u;
                }
            }
    }
    if (p.sq) {
        // the block's sum of squares: lanes by butterfly, then waves in order
        __shared__ double sd[kWaves];
        __shared__ int sn[kWaves];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            sqa += __shfl_xor(sqa, o);
            sqf |= __shfl_xor(sqf, o);
        }
        if (lane == 0) {
            sd[wave] = sqa;
            sn[wave] = sqf;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double t = 0.0;
            int f = 0;
            for (int w = 0; w < kWaves; ++w) {
                t += sd[w];
                f |= sn[w];
            }
            p.sq[blockIdx.x] = t;
            p.sq_nf[blockIdx.x] = f;
        }
    }
}

template <bool TA, bool TB, bool VEC, int NT>
void launch(const F32Params& p, int blocks, hipStream_t s) {
    const size_t lds = p.split > 1 ? static_cast<size_t>(kWaves) * NT * NT * 1024 : 0;
    static bool configured = false;
    if (!configured) {
        AIC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_f32_k<TA, TB, VEC, NT>),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, kWaves * NT * NT * 1024));
        configured = true;
    }
    hipLaunchKernelGGL((gemm_f32_k<TA, TB, VEC, NT>), dim3(blocks), dim3(64 * kWaves), lds, s, p);
    AIC_LAUNCH_CHECK("gemm_f32");
}

template <bool VEC, int NT>
void by_layout(const GemmArgs& a, const F32Params& p, int blocks, hipStream_t s) {
    if (!a.transA && a.transB) launch<false, true, VEC, NT>(p, blocks, s);
    else if (!a.transA) launch<false, false, VEC, NT>(p, blocks, s);
    else if (!a.transB) launch<true, false, VEC, NT>(p, blocks, s);
    else launch<true, true, VEC, NT>(p, blocks, s);
}

bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

struct Plan {
    int nt, split, blocks;
    int64_t tiles_m, tiles_n;
};

// 64x64 tiles from one per SIMD up (1024); below, 32x32 tiles with their K shared by up to eight
// waves until the chip has about two waves per SIMD, each with at least one 16-deep step (a floor of four
// left half the chip idle on the d 128 training step, 0.62 ms against 0.56).
Plan plan_of(int64_t M, int64_t N, int64_t K) {
    Plan q;
    q.nt = ((M + 63) / 64) * ((N + 63) / 64) >= 1024 ? 4 : 2;
    q.tiles_m = (M + 16 * q.nt - 1) / (16 * q.nt);
    q.tiles_n = (N + 16 * q.nt - 1) / (16 * q.nt);
    q.split = 1;
    while (q.split < kWaves && q.tiles_m * q.tiles_n * q.split < 2048 && K / 16 >= 2 * q.split) q.split *= 2;
    const int per = kWaves / q.split;
    q.blocks = static_cast<int>((q.tiles_m * q.tiles_n + per - 1) / per);
    return q;
}

}  // namespace

bool gemm_f32_eligible(const GemmArgs& a) {
    return a.ab == DType::Float32 && a.c == DType::Float32 && !a.Bq && a.r2 == 0 && !a.rope_cos && a.glu_f == 0 &&
           !a.dglu_gu && a.M > 0 && a.N > 0 && ((a.M + 31) / 32) * ((a.N + 31) / 32) < (int64_t{1} << 31);
}

bool gemm_f32_has_sq(const GemmArgs& a) {
    return gemm_f32_eligible(a) && (gemm_f32_parts(a) > 1 || plan_of(a.M, a.N, a.K).blocks <= a.sq_cap);
}

// Few tiles over a long K (the weight gradients): every XCD's L2 fetches every panel, and that
// traffic bounds the product.  With K in eight parts, one per XCD, and the pass that adds them:
// 320x128 over 8192 rows 56 -> 21 us, 768x256 56 -> 49 us.  Eight parts where the panels read seven times less
// outweigh the partial sums written and read.
int gemm_f32_parts(const GemmArgs& a) {
    const int64_t tiles = ((a.M + 31) / 32) * ((a.N + 31) / 32);
    return a.K >= 2048 && tiles <= 1024 && 16 * a.M * a.N < 7 * (a.M + a.N) * a.K ? 8 : 1;
}

void gemm_f32(const GemmArgs& a, hipStream_t s, int parts, float* partial) {
    AIC_CHECK(gemm_f32_eligible(a) && parts >= 1 && (parts == 1 || partial), InvalidArgument,
              "fp32 GEMM: unsupported arguments");
    const int64_t kpart = parts == 1 ? std::max<int64_t>(a.K, 1) : (a.K / 16 / parts + 1) * 16;
    AIC_CHECK((parts - 1) * kpart < std::max<int64_t>(a.K, 1), InvalidArgument, "fp32 GEMM: too many K parts");
    const Plan q = plan_of(a.M, a.N, kpart);
    F32Params p{};
    p.A = static_cast<const float*>(a.A);
    p.B = static_cast<const float*>(a.B);
    p.C = static_cast<float*>(a.C);
    p.R = static_cast<const float*>(a.R);
    p.lda = a.lda; p.ldb = a.ldb; p.ldc = a.ldc; p.ldr = a.ldr;
    p.M = static_cast<int>(a.M); p.N = static_cast<int>(a.N); p.K = static_cast<int>(a.K);
    p.alpha = a.alpha; p.beta = a.beta;
    p.tiles_m = static_cast<int>(q.tiles_m); p.tiles_n = static_cast<int>(q.tiles_n);
    p.split = q.split;
    p.parts = parts;
    p.kpart = static_cast<int>(kpart);
    if (parts > 1) {
        p.C = partial;
        p.R = nullptr;
        p.ldc = a.N;
        p.cz = a.M * a.N;
        p.alpha = 1.0f;
        p.beta = 0.0f;
    }
    const int blocks = q.blocks * parts;
    p.vec = p.ldc % 4 == 0 && p.cz % 4 == 0 && a16(p.C) && (!p.R || (p.ldr % 4 == 0 && a16(p.R)));
    if (a.sq_part && parts == 1) {
        AIC_CHECK(a.sq_nf && q.blocks <= a.sq_cap, InvalidArgument, "GEMM sums of squares: ", q.blocks, " slots needed, ",
                  a.sq_cap, " given");
        p.sq = a.sq_part;
        p.sq_nf = a.sq_nf;
    }
    // 16-byte loads of the operands that are contiguous along K
    // (a part starts at a multiple of 16)
    const bool vec = (a.transA || (a.K % 4 == 0 && a.lda % 4 == 0 && a16(a.A))) &&
                     (!a.transB || (a.K % 4 == 0 && a.ldb % 4 == 0 && a16(a.B)));
    if (vec) q.nt == 4 ? by_layout<true, 4>(a, p, blocks, s) : by_layout<true, 2>(a, p, blocks, s);
    else q.nt == 4 ? by_layout<false, 4>(a, p, blocks, s) : by_layout<false, 2>(a, p, blocks, s);
}

}  // namespace aic::hip
