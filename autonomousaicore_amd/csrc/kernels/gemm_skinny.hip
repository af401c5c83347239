// Products with few rows: C[M, N] = alpha * (x W^T + X2 Y2^T) + beta * C + R for M <= 64 (token by
// token decoding, short prompts, small batches, LoRA's rank-r products on them), W [N][K] as bf16,
// fp32 or packed INT4.  Replaces the same reference calls as gemm.hip (cuda_gemm.cuh:11-14).
//
// Bound: reading W once.  A block owns 16 rows of W (or two 16-row tiles: the gate row and its up
// row, the two halves of a rotary head, or neighbours) and all rows of x; its eight waves take the
// K steps in turn, so that a block reads whole W rows in contiguous pieces, and add their partial
// tiles through LDS in wave order (deterministic, one launch, no partial sums in HBM).  Operands go
// straight from global memory into the 16x16 MFMA fragment layout: lane % 16 is the row, 16 bytes
// of K per lane.  A 128x128 tile kernel reads the same W with N / 128 blocks and, for one row,
// spends 127 of 128 tile rows on padding.
//
// Done on the way: RMSNorm of x (every block normalises the few rows into LDS: less than the launch
// of a pass of its own), the low-rank term, the residual, SwiGLU, RoPE and the KV cache's new rows.
//
// Measured (bf16, x W^T, one row; the tile kernels before in brackets): 6144x2048 8.8 us (28.9),
// 11264x2048 13.4 (29.1), 2048x5632 9.1 (71.7), 32000x2048 28 us = 4.7 TB/s (42.5).  Sixteen rows:
// 10.6 (13.5), 14.4 (15.4), 11.9 (12.3), 34.3 (34.1).  One token of the 125M model at 512 positions:
// 1.44 ms -> 0.48 ms (148 launches -> 63); of the 1B-wide two-layer QLoRA model, four sequences:
// 1.09 -> 0.32 ms (its INT4 weights are no longer dequantized to a scratch copy below 8 rows).
#include <algorithm>

#include "common.hpp"
#include "gemm.hpp"

namespace aic::hip {

namespace {

enum WKind { kBf16, kF32, kInt4 };

struct SkinnyParams {
    const void* A;
    const void* W;
    const uint16_t* scales;  // INT4: fp16, one per G elements of the flat weight
    void* C;
    const void* R;
    int64_t lda, ldw, ldc, ldr;
    int M, N, K, G;
    int gshift;  // log2(G / 64), or -1
    float alpha, beta;
    const void* X2;
    const void* Y2;
    int64_t ldx2, ldy2;
    int r2, seg_n;
    const float* norm_w;
    float norm_eps;
    // the block's second W tile starts `pair` rows after its first; first tiles are consecutive
    // within runs of `run` rows, one run every `run_step` rows
    int pair, run, run_step;
    const float* rope_cos;
    const float* rope_sin;
    int rope_cols, rope_hd, rope_seq, rope_start;
    void* glu_out;
    int64_t ld_glu;
    void* kc;
    void* vc;
    int64_t kv_rows;
    int vec;      // C, R and glu_out rows take four-element vectors
    int store_c;  // 0: only glu_out is wanted
};

// Elements of x's type, K elements per step (four lanes per row), 16-byte x vectors per step.
template <int W> struct Kind;
template <> struct Kind<kBf16> {
    using T = bf16;
    static constexpr int step = 32, per_lane = 8, xv = 1;
};
template <> struct Kind<kF32> {
    using T = float;
    static constexpr int step = 16, per_lane = 4, xv = 1;
};
template <> struct Kind<kInt4> {
    using T = bf16;
    static constexpr int step = 128, per_lane = 32, xv = 4;
};

// One K step's operands: a lane's W row piece per tile and x row piece per 16 rows.
template <int W, int NT, int MT>
struct Frag {
    uint4 w[NT], x[MT][Kind<W>::xv];
    float s[NT];  // INT4: the piece's scale
};

template <int W, int NT, int MT>
__device__ __forceinline__ void mma(const Frag<W, NT, MT>& f, f32x4 (&acc)[NT][MT]) {
    if constexpr (W == kBf16) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m)
                acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f.w[n]),
                                                                    __builtin_bit_cast(bf16x8, f.x[m][0]), acc[n][m], 0, 0, 0);
    } else if constexpr (W == kF32) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const float4 a = __builtin_bit_cast(float4, f.w[n]), b = __builtin_bit_cast(float4, f.x[m][0]);
                acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc[n][m], 0, 0, 0);
                acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc[n][m], 0, 0, 0);
                acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc[n][m], 0, 0, 0);
                acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc[n][m], 0, 0, 0);
            }
    } else {
        // a lane's 32 values in four MFMAs: the k order is the same on both operands
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const uint32_t q[4] = {f.w[n].x, f.w[n].y, f.w[n].z, f.w[n].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bf16x8 a = __builtin_bit_cast(bf16x8, q4_dequant8(q[j], f.s[n], -8.0f * f.s[n]));
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, f.x[m][j]),
                                                                        acc[n][m], 0, 0, 0);
            }
        }
    }
}

__device__ __forceinline__ void unpack(const uint4 v, float (&o)[8]) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        o[2 * i] = __uint_as_float(w[i] << 16);
        o[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}

// Bytes between the normalised rows in LDS: consecutive rows' pieces fall on different banks.
__host__ __device__ constexpr int norm_stride(int K, int es) { return K * es + 16; }

// x row / rms * w into LDS, one wave per row (the arithmetic of rmsnorm_fwd_r): the row and the
// weight are loaded in one go, at most kNormChunks vectors per lane.
constexpr int kNormChunks = 4;
template <typename T>
__device__ __forceinline__ void norm_rows(const SkinnyParams& p, char* lds, int waves) {
    constexpr int VN = 16 / sizeof(T);
    const int lane = threadIdx.x & 63;
    for (int row = threadIdx.x >> 6; row < p.M; row += waves) {
        const T* x = static_cast<const T*>(p.A) + row * p.lda;
        char* out = lds + row * norm_stride(p.K, sizeof(T));
        uint4 u[kNormChunks];
        float4 w[kNormChunks][VN / 4];
        float ss = 0.0f;
#pragma unroll
        for (int t = 0; t < kNormChunks; ++t) {
            const int c = (t * 64 + lane) * VN;
            if (t * 64 * VN >= p.K) break;
            u[t] = c < p.K ? *reinterpret_cast<const uint4*>(x + c) : make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < VN / 4; ++i)
                w[t][i] = c < p.K ? *reinterpret_cast<const float4*>(p.norm_w + c + 4 * i) : make_float4(0, 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < kNormChunks; ++t) {
            if (t * 64 * VN >= p.K) break;
            if constexpr (sizeof(T) == 2) {
                float v[8];
                unpack(u[t], v);
#pragma unroll
                for (int i = 0; i < 8; ++i) ss += v[i] * v[i];
            } else {
                const float4 v = __builtin_bit_cast(float4, u[t]);
                ss += v.x * v.x;
                ss += v.y * v.y;
                ss += v.z * v.z;
                ss += v.w * v.w;
            }
        }
        ss = wave_sum(ss);
        const float inv = 1.0f / sqrtf(ss / static_cast<float>(p.K) + p.norm_eps);
#pragma unroll
        for (int t = 0; t < kNormChunks; ++t) {
            const int c = (t * 64 + lane) * VN;
            if (t * 64 * VN >= p.K) break;
            if (c >= p.K) continue;
            if constexpr (sizeof(T) == 2) {
                const float4 w0 = w[t][0], w1 = w[t][VN / 4 - 1];
                float v[8];
                unpack(u[t], v);
                *reinterpret_cast<uint4*>(out + c * 2) =
                    make_uint4(pack_bf16x2((v[0] * inv) * w0.x, (v[1] * inv) * w0.y),
                               pack_bf16x2((v[2] * inv) * w0.z, (v[3] * inv) * w0.w),
                               pack_bf16x2((v[4] * inv) * w1.x, (v[5] * inv) * w1.y),
                               pack_bf16x2((v[6] * inv) * w1.z, (v[7] * inv) * w1.w));
            } else {
                const float4 v = __builtin_bit_cast(float4, u[t]), w0 = w[t][0];
                *reinterpret_cast<float4*>(out + c * 4) =
                    make_float4((v.x * inv) * w0.x, (v.y * inv) * w0.y, (v.z * inv) * w0.z, (v.w * inv) * w0.w);
            }
        }
    }
}

// Four consecutive columns n..n+3 of a row (those below `end`).
template <typename T>
__device__ __forceinline__ void put4(T* row, int n, int end, bool vec, const float (&v)[4]) {
    if (vec && n + 4 <= end) {
        if constexpr (sizeof(T) == 2)
            *reinterpret_cast<uint2*>(row + n) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        else
            *reinterpret_cast<float4*>(row + n) = make_float4(v[0], v[1], v[2], v[3]);
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (n + i < end) st(row, n + i, v[i]);
}

constexpr int kWaves = 8;

template <int W, typename CT, int NT, int MT, bool NORM>
__global__ __launch_bounds__(64 * kWaves) void gemm_skinny_k(const SkinnyParams p) {
    using KD = Kind<W>;
    using T = typename KD::T;
    constexpr int U = MT == 4 ? 2 : (W == kInt4 ? 2 : 4);  // K steps in flight per wave
    extern __shared__ __attribute__((aligned(16))) char skinny_lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    const int first = static_cast<int>(blockIdx.x) * (NT == 2 && p.pair == 16 ? 32 : 16);
    const int n0 = first / p.run * p.run_step + first % p.run;
    f32x4* red = reinterpret_cast<f32x4*>(skinny_lds);              // [kWaves][NT * MT][64]
    char* xn = skinny_lds + kWaves * NT * MT * 1024;                // normalised rows
    int wrow[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) wrow[n] = min(n0 + n * p.pair + c, p.N - 1);
    auto load_w = [&](int step, Frag<W, NT, MT>& f, bool guard) {
        const int k = step * KD::step + KD::per_lane * g;
        const bool ok = !guard || k < p.K;
        const int ks = ok ? k : 0;
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int64_t at = wrow[n] * p.ldw + ks;
            if constexpr (W == kInt4) {
                f.w[n] = *reinterpret_cast<const uint4*>(static_cast<const uint8_t*>(p.W) + at / 2);
                const uint32_t at64 = static_cast<uint32_t>(at >> 6);
                const uint32_t grp = p.gshift >= 0 ? at64 >> p.gshift : at64 / static_cast<uint32_t>(p.G >> 6);
                f.s[n] = static_cast<float>(__builtin_bit_cast(_Float16, p.scales[grp]));
                if (guard && !ok) f.s[n] = 0.0f;
            } else {
                f.w[n] = *reinterpret_cast<const uint4*>(static_cast<const T*>(p.W) + at);
                if (guard && !ok) f.w[n] = make_uint4(0, 0, 0, 0);
            }
        }
    };
    auto load_x = [&](int step, Frag<W, NT, MT>& f, bool guard) {
        const int k = step * KD::step + KD::per_lane * g;
        const bool ok = !guard || k < p.K;
        const int ks = ok ? k : 0;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int row = min(16 * m + c, p.M - 1);
#pragma unroll
            for (int j = 0; j < KD::xv; ++j) {
                const int kj = ks + j * static_cast<int>(16 / sizeof(T));
                if constexpr (NORM)
                    f.x[m][j] = *reinterpret_cast<const uint4*>(xn + row * norm_stride(p.K, sizeof(T)) +
                                                                kj * static_cast<int>(sizeof(T)));
                else
                    f.x[m][j] = *reinterpret_cast<const uint4*>(static_cast<const T*>(p.A) + row * p.lda + kj);
                if (guard && !ok) f.x[m][j] = make_uint4(0, 0, 0, 0);
            }
        }
    };

    f32x4 acc[NT][MT] = {};
    const int full = p.K / KD::step;  // whole K steps
    int s = wave;
    Frag<W, NT, MT> f[U];
    // W does not wait for the rows to be normalised
    const int ahead = s < full ? min(U, (full - s + kWaves - 1) / kWaves) : 0;
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (u < ahead) load_w(s + u * kWaves, f[u], false);
    if (p.r2 > 0 && wave == kWaves - 1) {
        // the low-rank term: row pieces of X2 and Y2 in the dense layout
        constexpr int D = W == kF32 ? kF32 : kBf16;
        for (int k0 = 0; k0 < p.r2; k0 += Kind<D>::step) {
            const int k = k0 + Kind<D>::per_lane * g;
            const bool ok = k < p.r2;
            Frag<D, 1, 1> fr;
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const T* x2 = static_cast<const T*>(p.X2) + low_rank_segment(n0 + n * p.pair, p.N, p.seg_n) * p.r2;
                fr.w[0] = ok ? *reinterpret_cast<const uint4*>(static_cast<const T*>(p.Y2) + wrow[n] * p.ldy2 + k)
                            : make_uint4(0, 0, 0, 0);
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    fr.x[0][0] = ok ? *reinterpret_cast<const uint4*>(x2 + min(16 * m + c, p.M - 1) * p.ldx2 + k)
                                   : make_uint4(0, 0, 0, 0);
                    f32x4 t[1][1] = {{acc[n][m]}};
                    mma<D, 1, 1>(fr, t);
                    acc[n][m] = t[0][0];
                }
            }
        }
    }
    // nor does the residual of the wave that will add it wait for the product
    float res[NT][4] = {};
    if (p.R && wave < MT && 16 * wave + c < p.M) {
        const CT* r = static_cast<const CT*>(p.R) + (16 * wave + c) * p.ldr;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int col = n0 + n * p.pair + 4 * g + i;
                if (col < p.N) res[n][i] = ld(r, col);
            }
    }
    if constexpr (NORM) {
        norm_rows<T>(p, xn, kWaves);
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (u < ahead) {
            load_x(s + u * kWaves, f[u], false);
            mma<W, NT, MT>(f[u], acc);
        }
    s += ahead * kWaves;
    for (; s + (U - 1) * kWaves < full; s += U * kWaves) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            load_w(s + u * kWaves, f[u], false);
            load_x(s + u * kWaves, f[u], false);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) mma<W, NT, MT>(f[u], acc);
    }
    for (; s < full; s += kWaves) {
        load_w(s, f[0], false);
        load_x(s, f[0], false);
        mma<W, NT, MT>(f[0], acc);
    }
    if (full * KD::step < p.K && s == full) {  // the wave whose turn it is takes the rest
        load_w(full, f[0], true);
        load_x(full, f[0], true);
        mma<W, NT, MT>(f[0], acc);
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) red[(wave * NT * MT + n * MT + m) * 64 + lane] = acc[n][m];
    __syncthreads();
    if (wave >= MT) return;
    // wave m: rows 16 m + lane % 16, columns 4 g .. 4 g + 3 of each tile
    const int m = 16 * wave + c;
    float v[NT][4];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        f32x4 t = red[(n * MT + wave) * 64 + lane];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) t += red[(w * NT * MT + n * MT + wave) * 64 + lane];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[n][i] = p.alpha * t[i];
    }
    if (m >= p.M) return;
    CT* C = static_cast<CT*>(p.C) + m * p.ldc;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int col = n0 + n * p.pair + 4 * g;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (col + i >= p.N) continue;
            if (p.beta != 0.0f) v[n][i] += p.beta * ld(C, col + i);
            v[n][i] += res[n][i];
        }
    }
    if constexpr (NT == 2) {
        if (p.rope_cos && n0 < p.rope_cols) {
            const int64_t pos = p.rope_start + m % p.rope_seq;
            const int64_t at = pos * (p.rope_hd / 2) + n0 % p.rope_hd + 4 * g;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // on the values as the product would have stored them
                const float a = sizeof(CT) == 2 ? bf2f(f2bf(v[0][i])) : v[0][i], b = sizeof(CT) == 2 ? bf2f(f2bf(v[1][i])) : v[1][i];
                const float cc = p.rope_cos[at + i], ss = p.rope_sin[at + i];
                v[0][i] = a * cc - b * ss;
                v[1][i] = a * ss + b * cc;
            }
        }
        if (p.glu_out) {
            float h[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (sizeof(CT) == 2) {
                    const float x = bf2f(f2bf(v[0][i]));
                    h[i] = (x * sigmoid_rcp(x)) * bf2f(f2bf(v[1][i]));
                } else {
                    h[i] = v[0][i] / (1.0f + expf(-v[0][i])) * v[1][i];
                }
            }
            put4(static_cast<CT*>(p.glu_out) + m * p.ld_glu, n0 + 4 * g, p.pair, p.vec, h);
            if (!p.store_c) return;
        }
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int col = n0 + n * p.pair + 4 * g;
        // a gate tile ends with the gate columns, not with the matrix
        const int end = p.glu_out && n == 0 ? p.pair : p.N;
        put4(C, col, end, p.vec, v[n]);
        if (p.kc) {
            const int d = p.rope_cols / 2;  // q, k and v are d columns each
            if (col < d) continue;
            CT* cache = static_cast<CT*>(col < 2 * d ? p.kc : p.vc);
            const int64_t row = m / p.rope_seq * p.kv_rows + p.rope_start + m % p.rope_seq;
            put4(cache + row * d, col < 2 * d ? col - d : col - 2 * d, d, p.vec, v[n]);
        }
    }
}

bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
bool a8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }

template <int W, typename CT, int NT, int MT, bool NORM>
void launch(const SkinnyParams& p, int blocks, hipStream_t s) {
    const size_t lds = static_cast<size_t>(kWaves) * NT * MT * 1024 +
                       (NORM ? static_cast<size_t>(p.M) * norm_stride(p.K, sizeof(typename Kind<W>::T)) : 0);
    if (lds > 64 * 1024) {
        static bool configured = false;
        if (!configured) {
            AIC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_skinny_k<W, CT, NT, MT, NORM>),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
            configured = true;
        }
    }
    hipLaunchKernelGGL((gemm_skinny_k<W, CT, NT, MT, NORM>), dim3(blocks), dim3(64 * kWaves), lds, s, p);
    AIC_LAUNCH_CHECK("gemm_skinny");
}

template <int W, typename CT, int NT>
void by_rows(const SkinnyParams& p, int blocks, hipStream_t s) {
    if (p.norm_w) launch<W, CT, NT, 1, true>(p, blocks, s);
    else if (p.M <= 16) launch<W, CT, NT, 1, false>(p, blocks, s);
    else if (p.M <= 32) launch<W, CT, NT, 2, false>(p, blocks, s);
    else launch<W, CT, NT, 4, false>(p, blocks, s);
}

template <int W, typename CT>
void by_tiles(const SkinnyParams& p, int nt, int blocks, hipStream_t s) {
    if (nt == 2) by_rows<W, CT, 2>(p, blocks, s);
    else by_rows<W, CT, 1>(p, blocks, s);
}

}  // namespace

bool gemm_skinny_eligible(const SkinnyArgs& q) {
    const GemmArgs& a = q.g;
    if (a.transA || !a.transB || a.M < 1 || a.M > kSkinnyRows || a.N < 1 || a.K < 1 || a.sq_part || a.dglu_gu) return false;
    const bool f32 = a.ab == DType::Float32;
    const int64_t v = f32 ? 4 : 8;  // elements of 16 bytes
    if (a.K % v || a.lda % v || !a16(a.A)) return false;
    if (f32 && (a.c != DType::Float32 || a.Bq)) return false;
    if (a.Bq) {
        if (!a.Bscale || a.scale_t != DType::Float16 || a.K % 64 || a.ldb % 64 || a.group <= 0 || a.group % 64 ||
            a.group >= (int64_t{1} << 31) || !a16(a.Bq) || a.ldb < a.K || a.N * a.ldb / 64 >= (int64_t{1} << 32))
            return false;
    } else if (a.ldb % v || !a16(a.B)) {
        return false;
    }
    if (a.r2 > 0 && (a.y2_kmajor || a.r2 % v || a.ldx2 % v || a.ldy2 % v || !a16(a.X2) || !a16(a.Y2) || a.seg_n % 16))
        return false;
    if (a.rope_cos && (a.glu_f > 0 || a.rope_hd % 32 || a.rope_cols % a.rope_hd || a.N % a.rope_hd)) return false;
    if (a.glu_f > 0 && (a.N != 2 * a.glu_f || a.glu_f % 16)) return false;
    if (q.norm_w && (a.M > 16 || !a16(q.norm_w) || a.K > 64 * v * kNormChunks ||
                     a.M * norm_stride(static_cast<int>(a.K), static_cast<int>(dtype_size(a.ab))) > 128 * 1024))
        return false;
    if (q.kc && (!a.rope_cos || a.N != a.rope_cols / 2 * 3 || (a.rope_cols / 2) % 4)) return false;
    return true;
}

void gemm_skinny(const SkinnyArgs& q, hipStream_t s) {
    AIC_CHECK(gemm_skinny_eligible(q), InvalidArgument, "skinny GEMM: unsupported shape, layout or dtype");
    const GemmArgs& a = q.g;
    const int64_t es = static_cast<int64_t>(dtype_size(a.c));
    SkinnyParams p{};
    p.A = a.A;
    p.W = a.Bq ? static_cast<const void*>(a.Bq) : a.B;
    p.scales = static_cast<const uint16_t*>(a.Bscale);
    p.C = a.C;
    p.R = a.R;
    p.lda = a.lda; p.ldw = a.ldb; p.ldc = a.ldc; p.ldr = a.ldr;
    p.M = static_cast<int>(a.M); p.N = static_cast<int>(a.N); p.K = static_cast<int>(a.K);
    p.G = static_cast<int>(a.group);
    p.gshift = -1;
    for (int i = 0; i < 25; ++i)
        if (a.group == int64_t{64} << i) p.gshift = i;
    p.alpha = a.alpha; p.beta = a.beta;
    p.X2 = a.X2; p.Y2 = a.Y2;
    p.ldx2 = a.ldx2; p.ldy2 = a.ldy2;
    p.r2 = static_cast<int>(a.r2); p.seg_n = static_cast<int>(a.seg_n);
    p.norm_w = q.norm_w; p.norm_eps = q.norm_eps;
    p.rope_cos = a.rope_cos; p.rope_sin = a.rope_sin;
    p.rope_cols = static_cast<int>(a.rope_cols); p.rope_hd = static_cast<int>(a.rope_hd);
    p.rope_seq = static_cast<int>(a.rope_seq > 0 ? a.rope_seq : 1);
    p.rope_start = static_cast<int>(a.rope_start);
    p.glu_out = a.glu_f > 0 ? a.glu_out : nullptr;
    p.ld_glu = a.ld_glu;
    p.kc = q.kc; p.vc = q.vc; p.kv_rows = q.kv_rows;
    p.store_c = q.skip_c ? 0 : 1;
    auto ok4 = [&](const void* ptr, int64_t ld) { return !ptr || (ld % 4 == 0 && (es == 2 ? a8(ptr) : a16(ptr))); };
    p.vec = ok4(a.C, a.ldc) && ok4(p.glu_out, a.ld_glu) && ok4(q.kc, 4) && ok4(q.vc, 4);
    // which W tiles a block takes: the two halves of a rotary head or of a gate/up pair; otherwise
    // one tile, or two neighbours where that still leaves two blocks per CU (half the x reads)
    int nt = 1, blocks = static_cast<int>((a.N + 15) / 16);
    p.pair = 16;
    p.run = p.run_step = 1 << 30;
    if (a.rope_cos) {
        nt = 2;
        p.pair = p.run = static_cast<int>(a.rope_hd / 2);
        p.run_step = static_cast<int>(a.rope_hd);
        blocks = static_cast<int>(a.N / 32);
        if (p.pair == 16) p.run = 32;  // neighbours: 32 rows per block, which `first` counts in
    } else if (p.glu_out) {
        nt = 2;
        p.pair = static_cast<int>(a.glu_f);
        blocks = static_cast<int>(a.glu_f / 16);
        if (p.pair == 16) p.run = 32;
    } else if (a.N >= 32 * 512) {
        nt = 2;
        blocks = static_cast<int>((a.N + 31) / 32);
    }
    if (a.ab == DType::Float32) {
        by_tiles<kF32, float>(p, nt, blocks, s);
    } else if (a.Bq) {
        if (a.c == DType::Float32) by_tiles<kInt4, float>(p, nt, blocks, s);
        else by_tiles<kInt4, bf16>(p, nt, blocks, s);
    } else {
        if (a.c == DType::Float32) by_tiles<kBf16, float>(p, nt, blocks, s);
        else by_tiles<kBf16, bf16>(p, nt, blocks, s);
    }
}

}  // namespace aic::hip
