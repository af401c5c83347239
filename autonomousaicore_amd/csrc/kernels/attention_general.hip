// Attention for every shape, type and layout that the tuned training kernels (attention.hip) do
// not take: queries and keys of different lengths, a KV cache, fp32 operands, head_dim 16 and 32,
// rows without 16-byte alignment.  Replaces launch_flash_attention_forward/backward_gpu with
// seq_len_q != seq_len_k (src/cuda/cuda_flash_attention.cuh:12-46), the fp32 path of
// src/ops/flash_attention.cpp:32-260 and CausalSelfAttention::forward_with_cache
// (include/nn/attention.hpp:49-120).
//
// All products run on 16x16 MFMA tiles (v_mfma_f32_16x16x32_bf16, v_mfma_f32_16x16x4_f32); the
// scores, the probabilities and their gradients stay fp32.  For bf16 operands a probability (or
// dS) enters its second product as the sum of two bf16 values (the rounded value and the rounded
// remainder, 2^-17 relative), so nothing is rounded to 16 bits before the outputs are.
//
// A wave owns RT tiles of 16 "stationary" rows (queries for the forward and dQ, keys for dK/dV)
// whose operands stay in registers, and walks over blocks of 32 "streaming" rows.  A streaming
// row block is loaded once, straight from global memory in the layout of the first product's A
// operand (lane % 16 = row, 16 bytes of the head per lane), and written from those registers to
// the wave's own LDS, where the second product reads it transposed (ds_read_b64_tr_b16 for bf16).
// The first product gives [streaming x stationary] tiles whose lane layout is that of the second
// product's B operand (its k order permuted alike on both operands), so probabilities never
// leave their lane.  No wave waits for another inside the loop.
//
// Where there are too few stationary tiles to fill the chip (decode, short chunks), `split`
// waves of a block share one group of them, taking every split-th streaming block each, and add
// their partial results through LDS in wave order: deterministic, no atomics, one launch.  A few
// queries of a long cache are shared by blocks as well (key_parts), whose sums a second launch adds
// in block order.
//
// Bound: short sequences by latency (a handful of dependent loads per wave), longer ones by the
// MFMA pipe and LDS reads with 13 products where 7 are counted (the split probabilities).  Forward
// and backward of 64 heads of 128, 128 queries on 2048 keys, bf16: 172 us (32.1 ms with the
// one-thread-per-row kernels before); 512 queries 0.52 ms (74.8), fp32 1.83 ms (48.3); one query of
// 12 heads of 64 on 2048 keys 10 us (6.1 ms).  Error against 64 bits, beside the fp32 probabilities
// and expf of those kernels, over 40 shapes in bf16 (1 to 512 queries, 16 to 2048 keys): o and dv
// 1.7e-3 in both to four digits, dq and dk within 0.2% either way, lse 7e-8 and at the median 0.87 of
// theirs; fp32 1.0e-6 (1.2e-6).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "../runtime/memory_pool.hpp"

namespace aic::hip {

namespace {

typedef __attribute__((address_space(3))) v4i16_t lds_v4i16_t;

constexpr int kRows = 32;  // streaming rows per block: two 16-row tiles

template <typename T>
struct Args {
    const T* q;
    const T* k;
    const T* v;
    const T* o;     // backward: the forward's output (D = rowsum(dO O))
    const T* dout;
    T* out0;        // forward: o; dQ: dq; dK/dV: dk
    T* out1;        // dK/dV: dv
    float* lse;     // [B, H, Sq]: written by the forward (nullable), read by the backward
    float* D;       // [B, H, Sq]: written by the dQ kernel, read by dK/dV
    int64_t ldq, ldk, ldo, ld0, ld1;   // row strides of q; k, v; o and dout; out0; out1
    int64_t qb, kb;                    // rows from one batch to the next of q / o / dout, of k / v
    int B, H, Sq, Sk;
    int coff;       // key c is visible to query r when c <= r + coff
    int split;      // waves sharing a group of stationary rows (a divisor of the block's waves)
    int region;     // LDS bytes per wave
    int parts;      // forward: blocks sharing one group of queries; > 1: attn_general_parts follows
    float* part;    // their sums: [parts][B * H][Sq] rows of HD columns, then of m and l
    float scale;
};

// Per-type operand layout.  A lane's fragment of a 16-row tile is `frags` vectors of `width`
// elements: row lane % 16, head columns step * i + width * (lane / 16) ... + width - 1.
template <typename T, int HD>
struct Lay;
template <int HD>
struct Lay<bf16, HD> {
    using Vec = uint4;
    static constexpr int width = 8, step = 32, frags = HD < 32 ? 1 : HD / 32;
    // LDS row stride in bytes: the four rows of a transposed read fall on disjoint banks
    static constexpr int stride = 2 * HD + (HD >= 64 ? 64 : 0);
};
template <int HD>
struct Lay<float, HD> {
    using Vec = float4;
    static constexpr int width = 4, step = 16, frags = HD / 16;
    // rows four apart are 16 banks apart
    static constexpr int stride = 4 * HD + 16;
};

// One 16-byte vector of a row; VEC: the row pointer is 16-byte aligned.
template <bool VEC>
__device__ __forceinline__ uint4 load_vec(const bf16* p) {
    if constexpr (VEC) {
        return *reinterpret_cast<const uint4*>(p);
    } else {
        const uint16_t* u = reinterpret_cast<const uint16_t*>(p);
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = static_cast<uint32_t>(u[2 * i]) | (static_cast<uint32_t>(u[2 * i + 1]) << 16);
        return make_uint4(w[0], w[1], w[2], w[3]);
    }
}
template <bool VEC>
__device__ __forceinline__ float4 load_vec(const float* p) {
    if constexpr (VEC) return *reinterpret_cast<const float4*>(p);
    else return make_float4(p[0], p[1], p[2], p[3]);
}

// Fragments of row `row` (clamped by the caller) of a [rows][ld] operand at head offset p.
template <typename T, int HD, bool VEC>
__device__ __forceinline__ void load_row(const T* p, int64_t row, int64_t ld, typename Lay<T, HD>::Vec (&f)[Lay<T, HD>::frags]) {
    using L = Lay<T, HD>;
    const int g = (threadIdx.x & 63) >> 4;
    const T* r = p + row * ld;
#pragma unroll
    for (int i = 0; i < L::frags; ++i) {
        const int c = L::step * i + L::width * g;
        if (HD >= L::step || c < HD) f[i] = load_vec<VEC>(r + c);
        else f[i] = typename L::Vec{};
    }
}

template <typename T, int HD>
__device__ __forceinline__ void store_lds(char* tile, int row, const typename Lay<T, HD>::Vec (&f)[Lay<T, HD>::frags]) {
    using L = Lay<T, HD>;
    const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int i = 0; i < L::frags; ++i) {
        const int c = L::step * i + L::width * g;
        if (HD >= L::step || c < HD)
            *reinterpret_cast<typename L::Vec*>(tile + row * L::stride + c * static_cast<int>(sizeof(T))) = f[i];
    }
}

// The 16x16 tile A B^T of two fragment rows (rows of A by rows of B), summed over the head.
template <int HD>
__device__ __forceinline__ f32x4 dot(const uint4 (&a)[Lay<bf16, HD>::frags], const uint4 (&b)[Lay<bf16, HD>::frags]) {
    f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < Lay<bf16, HD>::frags; ++i)
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[i]), __builtin_bit_cast(bf16x8, b[i]), c,
                                                    0, 0, 0);
    return c;
}
template <int HD>
__device__ __forceinline__ f32x4 dot(const float4 (&a)[Lay<float, HD>::frags], const float4 (&b)[Lay<float, HD>::frags]) {
    f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < Lay<float, HD>::frags; ++i) {
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].x, b[i].x, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].y, b[i].y, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].z, b[i].z, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].w, b[i].w, c, 0, 0, 0);
    }
    return c;
}

// The second product's B operand from the 2 x 4 fp32 values a lane holds of a 32-row block (rows
// 16 t + 4 g + i of column lane % 16).
template <typename T>
struct Weights;
template <>
struct Weights<bf16> {
    bf16x8 hi, lo;
    __device__ __forceinline__ void set(const float (&p)[2][4]) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bf16 h = f2bf(p[t][i]);
                hi[4 * t + i] = h;
                lo[4 * t + i] = f2bf(p[t][i] - bf2f(h));
            }
    }
};
template <>
struct Weights<float> {
    float w[2][4];
    __device__ __forceinline__ void set(const float (&p)[2][4]) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) w[t][i] = p[t][i];
    }
};

// acc[dt][r] (rows: head columns 16 dt + 4 g + i, columns: stationary rows) += X^T W of the 32
// streaming rows X in `tile`.
template <int HD, int RT>
__device__ __forceinline__ void accumulate(const char* tile, const Weights<bf16> (&w)[RT], f32x4 (&acc)[HD / 16][RT]) {
    using L = Lay<bf16, HD>;
    const int lane = threadIdx.x & 63, g = lane >> 4, j = (lane & 15) >> 2, c = lane & 3;
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) {
        v4i16_t r[2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
            r[t] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_v4i16_t*)(tile + (16 * t + 4 * g + j) * L::stride + 2 * (16 * dt + 4 * c)));
        const uint2 a = __builtin_bit_cast(uint2, r[0]), b = __builtin_bit_cast(uint2, r[1]);
        const bf16x8 x = __builtin_bit_cast(bf16x8, make_uint4(a.x, a.y, b.x, b.y));
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            acc[dt][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, w[i].lo, acc[dt][i], 0, 0, 0);
            acc[dt][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, w[i].hi, acc[dt][i], 0, 0, 0);
        }
    }
}
template <int HD, int RT>
__device__ __forceinline__ void accumulate(const char* tile, const Weights<float> (&w)[RT], f32x4 (&acc)[HD / 16][RT]) {
    using L = Lay<float, HD>;
    const int lane = threadIdx.x & 63, g = lane >> 4;
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = *reinterpret_cast<const float*>(tile + (16 * t + 4 * g + e) * L::stride +
                                                                4 * (16 * dt + (lane & 15)));
#pragma unroll
                for (int i = 0; i < RT; ++i)
                    acc[dt][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, w[i].w[t][e], acc[dt][i], 0, 0, 0);
            }
}

template <typename T>
__device__ __forceinline__ float exp_of(float x) {
    if constexpr (sizeof(T) == 2) return __expf(x);
    else return expf(x);
}

// Four consecutive elements of an output row.
template <bool VEC>
__device__ __forceinline__ void store4(float* p, float a, float b, float c, float d) {
    if constexpr (VEC) {
        *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d);
    } else {
        p[0] = a;
        p[1] = b;
        p[2] = c;
        p[3] = d;
    }
}
template <bool VEC>
__device__ __forceinline__ void store4(bf16* p, float a, float b, float c, float d) {
    if constexpr (VEC) {
        *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(a, b), pack_bf16x2(c, d));
    } else {
        p[0] = f2bf(a);
        p[1] = f2bf(b);
        p[2] = f2bf(c);
        p[3] = f2bf(d);
    }
}

// LDS of one wave: its streaming tiles, later (split > 1) its partial accumulators as
// [HD / 16][RT][64 lanes] x 16 bytes per array, and two floats per lane and tile.
template <typename T, int HD, int RT, int TILES, int ACCS>
constexpr int region_bytes() {
    constexpr int tiles = TILES * kRows * Lay<T, HD>::stride;
    constexpr int accs = ACCS > 0 ? ACCS * HD / 16 * RT * 1024 + 2 * RT * 64 * 4 : 0;
    return ((tiles > accs ? tiles : accs) + 15) & ~15;
}

template <int HD, int RT>
__device__ __forceinline__ void park(char* region, const f32x4 (&acc)[HD / 16][RT]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt)
#pragma unroll
        for (int r = 0; r < RT; ++r) *reinterpret_cast<f32x4*>(region + ((dt * RT + r) * 64 + lane) * 16) = acc[dt][r];
}

// A hidden or missing row enters the tiles with weight zero, and zero times an infinity is NaN;
// so is an infinity times the zero remainder of a bf16 weight.  Rows whose sums came out
// non-finite are therefore summed again by `outer`, in fp32 and over exactly the rows they see: bit c
// of the result is stationary row c of tile r.  Not where the row's weights are NaN themselves (a NaN or
// an overflow in what it sees): then so is every sum.  64 heads of 64, 512 causal tokens, bf16,
// forward and backward: 77 us, with NaN throughout 78, with an infinity in every value row 736 (15 ms each
// when one wave formed such rows one after the other; 2.4 ms with one thread per row throughout).
template <int HD, int RT>
__device__ __forceinline__ unsigned non_finite(const f32x4 (&acc)[HD / 16][RT], int r) {
    bool bad = false;
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) bad |= !(fabsf(acc[dt][r][i]) <= 3.402823466e38f);
    const unsigned long long m = __ballot(bad);
    return static_cast<unsigned>((m | (m >> 16) | (m >> 32) | (m >> 48)) & 0xffffu);
}
// Bit c: x of stationary row c (every lane c of the four groups holds it) is a number.
__device__ __forceinline__ unsigned numbers(float x) { return static_cast<unsigned>(__ballot(x == x) & 0xffffu); }

__device__ __forceinline__ float vec_dot(const uint4& a, const uint4& b, float s) {
    const uint32_t x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        s = fmaf(__uint_as_float(x[e] << 16), __uint_as_float(y[e] << 16), s);
        s = fmaf(__uint_as_float(x[e] & 0xffff0000u), __uint_as_float(y[e] & 0xffff0000u), s);
    }
    return s;
}
__device__ __forceinline__ float vec_dot(const float4& a, const float4& b, float s) {
    return fmaf(a.w, b.w, fmaf(a.z, b.z, fmaf(a.y, b.y, fmaf(a.x, b.x, s))));
}

// acc += X^T W as accumulate for one tile of stationary rows, a streaming row at a time and only
// where seen(row) holds for this lane's stationary row; x: the weights as a lane holds them.
__device__ __forceinline__ f32x4 four(const bf16* p) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    return f32x4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                 __uint_as_float(u.y & 0xffff0000u)};
}
__device__ __forceinline__ f32x4 four(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
template <typename T, int HD, typename Seen>
__device__ __forceinline__ void outer(const char* tile, const float (&x)[2][4], Seen&& seen, f32x4 (&acc)[HD / 16]) {
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll 1
            for (int j = 0; j < 4; ++j) {
                const int row = 16 * t + 4 * j + i;
                const T* p = reinterpret_cast<const T*>(tile + row * Lay<T, HD>::stride) + 4 * g;
                const float w = __shfl(x[t][i], 16 * j + c);
                if (seen(row)) {
#pragma unroll
                    for (int dt = 0; dt < HD / 16; ++dt) acc[dt] += w * four(p + 16 * dt);
                }
            }
}

// The same for one query (attn_general_parts): 64 keys at a time, a lane each for the products of whole rows
// (row_dot), then the lanes as columns for the weighted sums (Sums): lane l holds the columns l % 64
// and l % 64 + 64 of a head, heads of 16 and 32 in groups of lanes with every 4th and 2nd row.
template <typename T, int HD>
__device__ __forceinline__ float row_dot(const T* a, const T* b) {
    float s = 0.0f;
#pragma unroll 4
    for (int c = 0; c < HD; c += Lay<T, HD>::width) s = vec_dot(load_vec<false>(a + c), load_vec<false>(b + c), s);
    return s;
}
template <typename T, int HD>
struct Sums {
    static constexpr int C = HD < 64 ? HD : 64, G = 64 / C;
    float a = 0.0f, b = 0.0f;
    // += the rows p, p + ld, ... of n lanes, weighted by each lane's w
    __device__ __forceinline__ void add(const T* p, int64_t ld, int n, float w) {
        const int lane = threadIdx.x & 63, g = lane / C, c = lane % C;
#pragma unroll 8
        for (int j = 0; j < n; j += G) {
            const int r = min(j + g, n - 1);
            const float x = aic::hip::ld(p + r * ld, c), y = HD > 64 ? aic::hip::ld(p + r * ld, c + 64) : 0.0f;
            const float wr = __shfl(w, r);
            if (j + g < n) {
                a = fmaf(wr, x, a);
                if (HD > 64) b = fmaf(wr, y, b);
            }
        }
    }
    __device__ __forceinline__ void store(T* p, float f) {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int o = C; o < 64; o *= 2) a += __shfl_xor(a, o);
        if (lane < HD) st(p, lane, a * f);
        if (HD > 64) st(p, lane + 64, b * f);
    }
};

__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

extern __shared__ __attribute__((aligned(16))) char gen_lds[];

// Query qi's output from exactly the keys it sees; m and l: its scores' maximum and weights' sum.
template <typename T, int HD>
__device__ __forceinline__ void redo_row(const Args<T>& p, const T* qh, const T* kh, const T* vh, int64_t qi, float m,
                                         float l, T* out) {
    const int lane = threadIdx.x & 63, end = min(p.Sk, static_cast<int>(qi) + p.coff + 1);
    const float base = m == -INFINITY ? 0.0f : m;
    Sums<T, HD> o;
    for (int k0 = 0; k0 < end; k0 += 64) {
        const int n = min(64, end - k0);
        const float x = row_dot<T, HD>(qh + qi * p.ldq, kh + (k0 + min(lane, n - 1)) * p.ldk) * p.scale;
        o.add(vh + k0 * p.ldk, p.ldk, n, exp_of<T>(x - base));
    }
    o.store(out, 1.0f / l);
}

// ---------------------------------------------------------------------------------------
// Forward: out0 = softmax(q k^T scale) v, lse.
// ---------------------------------------------------------------------------------------
// PARTS: block b / (B H) of a group takes every parts-th round of its keys and leaves its sums to
// attn_general_parts.
template <typename T, int HD, int RT, bool VEC, bool PARTS>
__global__ __launch_bounds__(512) void attn_general_fwd(const Args<T> p) {
    using L = Lay<T, HD>;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    const int nbh = p.B * p.H, bh = static_cast<int>(blockIdx.x) % nbh;
    const int per_block = (blockDim.x >> 6) / p.split;
    const int part = wave % p.split;
    const int share = PARTS ? static_cast<int>(blockIdx.x) / nbh : 0;
    const int q0 = PARTS ? 0 : (static_cast<int>(blockIdx.x) / nbh * per_block + wave / p.split) * 16 * RT;
    const int b = bh / p.H, h = bh % p.H;
    const T* qh = p.q + static_cast<int64_t>(b) * p.qb * p.ldq + static_cast<int64_t>(h) * HD;
    const T* kh = p.k + static_cast<int64_t>(b) * p.kb * p.ldk + static_cast<int64_t>(h) * HD;
    const T* vh = p.v + static_cast<int64_t>(b) * p.kb * p.ldk + static_cast<int64_t>(h) * HD;
    char* region = gen_lds + wave * p.region;

    f32x4 acc[HD / 16][RT] = {};
    float m[RT], l[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        m[r] = -INFINITY;
        l[r] = 0.0f;
    }
    if (q0 < p.Sq) {
        typename L::Vec qf[RT][L::frags];
        int vis[RT];  // visible keys of this lane's queries
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int qi = min(q0 + 16 * r + c, p.Sq - 1);
            load_row<T, HD, VEC>(qh, qi, p.ldq, qf[r]);
            vis[r] = min(p.Sk, qi + p.coff + 1);
        }
        const int kend = min(p.Sk, min(q0 + 16 * RT, p.Sq) + p.coff);
        const int kfull = min(p.Sk, q0 + p.coff + 1);  // keys every query of the wave sees
        typename L::Vec kf[2][L::frags], vf[2][L::frags];
        auto load = [&](int k0) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int row = min(k0 + 16 * t + c, p.Sk - 1);
                load_row<T, HD, VEC>(kh, row, p.ldk, kf[t]);
                load_row<T, HD, VEC>(vh, row, p.ldk, vf[t]);
            }
        };
        const int stride = kRows * p.split * (PARTS ? p.parts : 1);
        int k0 = kRows * (share * p.split + part);
        if (k0 < kend) load(k0);
        for (; k0 < kend; k0 += stride) {
            wait_lds();  // the previous block's transposed reads
#pragma unroll
            for (int t = 0; t < 2; ++t) store_lds<T, HD>(region, 16 * t + c, vf[t]);
            f32x4 s[2][RT];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < RT; ++r) s[t][r] = dot<HD>(kf[t], qf[r]);
            if (k0 + stride < kend) load(k0 + stride);
            Weights<T> w[RT];
            const bool masked = k0 + kRows > kfull;
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                float x[2][4], mx = -INFINITY;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        x[t][i] = s[t][r][i] * p.scale;
                        if (masked && k0 + 16 * t + 4 * g + i >= vis[r]) x[t][i] = -INFINITY;
                        mx = fmaxf(mx, x[t][i]);
                    }
                mx = fmaxf(mx, __shfl_xor(mx, 16));
                mx = fmaxf(mx, __shfl_xor(mx, 32));
                const float mn = fmaxf(m[r], mx);
                // nothing visible so far: keep the sums at zero instead of -inf - -inf
                const float base = mn == -INFINITY ? 0.0f : mn;
                const float f = exp_of<T>(m[r] - base);
                float sum = 0.0f;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        x[t][i] = exp_of<T>(x[t][i] - base);
                        sum += x[t][i];
                    }
                l[r] = l[r] * f + sum;  // this lane's keys only; added across lanes at the end
                m[r] = mn;
                if (__any(f != 1.0f)) {
#pragma unroll
                    for (int dt = 0; dt < HD / 16; ++dt) acc[dt][r] *= f;
                }
                w[r].set(x);
            }
            wait_lds();
            accumulate<HD, RT>(region, w, acc);
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            l[r] += __shfl_xor(l[r], 16);
            l[r] += __shfl_xor(l[r], 32);
        }
    }
    if (p.split > 1) {
        // every wave of the block reaches the barriers; the group's waves add the partial sums of
        // a share of the head columns each, part 0 collects them
        wait_lds();
        constexpr int STAT = HD / 16 * RT * 1024;
        park<HD, RT>(region, acc);
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            reinterpret_cast<float*>(region + STAT)[r * 64 + lane] = m[r];
            reinterpret_cast<float*>(region + STAT)[(RT + r) * 64 + lane] = l[r];
        }
        __syncthreads();
        char* group = gen_lds + (wave - part) * p.region;
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            float pm[8], mx = -INFINITY;
#pragma unroll
            for (int w = 0; w < 8; ++w)
                if (w < p.split) {
                    pm[w] = reinterpret_cast<const float*>(group + w * p.region + STAT)[r * 64 + lane];
                    mx = fmaxf(mx, pm[w]);
                }
            const float base = mx == -INFINITY ? 0.0f : mx;
            l[r] = 0.0f;
#pragma unroll
            for (int w = 0; w < 8; ++w)
                if (w < p.split) {
                    pm[w] = exp_of<T>(pm[w] - base);
                    l[r] += pm[w] * reinterpret_cast<const float*>(group + w * p.region + STAT)[(RT + r) * 64 + lane];
                }
            m[r] = mx;
            for (int dt = part; dt < HD / 16; dt += p.split) {
                f32x4 t = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int w = 0; w < 8; ++w)
                    if (w < p.split)
                        t += pm[w] * *reinterpret_cast<const f32x4*>(group + w * p.region + ((dt * RT + r) * 64 + lane) * 16);
                *reinterpret_cast<f32x4*>(group + ((dt * RT + r) * 64 + lane) * 16) = t;
            }
        }
        __syncthreads();
        if (part != 0) return;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt)
#pragma unroll
            for (int r = 0; r < RT; ++r) acc[dt][r] = *reinterpret_cast<const f32x4*>(region + ((dt * RT + r) * 64 + lane) * 16);
    }
    if constexpr (PARTS) {
        if (c >= p.Sq) return;
        const int64_t row = (static_cast<int64_t>(share) * nbh + bh) * p.Sq + c;
        float* st = p.part + static_cast<int64_t>(p.parts) * nbh * p.Sq * HD + 2 * row;
        if (g == 0) {
            st[0] = m[0];
            st[1] = l[0];
        }
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) *reinterpret_cast<f32x4*>(p.part + row * HD + 16 * dt + 4 * g) = acc[dt][0];
        return;
    }
    unsigned redo = 0;  // bit 16 r + c: row c of tile r
    T* out = p.out0 + (static_cast<int64_t>(b) * p.qb + q0 + c) * p.ld0 + static_cast<int64_t>(h) * HD + 4 * g;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const unsigned bad = non_finite<HD, RT>(acc, r) & numbers(l[r]);
        redo |= bad << (16 * r);
        const int qi = q0 + 16 * r + c;
        if (qi >= p.Sq) continue;
        if (p.lse && g == 0) p.lse[(static_cast<int64_t>(b) * p.H + h) * p.Sq + qi] = m[r] + logf(l[r]);
        if ((bad >> c) & 1) continue;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) {
            const f32x4 a = acc[dt][r] / l[r];
            store4<VEC>(out + 16 * r * p.ld0 + 16 * dt, a[0], a[1], a[2], a[3]);
        }
    }
#pragma unroll 1
    for (int r = 0; r < RT; ++r) {
        if (!((redo >> (16 * r)) & 0xffffu)) continue;
        const int qi = q0 + 16 * r + c, end = min(p.Sk, qi + p.coff + 1);
        const int kend = min(p.Sk, min(q0 + 16 * r + 16, p.Sq) + p.coff);
        const float mr = RT > 1 && r ? m[RT - 1] : m[0], lr = RT > 1 && r ? l[RT - 1] : l[0];
        const float base = mr == -INFINITY ? 0.0f : mr;
        typename L::Vec qf[L::frags], f[L::frags];
        load_row<T, HD, VEC>(qh, min(qi, p.Sq - 1), p.ldq, qf);
        f32x4 sum[HD / 16] = {};
        for (int k0 = 0; k0 < kend; k0 += kRows) {
            float x[2][4];
            wait_lds();
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int row = min(k0 + 16 * t + c, p.Sk - 1);
                load_row<T, HD, VEC>(vh, row, p.ldk, f);
                store_lds<T, HD>(region, 16 * t + c, f);
                load_row<T, HD, VEC>(kh, row, p.ldk, f);
                const f32x4 s = dot<HD>(f, qf);
#pragma unroll
                for (int i = 0; i < 4; ++i) x[t][i] = exp_of<T>(s[i] * p.scale - base);
            }
            wait_lds();
            outer<T, HD>(region, x, [&](int row) { return k0 + row < end; }, sum);
        }
        if (qi >= p.Sq || !((redo >> (16 * r + c)) & 1)) continue;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) {
            const f32x4 a = sum[dt] / lr;
            store4<VEC>(out + 16 * r * p.ld0 + 16 * dt, a[0], a[1], a[2], a[3]);
        }
    }
}

// The parts' sums of one query and head added in part order, one wave each.
template <typename T, int HD>
__global__ __launch_bounds__(64) void attn_general_parts(const Args<T> p) {
    const int lane = threadIdx.x, nbh = p.B * p.H, rows = nbh * p.Sq, row = static_cast<int>(blockIdx.x);
    const int bh = row / p.Sq, qi = row % p.Sq, b = bh / p.H, h = bh % p.H;
    const float* st = p.part + static_cast<int64_t>(p.parts) * rows * HD;
    const float m = lane < p.parts ? st[2 * (lane * static_cast<int64_t>(rows) + row)] : -INFINITY;
    const float l = lane < p.parts ? st[2 * (lane * static_cast<int64_t>(rows) + row) + 1] : 0.0f;
    float mx = m;
#pragma unroll
    for (int o = 1; o < 64; o *= 2) mx = fmaxf(mx, __shfl_xor(mx, o));
    const float w = exp_of<T>(m - (mx == -INFINITY ? 0.0f : mx));
    const float sum = wave_sum(w * l);
    float oa = 0.0f, ob = 0.0f;
#pragma unroll 4
    for (int u = 0; u < p.parts; ++u) {
        const float* v = p.part + (static_cast<int64_t>(u) * rows + row) * HD;
        const float wu = __shfl(w, u);
        oa = fmaf(wu, lane < HD ? v[lane] : 0.0f, oa);
        ob = fmaf(wu, lane + 64 < HD ? v[lane + 64] : 0.0f, ob);
    }
    T* out = p.out0 + (static_cast<int64_t>(b) * p.qb + qi) * p.ld0 + static_cast<int64_t>(h) * HD;
    if (p.lse && lane == 0) p.lse[row] = mx + logf(sum);
    const bool bad = !(fabsf(oa) <= 3.402823466e38f) || !(fabsf(ob) <= 3.402823466e38f);
    if (sum == sum && __any(bad)) {  // as non_finite
        const T* qh = p.q + static_cast<int64_t>(b) * p.qb * p.ldq + static_cast<int64_t>(h) * HD;
        const int64_t kv = static_cast<int64_t>(b) * p.kb * p.ldk + static_cast<int64_t>(h) * HD;
        redo_row<T, HD>(p, qh, p.k + kv, p.v + kv, qi, mx, sum, out);
    } else {
        if (lane < HD) aic::hip::st(out, lane, oa / sum);
        if (lane + 64 < HD) aic::hip::st(out, lane + 64, ob / sum);
    }
}

// Adds the partial accumulators of a group's other waves (parked in their regions) to part 0's.
template <int HD, int RT>
__device__ __forceinline__ void gather(const char* region, int stride, int at, int split, f32x4 (&acc)[HD / 16][RT]) {
    const int lane = threadIdx.x & 63;
    for (int w = 1; w < split; ++w)
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt)
#pragma unroll
            for (int r = 0; r < RT; ++r)
                acc[dt][r] += *reinterpret_cast<const f32x4*>(region + w * stride + at + ((dt * RT + r) * 64 + lane) * 16);
}

// ---------------------------------------------------------------------------------------
// Backward, queries: D = rowsum(dO O) (written for dK/dV) and dq = scale sum_k dS k.
// ---------------------------------------------------------------------------------------
template <typename T, int HD, int RT, bool VEC>
__global__ __launch_bounds__(256) void attn_general_dq(const Args<T> p) {
    using L = Lay<T, HD>;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    const int nbh = p.B * p.H, bh = static_cast<int>(blockIdx.x) % nbh;
    const int per_block = (blockDim.x >> 6) / p.split;
    const int part = wave % p.split;
    const int q0 = (static_cast<int>(blockIdx.x) / nbh * per_block + wave / p.split) * 16 * RT;
    const int b = bh / p.H, h = bh % p.H;
    const int64_t hoff = static_cast<int64_t>(h) * HD, tok0 = static_cast<int64_t>(b) * p.qb;
    const T* kh = p.k + static_cast<int64_t>(b) * p.kb * p.ldk + hoff;
    const T* vh = p.v + static_cast<int64_t>(b) * p.kb * p.ldk + hoff;
    char* region = gen_lds + wave * p.region;

    f32x4 acc[HD / 16][RT] = {};
    float lse[RT] = {}, D[RT] = {};
    if (q0 < p.Sq) {
        typename L::Vec qf[RT][L::frags], df[RT][L::frags];
        int vis[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int qi = min(q0 + 16 * r + c, p.Sq - 1);
            load_row<T, HD, VEC>(p.q + tok0 * p.ldq + hoff, qi, p.ldq, qf[r]);
            load_row<T, HD, VEC>(p.dout + tok0 * p.ldo + hoff, qi, p.ldo, df[r]);
            vis[r] = min(p.Sk, qi + p.coff + 1);
            const int64_t at = (static_cast<int64_t>(b) * p.H + h) * p.Sq + qi;
            lse[r] = p.lse[at];
            typename L::Vec of[L::frags];
            load_row<T, HD, VEC>(p.o + tok0 * p.ldo + hoff, qi, p.ldo, of);
            float d = 0.0f;
#pragma unroll
            for (int i = 0; i < L::frags; ++i) d = vec_dot(of[i], df[r][i], d);
            d += __shfl_xor(d, 16);
            d += __shfl_xor(d, 32);
            D[r] = d;
            if (part == 0 && g == 0 && q0 + 16 * r + c < p.Sq) p.D[at] = d;
        }
        const int kend = min(p.Sk, min(q0 + 16 * RT, p.Sq) + p.coff);
        const int kfull = min(p.Sk, q0 + p.coff + 1);
        for (int k0 = kRows * part; k0 < kend; k0 += kRows * p.split) {
            typename L::Vec kf[2][L::frags], vf[2][L::frags];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int row = min(k0 + 16 * t + c, p.Sk - 1);
                load_row<T, HD, VEC>(kh, row, p.ldk, kf[t]);
                load_row<T, HD, VEC>(vh, row, p.ldk, vf[t]);
            }
            wait_lds();  // the previous block's transposed reads
#pragma unroll
            for (int t = 0; t < 2; ++t) store_lds<T, HD>(region, 16 * t + c, kf[t]);
            Weights<T> w[RT];
            const bool masked = k0 + kRows > kfull;
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                float x[2][4];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const f32x4 s = dot<HD>(kf[t], qf[r]), dp = dot<HD>(vf[t], df[r]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float pr = exp_of<T>(fmaf(s[i], p.scale, -lse[r]));
                        x[t][i] = masked && k0 + 16 * t + 4 * g + i >= vis[r] ? 0.0f : pr * (dp[i] - D[r]);
                    }
                }
                w[r].set(x);
            }
            wait_lds();
            accumulate<HD, RT>(region, w, acc);
        }
    }
    if (p.split > 1) {
        wait_lds();
        park<HD, RT>(region, acc);
        __syncthreads();
        if (part != 0) return;
        gather<HD, RT>(region, p.region, 0, p.split, acc);
    }
    unsigned redo = 0;  // as the forward's
    T* out = p.out0 + (tok0 + q0 + c) * p.ld0 + hoff + 4 * g;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const unsigned bad = non_finite<HD, RT>(acc, r) & numbers(lse[r]) & numbers(D[r]);
        redo |= bad << (16 * r);
        if (q0 + 16 * r + c >= p.Sq || ((bad >> c) & 1)) continue;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) {
            const f32x4 a = acc[dt][r] * p.scale;
            store4<VEC>(out + 16 * r * p.ld0 + 16 * dt, a[0], a[1], a[2], a[3]);
        }
    }
#pragma unroll 1
    for (int r = 0; r < RT; ++r) {
        if (!((redo >> (16 * r)) & 0xffffu)) continue;
        const int qi = q0 + 16 * r + c, end = min(p.Sk, qi + p.coff + 1);
        const int kend = min(p.Sk, min(q0 + 16 * r + 16, p.Sq) + p.coff);
        const float lr = RT > 1 && r ? lse[RT - 1] : lse[0], Dr = RT > 1 && r ? D[RT - 1] : D[0];
        typename L::Vec qf[L::frags], df[L::frags], f[L::frags];
        load_row<T, HD, VEC>(p.q + tok0 * p.ldq + hoff, min(qi, p.Sq - 1), p.ldq, qf);
        load_row<T, HD, VEC>(p.dout + tok0 * p.ldo + hoff, min(qi, p.Sq - 1), p.ldo, df);
        f32x4 sum[HD / 16] = {};
        for (int k0 = 0; k0 < kend; k0 += kRows) {
            float x[2][4];
            wait_lds();
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int row = min(k0 + 16 * t + c, p.Sk - 1);
                load_row<T, HD, VEC>(vh, row, p.ldk, f);
                const f32x4 dp = dot<HD>(f, df);
                load_row<T, HD, VEC>(kh, row, p.ldk, f);
                store_lds<T, HD>(region, 16 * t + c, f);
                const f32x4 s = dot<HD>(f, qf);
#pragma unroll
                for (int i = 0; i < 4; ++i) x[t][i] = exp_of<T>(fmaf(s[i], p.scale, -lr)) * (dp[i] - Dr);
            }
            wait_lds();
            outer<T, HD>(region, x, [&](int row) { return k0 + row < end; }, sum);
        }
        if (qi >= p.Sq || !((redo >> (16 * r + c)) & 1)) continue;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) {
            const f32x4 a = sum[dt] * p.scale;
            store4<VEC>(out + 16 * r * p.ld0 + 16 * dt, a[0], a[1], a[2], a[3]);
        }
    }
}

// ---------------------------------------------------------------------------------------
// Backward, keys: dk = scale sum_q dS q, dv = sum_q P dO.  Zero where no query sees the key.
// ---------------------------------------------------------------------------------------
template <typename T, int HD, int RT, bool VEC>
__global__ __launch_bounds__(256) void attn_general_dkdv(const Args<T> p) {
    using L = Lay<T, HD>;
    constexpr int ACC = HD / 16 * RT * 1024;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    const int nbh = p.B * p.H, bh = static_cast<int>(blockIdx.x) % nbh;
    const int per_block = (blockDim.x >> 6) / p.split;
    const int part = wave % p.split;
    const int k0 = (static_cast<int>(blockIdx.x) / nbh * per_block + wave / p.split) * 16 * RT;
    const int b = bh / p.H, h = bh % p.H;
    const int64_t hoff = static_cast<int64_t>(h) * HD;
    const T* qh = p.q + static_cast<int64_t>(b) * p.qb * p.ldq + hoff;
    const T* dh = p.dout + static_cast<int64_t>(b) * p.qb * p.ldo + hoff;
    const float* lse_h = p.lse + (static_cast<int64_t>(b) * p.H + h) * p.Sq;
    const float* D_h = p.D + (static_cast<int64_t>(b) * p.H + h) * p.Sq;
    char* region = gen_lds + wave * p.region;
    char* region_d = region + kRows * L::stride;

    f32x4 dk[HD / 16][RT] = {}, dv[HD / 16][RT] = {};
    if (k0 < p.Sk) {
        typename L::Vec kf[RT][L::frags], vf[RT][L::frags];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int row = min(k0 + 16 * r + c, p.Sk - 1);
            load_row<T, HD, VEC>(p.k + static_cast<int64_t>(b) * p.kb * p.ldk + hoff, row, p.ldk, kf[r]);
            load_row<T, HD, VEC>(p.v + static_cast<int64_t>(b) * p.kb * p.ldk + hoff, row, p.ldk, vf[r]);
        }
        // the first query that sees a key of the wave, and the first that sees them all
        const int qfirst = max(0, k0 - p.coff), qfull = max(0, min(k0 + 16 * RT, p.Sk) - 1 - p.coff);
        for (int q0 = qfirst / kRows * kRows + kRows * part; q0 < p.Sq; q0 += kRows * p.split) {
            typename L::Vec qf[2][L::frags], df[2][L::frags];
            float lse[2][4], D[2][4];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int row = min(q0 + 16 * t + c, p.Sq - 1);
                load_row<T, HD, VEC>(qh, row, p.ldq, qf[t]);
                load_row<T, HD, VEC>(dh, row, p.ldo, df[t]);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int qi = min(q0 + 16 * t + 4 * g + i, p.Sq - 1);
                    lse[t][i] = lse_h[qi];
                    D[t][i] = D_h[qi];
                }
            }
            wait_lds();  // the previous block's transposed reads
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                store_lds<T, HD>(region, 16 * t + c, qf[t]);
                store_lds<T, HD>(region_d, 16 * t + c, df[t]);
            }
            Weights<T> wp[RT], ws[RT];
            const bool masked = q0 < qfull || q0 + kRows > p.Sq;
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                float x[2][4], y[2][4];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const f32x4 s = dot<HD>(qf[t], kf[r]), dp = dot<HD>(df[t], vf[r]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int qi = q0 + 16 * t + 4 * g + i;
                        const bool hide = masked && (qi >= p.Sq || k0 + 16 * r + c > qi + p.coff);
                        x[t][i] = hide ? 0.0f : exp_of<T>(fmaf(s[i], p.scale, -lse[t][i]));
                        y[t][i] = hide ? 0.0f : x[t][i] * (dp[i] - D[t][i]);
                    }
                }
                wp[r].set(x);
                ws[r].set(y);
            }
            wait_lds();
            accumulate<HD, RT>(region_d, wp, dv);
            accumulate<HD, RT>(region, ws, dk);
        }
    }
    if (p.split > 1) {
        wait_lds();
        park<HD, RT>(region, dk);
        park<HD, RT>(region + ACC, dv);
        __syncthreads();
        if (part != 0) return;
        gather<HD, RT>(region, p.region, 0, p.split, dk);
        gather<HD, RT>(region, p.region, ACC, p.split, dv);
    }
    unsigned redo = 0;  // as the forward's
    const int64_t row0 = static_cast<int64_t>(b) * p.kb + k0 + c;
    T *out_k = p.out0 + row0 * p.ld0 + hoff + 4 * g, *out_v = p.out1 + row0 * p.ld1 + hoff + 4 * g;
    int nan_lse = -2, nan_D = -2;  // the last query whose lse, D is NaN; -2: not looked for yet
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const unsigned bad_k = non_finite<HD, RT>(dk, r), bad_v = non_finite<HD, RT>(dv, r);
        if ((bad_k | bad_v) && nan_lse == -2) {
            nan_lse = nan_D = -1;
#pragma unroll 4
            for (int qi = lane; qi < p.Sq; qi += 64) {
                if (lse_h[qi] != lse_h[qi]) nan_lse = qi;
                if (D_h[qi] != D_h[qi]) nan_D = qi;
            }
#pragma unroll
            for (int o = 1; o < 64; o *= 2) {
                nan_lse = max(nan_lse, __shfl_xor(nan_lse, o));
                nan_D = max(nan_D, __shfl_xor(nan_D, o));
            }
        }
        // a NaN lse that the key is seen with makes both sums NaN, a NaN D dK's
        const int key = k0 + 16 * r + c, first = max(0, key - p.coff);
        const bool bad = nan_lse < first && ((((nan_D < first ? bad_k : 0u) | bad_v) >> c) & 1);
        redo |= static_cast<unsigned>(__ballot(bad) & 0xffffu) << (16 * r);
        if (key >= p.Sk || bad) continue;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) {
            const f32x4 a = dk[dt][r] * p.scale, d = dv[dt][r];
            store4<VEC>(out_k + 16 * r * p.ld0 + 16 * dt, a[0], a[1], a[2], a[3]);
            store4<VEC>(out_v + 16 * r * p.ld1 + 16 * dt, d[0], d[1], d[2], d[3]);
        }
    }
#pragma unroll 1
    for (int r = 0; r < RT; ++r) {
        if (!((redo >> (16 * r)) & 0xffffu)) continue;
        const int key = k0 + 16 * r + c;
        const int64_t krow = min(key, p.Sk - 1);
        typename L::Vec kf[L::frags], vf[L::frags], f[L::frags];
        load_row<T, HD, VEC>(p.k + static_cast<int64_t>(b) * p.kb * p.ldk + hoff, krow, p.ldk, kf);
        load_row<T, HD, VEC>(p.v + static_cast<int64_t>(b) * p.kb * p.ldk + hoff, krow, p.ldk, vf);
        f32x4 sk[HD / 16] = {}, sv[HD / 16] = {};
        for (int q0 = max(0, k0 + 16 * r - p.coff) / kRows * kRows; q0 < p.Sq; q0 += kRows) {
            float x[2][4], y[2][4];
            wait_lds();
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int row = min(q0 + 16 * t + c, p.Sq - 1);
                load_row<T, HD, VEC>(qh, row, p.ldq, f);
                store_lds<T, HD>(region, 16 * t + c, f);
                const f32x4 s = dot<HD>(f, kf);
                load_row<T, HD, VEC>(dh, row, p.ldo, f);
                store_lds<T, HD>(region_d, 16 * t + c, f);
                const f32x4 dp = dot<HD>(f, vf);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int qi = min(q0 + 16 * t + 4 * g + i, p.Sq - 1);
                    x[t][i] = exp_of<T>(fmaf(s[i], p.scale, -lse_h[qi]));
                    y[t][i] = x[t][i] * (dp[i] - D_h[qi]);
                }
            }
            wait_lds();
            auto seen = [&](int row) { return q0 + row < p.Sq && key <= q0 + row + p.coff; };
            outer<T, HD>(region_d, x, seen, sv);
            outer<T, HD>(region, y, seen, sk);
        }
        if (key >= p.Sk || !((redo >> (16 * r + c)) & 1)) continue;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) {
            const f32x4 a = sk[dt] * p.scale, d = sv[dt];
            store4<VEC>(out_k + 16 * r * p.ld0 + 16 * dt, a[0], a[1], a[2], a[3]);
            store4<VEC>(out_v + 16 * r * p.ld1 + 16 * dt, d[0], d[1], d[2], d[3]);
        }
    }
}

// V: the copied vector type; n vectors per d columns.
template <typename V>
__global__ __launch_bounds__(256) void kv_append_k(const V* __restrict__ qkv, V* kc, V* vc, int64_t rows, int S, int n,
                                                   int64_t cache_rows, int64_t start) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= rows * 2 * n) return;
    const int64_t t = i / (2 * n);
    const int c = static_cast<int>(i % (2 * n));
    const int64_t row = t / S * cache_rows + start + t % S;
    (c < n ? kc : vc)[row * n + (c < n ? c : c - n)] = qkv[t * 3 * n + n + c];
}

enum Kind { kFwd, kDq, kDkDv };

bool rows16(const void* p, int64_t ld, size_t es) {
    return (reinterpret_cast<uintptr_t>(p) & 15u) == 0 && ld % static_cast<int64_t>(16 / es) == 0;
}

// Waves per block and waves per group for n groups of stationary rows over `blocks` streaming
// blocks.  1024 waves are one per SIMD; below that a group's streaming blocks are shared among
// its waves (as many as the block holds, and no more than there are streaming blocks).
void choose(int64_t groups, int64_t blocks, int max_waves, int& waves, int& split) {
    split = 1;
    while (split < max_waves && groups * split < 1024 && 2 * split <= blocks) split *= 2;
    waves = std::max(4, split);
}

// Blocks sharing the keys of one group of up to 16 queries: one per round of 8 waves x 32 keys, as
// far as the chip has a CU for each (16 x 12 heads, 2048 keys: two blocks each on fewer CUs 29 us,
// one 24).  The second launch pays from 2816 bytes of a head's columns per streaming lane up, which
// is 705 keys of 128 bytes or 353 of 256.  bf16, one query of 12 heads of 64: 768 keys 10.8 us in
// one block and 9.8 in parts, 1001 12.1 and 10.0, 2048 19.2 and 10.2; 16 heads of 128: 257 keys
// 10.2 and 11.2, 400 12.6 and 11.2, 2048 34.3 and 12.1; 4 x 16 heads, 2048 34.8 and 18.9.
int key_parts(int64_t groups, int64_t blocks, int64_t row_bytes) {
    if (blocks * row_bytes <= 2816) return 1;
    return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>({(blocks + 7) / 8, 256 / groups, 64})));
}

template <typename T, int HD, int RT, bool VEC, Kind K>
void launch(Args<T> p, hipStream_t s) {
    constexpr int TILES = K == kDkDv ? 2 : 1;
    constexpr int REGION = region_bytes<T, HD, RT, TILES, TILES>();
    constexpr int ALONE = region_bytes<T, HD, RT, TILES, 0>();  // no partial sums to exchange
    constexpr int max_waves = K == kFwd ? 8 : 4;
    static_assert(max_waves * REGION <= 160 * 1024, "LDS per block");
    const int64_t rows = K == kDkDv ? p.Sk : p.Sq, stream = K == kDkDv ? p.Sq : p.Sk;
    const int64_t per = (rows + 16 * RT - 1) / (16 * RT), nbh = static_cast<int64_t>(p.B) * p.H;
    int waves;
    choose(per * nbh, (stream + kRows - 1) / kRows, max_waves, waves, p.split);
    p.region = p.split > 1 ? REGION : ALONE;
    int64_t grid = (per + waves / p.split - 1) / (waves / p.split) * nbh;
    p.parts = 1;
    const StreamScratchUse use(s);
    if (K == kFwd && RT == 1 && per == 1 && p.split == max_waves) {
        p.parts = key_parts(nbh, (std::min<int64_t>(p.Sk, p.Sq + static_cast<int64_t>(p.coff)) + kRows - 1) / kRows,
                            static_cast<int64_t>(sizeof(T)) * HD);
        const size_t bytes = sizeof(float) * p.parts * nbh * p.Sq * (HD + 2);
        if (p.parts > 1 && !stream_scratch_ready(s)) p.parts = 1;
        if (p.parts > 1) p.part = static_cast<float*>(stream_scratch(bytes, s));
        grid *= p.parts;
    }
    AIC_CHECK(grid < (int64_t{1} << 31), InvalidArgument, "attention: too many query or key blocks");
    void (*kernel)(Args<T>) = nullptr;
    if constexpr (K == kFwd && RT == 1)
        kernel = p.parts > 1 ? attn_general_fwd<T, HD, 1, VEC, true> : attn_general_fwd<T, HD, 1, VEC, false>;
    else if constexpr (K == kFwd) kernel = attn_general_fwd<T, HD, RT, VEC, false>;
    else if constexpr (K == kDq) kernel = attn_general_dq<T, HD, RT, VEC>;
    else kernel = attn_general_dkdv<T, HD, RT, VEC>;
    static bool configured[2] = {};  // without and with parts
    if (!configured[p.parts > 1]) {
        AIC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, max_waves * REGION));
        configured[p.parts > 1] = true;
    }
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(64 * waves),
                       static_cast<size_t>(waves) * p.region, s, p);
    AIC_LAUNCH_CHECK("attn_general");
    if constexpr (K == kFwd && RT == 1) {
        if (p.parts > 1) {
            hipLaunchKernelGGL((attn_general_parts<T, HD>), dim3(static_cast<unsigned>(nbh * p.Sq)), dim3(64), 0, s, p);
            AIC_LAUNCH_CHECK("attn_general_parts");
        }
    }
}

// Tiles of stationary rows per wave: two share every streaming fragment where the registers
// allow (not fp32 heads of 128) and there are more than 16 rows.
template <typename T, int HD, Kind K>
void by_rows(const Args<T>& p, bool vec, hipStream_t s) {
    constexpr bool wide = sizeof(T) == 2 || HD <= 64;
    const int rows = K == kDkDv ? p.Sk : p.Sq;
    if (!vec) launch<T, HD, 1, false, K>(p, s);
    else if (wide && rows > 16) launch<T, HD, wide ? 2 : 1, true, K>(p, s);
    else launch<T, HD, 1, true, K>(p, s);
}

template <typename T, Kind K>
void by_head(const Args<T>& p, int64_t hd, bool vec, hipStream_t s) {
    if (hd == 16) by_rows<T, 16, K>(p, vec, s);
    else if (hd == 32) by_rows<T, 32, K>(p, vec, s);
    else if (hd == 64) by_rows<T, 64, K>(p, vec, s);
    else if (hd == 128) by_rows<T, 128, K>(p, vec, s);
    else AIC_THROW(NotImplemented, "attention: head_dim ", hd, " is not supported on this path");
}

template <typename T>
void fwd(const GenAttn& a, hipStream_t s) {
    Args<T> p{};
    p.q = static_cast<const T*>(a.q);
    p.k = static_cast<const T*>(a.k);
    p.v = static_cast<const T*>(a.v);
    p.out0 = static_cast<T*>(a.o_out);
    p.lse = a.lse_out;
    p.ldq = a.ldq; p.ldk = a.ldk; p.ld0 = a.ldo;
    p.qb = a.Sq; p.kb = a.kv_rows;
    p.B = static_cast<int>(a.B); p.H = static_cast<int>(a.H);
    p.Sq = static_cast<int>(a.Sq); p.Sk = static_cast<int>(a.Sk);
    p.coff = a.causal ? static_cast<int>(a.start) : 1 << 30;
    p.scale = a.scale;
    const bool vec = rows16(a.q, a.ldq, sizeof(T)) && rows16(a.k, a.ldk, sizeof(T)) && rows16(a.v, a.ldk, sizeof(T)) &&
                     rows16(a.o_out, a.ldo, sizeof(T));
    by_head<T, kFwd>(p, a.hd, vec, s);
}

template <typename T>
void bwd(const GenAttn& a, hipStream_t s) {
    Args<T> p{};
    p.q = static_cast<const T*>(a.q);
    p.k = static_cast<const T*>(a.k);
    p.v = static_cast<const T*>(a.v);
    p.o = static_cast<const T*>(a.o);
    p.dout = static_cast<const T*>(a.dout);
    p.lse = const_cast<float*>(a.lse);
    const StreamScratchUse use(s);
    // no queries: the key kernel's empty loop writes zero dK and dV
    p.D = static_cast<float*>(stream_scratch(sizeof(float) * std::max<int64_t>(a.B * a.H * a.Sq, 1), s));
    p.ldq = a.ldq; p.ldk = a.ldk; p.ldo = a.ldo;
    p.qb = a.Sq; p.kb = a.kv_rows;
    p.B = static_cast<int>(a.B); p.H = static_cast<int>(a.H);
    p.Sq = static_cast<int>(a.Sq); p.Sk = static_cast<int>(a.Sk);
    p.coff = a.causal ? static_cast<int>(a.start) : 1 << 30;
    p.scale = a.scale;
    const bool in = rows16(a.q, a.ldq, sizeof(T)) && rows16(a.k, a.ldk, sizeof(T)) && rows16(a.v, a.ldk, sizeof(T)) &&
                    rows16(a.o, a.ldo, sizeof(T)) && rows16(a.dout, a.ldo, sizeof(T));
    if (a.Sq > 0) {
        p.out0 = static_cast<T*>(a.dq);
        p.ld0 = a.ld_dq;
        by_head<T, kDq>(p, a.hd, in && rows16(a.dq, a.ld_dq, sizeof(T)), s);
    }
    p.out0 = static_cast<T*>(a.dk);
    p.out1 = static_cast<T*>(a.dv);
    p.ld0 = p.ld1 = a.ld_dkv;
    by_head<T, kDkDv>(p, a.hd, in && rows16(a.dk, a.ld_dkv, sizeof(T)) && rows16(a.dv, a.ld_dkv, sizeof(T)), s);
}

}  // namespace

void attn_general_forward(const GenAttn& a, DType dt, hipStream_t s) {
    if (dt == DType::Float32) fwd<float>(a, s);
    else if (dt == DType::BFloat16) fwd<bf16>(a, s);
    else AIC_THROW(DTypeMismatch, "attention: dtype must be f32 or bf16");
}

void attn_general_backward(const GenAttn& a, DType dt, hipStream_t s) {
    if (dt == DType::Float32) bwd<float>(a, s);
    else if (dt == DType::BFloat16) bwd<bf16>(a, s);
    else AIC_THROW(DTypeMismatch, "attention: dtype must be f32 or bf16");
}

void kv_append(const void* qkv, void* kc, void* vc, int64_t B, int64_t S, int64_t d, int64_t cache_rows,
               int64_t start_pos, DType dt, hipStream_t s) {
    const int64_t rows = B * S, bytes = d * static_cast<int64_t>(dtype_size(dt));
    if (rows == 0) return;
    auto run = [&](auto v) {
        using V = decltype(v);
        const int64_t n = bytes / static_cast<int64_t>(sizeof(V));
        const int64_t grid = (rows * 2 * n + 255) / 256;
        AIC_CHECK(grid < (int64_t{1} << 31) && S < (int64_t{1} << 31), InvalidArgument, "kv_append: too many tokens");
        hipLaunchKernelGGL(kv_append_k<V>, dim3(static_cast<unsigned>(grid)), dim3(256), 0, s, static_cast<const V*>(qkv),
                           static_cast<V*>(kc), static_cast<V*>(vc), rows, static_cast<int>(S), static_cast<int>(n),
                           cache_rows, start_pos);
        AIC_LAUNCH_CHECK("kv_append");
    };
    auto fits = [&](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    if (bytes % 16 == 0 && fits(qkv) && fits(kc) && fits(vc)) run(uint4{});
    else run(uint16_t{});
}

}  // namespace aic::hip
