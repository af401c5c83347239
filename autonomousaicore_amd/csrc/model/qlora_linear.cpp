#include "qlora_linear.hpp"

#include "../kernels/gemm.hpp"
#include "../kernels/kernels.hpp"
#include "../runtime/error.hpp"

namespace aic::models {

namespace {

void gemm(int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha, const void* A, int64_t lda, const void* B,
          int64_t ldb, float beta, void* C, int64_t ldc, DType ab, DType c, hipStream_t s, const void* R = nullptr,
          int64_t ldr = 0) {
    hip::GemmArgs a;
    a.transA = ta;
    a.transB = tb;
    a.M = M;
    a.N = N;
    a.K = K;
    a.alpha = alpha;
    a.A = A;
    a.lda = lda;
    a.B = B;
    a.ldb = ldb;
    a.beta = beta;
    a.C = C;
    a.ldc = ldc;
    a.R = R;
    a.ldr = ldr;
    a.ab = ab;
    a.c = c;
    hip::gemm(a, s);
}

// The product of `a` (its B operand the INT4 weight: transB and the sizes say which way round),
// dequantized inside the GEMM kernel where it takes the shape, else from a dequantized copy in a
// pool buffer (other shapes, fp32 operands).
void q4_product(hip::GemmArgs a, const uint8_t* Wq, const void* scales, DType scale_t, int64_t group, hipStream_t s) {
    a.ldb = a.transB ? a.K : a.N;
    hip::SkinnyArgs few;
    few.g = a;
    few.g.r2 = 0;  // a low-rank term that the kernels cannot take is added after them
    few.g.Bq = Wq;
    few.g.Bscale = scales;
    few.g.scale_t = scale_t;
    few.g.group = hip::int4_group(a.N * a.K, group);
    if (hip::gemm_q4_eligible(few.g) || hip::gemm_skinny_eligible(few)) {
        few.g.r2 = a.r2;
        hip::gemm(few.g, s);
        return;
    }
    DeviceBuffer w(dtype_size(a.ab) * static_cast<size_t>(a.N * a.K > 0 ? a.N * a.K : 1), s);
    hip::int4_dequant(Wq, scales, scale_t, a.N * a.K, group, w.get(), a.ab, s);
    a.B = w.get();
    hip::gemm(a, s);
}

void check_dt(DType ab, DType c, DType scale_t) {
    AIC_CHECK(ab == DType::Float32 || ab == DType::BFloat16, DTypeMismatch, "int4 GEMM: operands must be f32 or bf16");
    AIC_CHECK(c == DType::Float32 || c == DType::BFloat16, DTypeMismatch, "int4 GEMM: output must be f32 or bf16");
    AIC_CHECK(scale_t == DType::Float32 || scale_t == DType::Float16, DTypeMismatch, "int4: scales must be f32 or f16");
}

}  // namespace

void int4_dequant_gemm(int transW, int64_t M, int64_t N, int64_t K, float alpha, const void* X, int64_t ldx,
                       const uint8_t* Wq, const void* scales, DType scale_t, int64_t group, float beta, void* C,
                       int64_t ldc, const void* R, int64_t ldr, DType ab, DType c, hipStream_t s) {
    check_dt(ab, c, scale_t);
    AIC_CHECK(M >= 0 && N >= 0 && K >= 0, InvalidArgument, "int4_dequant_gemm: negative size");
    if (M == 0 || N == 0) return;
    AIC_CHECK(X && Wq && scales && C, InvalidArgument, "int4_dequant_gemm: null pointer");
    hip::GemmArgs a;
    a.transB = transW ? 1 : 0;
    a.M = M;
    a.N = N;
    a.K = K;
    a.alpha = alpha;
    a.A = X;
    a.lda = ldx;
    a.beta = beta;
    a.C = C;
    a.ldc = ldc;
    a.R = R;
    a.ldr = ldr;
    a.ab = ab;
    a.c = c;
    q4_product(a, Wq, scales, scale_t, group, s);
}

QLoRALinear::QLoRALinear(int64_t in, int64_t out, int64_t rank, float alpha, int64_t group, DType scale_t, DType dt)
    : in_(in), out_(out), rank_(rank), group_(group), alpha_(alpha), scale_t_(scale_t), dt_(dt) {
    AIC_CHECK(in > 0 && out > 0 && rank >= 0, InvalidArgument, "QLoRALinear: need in, out > 0 and rank >= 0");
    check_dt(dt, dt, scale_t);
    hip::int4_group(in * out, group);  // rejects an odd multi-group size now
}

void QLoRALinear::forward(const void* x, int64_t T, const uint8_t* Wq, const void* scales, const void* A,
                          const void* B, const void* R, void* y, hipStream_t s) {
    AIC_CHECK(x && Wq && scales && y && T > 0, InvalidArgument, "QLoRALinear::forward: bad arguments");
    AIC_CHECK(rank_ == 0 || (A && B), InvalidArgument, "QLoRALinear::forward: null adapter");
    const size_t es = dtype_size(dt_);
    T_ = T;
    x_ = x;
    A_ = A;
    B_ = B;
    Wq_ = Wq;
    scales_ = scales;
    hip::GemmArgs a;
    a.transB = 1;
    a.M = T;
    a.N = out_;
    a.K = in_;
    a.A = x;
    a.lda = in_;
    a.C = y;
    a.ldc = out_;
    a.R = R;
    a.ldr = out_;
    a.ab = a.c = dt_;
    if (rank_ > 0) {
        // s x A^T in one pass over x, then one product: the base plus the low-rank term in its
        // accumulators (2048 -> 5632, rank 16, 8192 tokens: 11 + 224 us; as a K = 16 product into y
        // and the base added to it 79 + 221 + 18 us)
        xs_ = DeviceBuffer(es * static_cast<size_t>(T * rank_), s);
        hip::LoraSkinny q;
        q.Y = x;
        q.ldy = in_;
        q.T = T;
        q.N = q.n_seg = in_;
        q.r_seg = rank_;
        q.W = A;
        q.w_n = 1;
        q.w_j = in_;
        q.out1 = xs_.get();
        q.ldo1 = rank_;
        q.scale = scaling();
        if (one_pass(q)) hip::lora_skinny(q, s);
        else gemm(0, 1, T, rank_, in_, scaling(), x, in_, A, in_, 0.0f, xs_.get(), rank_, dt_, dt_, s);
        a.X2 = xs_.get();
        a.ldx2 = rank_;
        a.Y2 = B;
        a.ldy2 = rank_;
        a.r2 = rank_;
    }
    q4_product(a, Wq, scales, scale_t_, group_, s);  // x deq(Wq)^T + s (x A^T) B^T (+ R)
}

// The one-pass kernels (bf16) from the token counts up at which a tile product of rank_ columns
// would be mostly padding read by few blocks.
bool QLoRALinear::one_pass(const hip::LoraSkinny& q) const {
    return dt_ == DType::BFloat16 && T_ > hip::kSkinnyRows && hip::lora_skinny_ok(q);
}

void QLoRALinear::backward(const void* dy, void* dx, float* dA, float* dB, bool accumulate, hipStream_t s) {
    AIC_CHECK(dy && T_ > 0 && Wq_, InvalidArgument, "QLoRALinear::backward: no forward to differentiate");
    AIC_CHECK(rank_ == 0 || (dA && dB), InvalidArgument, "QLoRALinear::backward: null adapter gradient");
    const float acc = accumulate ? 1.0f : 0.0f;
    DeviceBuffer dxa;
    hip::GemmArgs a;
    a.transB = 0;
    a.M = T_;
    a.N = in_;
    a.K = out_;
    a.A = dy;
    a.lda = out_;
    a.C = dx;
    a.ldc = in_;
    a.ab = a.c = dt_;
    if (rank_ > 0) {
        dxa = DeviceBuffer(dtype_size(dt_) * static_cast<size_t>(T_ * rank_), s);
        hip::LoraSkinny q;  // s dy B and dy^T xs from one pass over dy
        q.Y = dy;
        q.ldy = out_;
        q.T = T_;
        q.N = q.n_seg = out_;
        q.r_seg = rank_;
        q.W = B_;
        q.w_n = rank_;
        q.w_j = 1;
        q.out1 = dxa.get();
        q.ldo1 = rank_;
        q.scale = scaling();
        q.Z = xs_.get();
        q.ldz = rank_;
        q.out2 = dB;
        q.o2n = rank_;
        q.o2j = 1;
        q.accumulate = accumulate;
        if (one_pass(q)) {
            hip::lora_skinny(q, s);
        } else {
            gemm(0, 0, T_, rank_, out_, scaling(), dy, out_, B_, rank_, 0.0f, dxa.get(), rank_, dt_, dt_, s);
            gemm(1, 0, out_, rank_, T_, 1.0f, dy, out_, xs_.get(), rank_, acc, dB, rank_, dt_, DType::Float32, s);
        }
        hip::LoraSkinny r;  // dxa^T x
        r.Y = x_;
        r.ldy = in_;
        r.T = T_;
        r.N = r.n_seg = in_;
        r.r_seg = rank_;
        r.Z = dxa.get();
        r.ldz = rank_;
        r.out2 = dA;
        r.o2n = 1;
        r.o2j = in_;
        r.accumulate = accumulate;
        if (one_pass(r)) hip::lora_skinny(r, s);
        else gemm(1, 0, rank_, in_, T_, 1.0f, dxa.get(), rank_, x_, in_, acc, dA, in_, dt_, DType::Float32, s);
        a.X2 = dxa.get();
        a.ldx2 = rank_;
        a.Y2 = A_;
        a.ldy2 = in_;
        a.r2 = rank_;
        a.y2_kmajor = 1;
    }
    if (dx) q4_product(a, Wq_, scales_, scale_t_, group_, s);  // dy deq(Wq) + dxa A
}

}  // namespace aic::models
