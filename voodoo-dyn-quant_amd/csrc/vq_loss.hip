// Fused distillation loss over full logits: token cross-entropy against the
// labels plus KL(teacher || student) of the temperature-softened
// distributions, and its gradient with respect to the student logits
// (reference training/trainer.py:2566-2575: F.cross_entropy, F.log_softmax,
// F.softmax and F.kl_div over [tokens, vocab] logits, then autograd).
//
// Forward: one workgroup per token row streams the student and teacher rows
// once (16-byte loads, the next ones in flight while these are summed) and keeps per-lane online log-sum-exps of s, s/T and
// t/T, plus A = sum exp(t/T - m_t) (t - s), so that
//   CE_r = lse(s) - s[y_r]
//   KL_r = T^2 (A / Z_t / T - lse(t/T) + lse(s/T))     (= T^2 sum p (log p - log q))
// and stores the three log-sum-exps of the row for the backward.  A fixed-
// order fp64 reduction gives the means (labels equal to -100 are ignored by
// the cross-entropy, as F.cross_entropy's default ignore_index).
// Backward: one more pass writes
//   dS = g_ce / N_ce (softmax(s) - onehot(y)) + g_kl T / N (softmax(s/T) - softmax(t/T)).
// At T = 1 (the trainer's default) s/T is s, and at T = 2 e^s is the square of
// e^(s/2): both passes then take one exponential of s per logit instead of two
// (LossT).  The forward at other T is bound by its three exponentials and about
// twenty more VALU operations per logit, not by memory.
#include <cfloat>
#include <type_traits>

#include "vq_internal.h"

namespace vq {

namespace {

// Threads per row: few rows leave CUs idle, so each takes a larger workgroup
// there (MI355X, 64 x 151936, T = 2: forward 37 -> 30 us, backward 37 -> 26 us;
// before, without the loads ahead, 55 and 52 us).  At 400 x 32000 a thread would
// have four loads left to sum, and the larger workgroup's reduction loses:
// forward 20 -> 22 us.
constexpr int kLossThreads = 256, kLossFewThreads = 1024, kLossFewRows = 512, kLossFewVocab = 1 << 16;
// Logits past this size do not stay in the last-level cache (256 MiB, shared by
// both models' logits and the gradient) from one pass to the next: they are then
// streamed past it.  2048 x 151936: forward 226 -> 199 us, backward 380 -> 357 us
// (the loads of the next 8 logits ahead of the sums included); 1000 x 32000,
// which fits, 32 -> 35 us for a streamed backward.
constexpr int64_t kLossStreamBytes = (int64_t)128 << 20;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// e^x through the hardware base-2 exponential, v_exp_f32 alone: results
// below 2^-126 flush to zero (exp2f would rescale its input around them, four
// more instructions per exponential).  Such terms sit more than 87 nats below
// the row maximum's, whose term is 1 in every sum, and the gradient elements
// they would give are below 2^-126 times the loss weights.
__device__ __forceinline__ float fexp(float x) { return __builtin_amdgcn_exp2f(x * kLog2e); }

template <bool STREAM>
__device__ __forceinline__ u32x4 load_logits(const bf16_t* p) {
    const u32x4* q = reinterpret_cast<const u32x4*>(p);
    return STREAM ? __builtin_nontemporal_load(q) : *q;
}

__device__ __forceinline__ void unpack8(const u32x4& w, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}

// How the exponentials of s and of s / T go together: apart, as one (T = 1),
// or e^s as the square of e^(s / 2) (T = 2).
enum LossT : int { ANY_T = 0, UNIT_T = 1, TWO_T = 2 };

// (m, z): z = sum exp(x - m).  Merge b into a.
__device__ __forceinline__ void lse_merge(float& ma, float& za, float mb, float zb) {
    const float m = fmaxf(ma, mb);
    za = za * fexp(ma - m) + zb * fexp(mb - m);
    ma = m;
}

struct RowAcc {
    float ms, zs;      // s
    float mq, zq;      // s / T
    float mt, zt, at;  // t / T, and sum exp(t/T - mt) (t - s)
};

__device__ __forceinline__ void acc_merge(RowAcc& a, const RowAcc& b) {
    lse_merge(a.ms, a.zs, b.ms, b.zs);
    lse_merge(a.mq, a.zq, b.mq, b.zq);
    const float m = fmaxf(a.mt, b.mt);
    const float fa = fexp(a.mt - m), fb = fexp(b.mt - m);
    a.zt = a.zt * fa + b.zt * fb;
    a.at = a.at * fa + b.at * fb;
    a.mt = m;
}

__device__ __forceinline__ RowAcc shfl_acc(const RowAcc& a, int lane) {
    RowAcc b;
    b.ms = __shfl(a.ms, lane, 64);
    b.zs = __shfl(a.zs, lane, 64);
    b.mq = __shfl(a.mq, lane, 64);
    b.zq = __shfl(a.zq, lane, 64);
    b.mt = __shfl(a.mt, lane, 64);
    b.zt = __shfl(a.zt, lane, 64);
    b.at = __shfl(a.at, lane, 64);
    return b;
}

}  // namespace

// Running sums over 8 more logits of each model.
template <LossT LT>
__device__ __forceinline__ void loss_accumulate(RowAcc& a, const float (&sv)[8], const float (&tv)[8], float inv_tau) {
    float cs = sv[0], ct = tv[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) {
        cs = fmaxf(cs, sv[j]);
        ct = fmaxf(ct, tv[j]);
    }
    // rescale the running sums once per 8 values
    const float nt = fmaxf(a.mt, LT == UNIT_T ? ct : ct * inv_tau);
    const float ft = fexp(a.mt - nt);
    a.zt *= ft;
    a.at *= ft;
    a.mt = nt;
    if constexpr (LT != TWO_T) {
        const float ns = fmaxf(a.ms, cs);
        a.zs *= fexp(a.ms - ns);
        a.ms = ns;
    }
    if constexpr (LT != UNIT_T) {
        const float nq = fmaxf(a.mq, cs * inv_tau);
        const float fq = fexp(a.mq - nq);
        a.zq *= fq;
        if constexpr (LT == TWO_T) a.zs *= fq * fq;
        a.mq = nq;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        if constexpr (LT != TWO_T) a.zs += fexp(sv[j] - a.ms);
        if constexpr (LT != UNIT_T) {
            const float eq = fexp(sv[j] * inv_tau - a.mq);
            a.zq += eq;
            if constexpr (LT == TWO_T) a.zs = fmaf(eq, eq, a.zs);
        }
        const float e = fexp((LT == UNIT_T ? tv[j] : tv[j] * inv_tau) - nt);
        a.zt += e;
        a.at += e > 0.f ? e * (tv[j] - sv[j]) : 0.f;
    }
}

template <LossT LT, bool STREAM, int THREADS>
__global__ __launch_bounds__(THREADS) void distill_fwd_kernel(const bf16_t* __restrict__ S,
                                                                   const bf16_t* __restrict__ Tl,
                                                                   const int64_t* __restrict__ labels, int64_t V,
                                                                   float inv_tau, float tau2,
                                                                   float* __restrict__ stats,
                                                                   float* __restrict__ row_loss) {
    __shared__ RowAcc part[THREADS / 64];
    const int64_t r = blockIdx.x;
    const bf16_t* s = S + r * V;
    const bf16_t* t = Tl + r * V;
    RowAcc a{-FLT_MAX, 0.f, -FLT_MAX, 0.f, -FLT_MAX, 0.f, 0.f};
    // the next 8 logits of each are in flight while these are summed
    const int64_t step = THREADS * 8;
    int64_t i = (int64_t)threadIdx.x * 8;
    u32x4 qs, qt;
    if (i < V) {
        qs = load_logits<STREAM>(s + i);
        qt = load_logits<STREAM>(t + i);
    }
    for (; i < V; i += step) {
        float sv[8], tv[8];
        unpack8(qs, sv);
        unpack8(qt, tv);
        if (i + step < V) {
            qs = load_logits<STREAM>(s + i + step);
            qt = load_logits<STREAM>(t + i + step);
        }
        loss_accumulate<LT>(a, sv, tv, inv_tau);
    }
    if constexpr (LT == TWO_T) a.ms = fmaxf(2.0f * a.mq, -FLT_MAX);  // a thread without logits: not -inf
    if constexpr (LT == UNIT_T) {
        a.mq = a.ms;
        a.zq = a.zs;
    }
    // wave then workgroup reduction (fixed order)
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const RowAcc b = shfl_acc(a, (int)(threadIdx.x ^ off) & 63);
        acc_merge(a, b);
    }
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = a;
    __syncthreads();
    if (threadIdx.x == 0) {
        RowAcc w = part[0];
#pragma unroll
        for (int k = 1; k < THREADS / 64; ++k) acc_merge(w, part[k]);
        const float lse_s = w.ms + __log2f(w.zs) * kLn2;
        const float lse_q = w.mq + __log2f(w.zq) * kLn2;
        const float lse_t = w.mt + __log2f(w.zt) * kLn2;
        const int64_t y = labels[r];
        float ce = 0.f;
        if (y != -100) ce = (y >= 0 && y < V) ? lse_s - __uint_as_float((uint32_t)s[y] << 16) : __int_as_float(0x7fc00000);
        const float kl = tau2 * (w.at / w.zt * inv_tau - lse_t + lse_q);
        stats[3 * r] = lse_s;
        stats[3 * r + 1] = lse_q;
        stats[3 * r + 2] = lse_t;
        row_loss[2 * r] = ce;
        row_loss[2 * r + 1] = kl;
    }
}

// out = {CE mean over labelled rows, KL mean over all rows}; aux = {1/N_ce, 1/N}
__global__ __launch_bounds__(256) void distill_reduce_kernel(const float* __restrict__ row_loss,
                                                             const int64_t* __restrict__ labels, int64_t rows,
                                                             float* __restrict__ out, float* __restrict__ aux) {
    __shared__ double sh[3][256];
    double ce = 0.0, kl = 0.0, n = 0.0;
    for (int64_t r = threadIdx.x; r < rows; r += 256) {
        ce += (double)row_loss[2 * r];
        kl += (double)row_loss[2 * r + 1];
        n += labels[r] != -100 ? 1.0 : 0.0;
    }
    sh[0][threadIdx.x] = ce;
    sh[1][threadIdx.x] = kl;
    sh[2][threadIdx.x] = n;
    __syncthreads();
    for (int w = 128; w >= 1; w >>= 1) {
        if ((int)threadIdx.x < w) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + w];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + w];
            sh[2][threadIdx.x] += sh[2][threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = (float)(sh[0][0] / sh[2][0]);  // 0/0 = NaN with no labelled row, as torch's mean
        out[1] = (float)(sh[1][0] / (double)rows);
        aux[0] = (float)(1.0 / sh[2][0]);
        aux[1] = (float)(1.0 / (double)rows);
    }
}

template <LossT LT, bool STREAM, int THREADS>
__global__ __launch_bounds__(THREADS) void distill_bwd_kernel(const bf16_t* __restrict__ S,
                                                                   const bf16_t* __restrict__ Tl,
                                                                   const int64_t* __restrict__ labels, int64_t V,
                                                                   float inv_tau, float tau,
                                                                   const float* __restrict__ stats,
                                                                   const float* __restrict__ aux,
                                                                   const float* __restrict__ grad_out,
                                                                   bf16_t* __restrict__ dS) {
    const int64_t r = blockIdx.x;
    const bf16_t* s = S + r * V;
    const bf16_t* t = Tl + r * V;
    bf16_t* d = dS + r * V;
    const float lse_s = stats[3 * r], lse_q = stats[3 * r + 1], lse_t = stats[3 * r + 2];
    const int64_t y = labels[r];
    const float a = y != -100 ? grad_out[0] * aux[0] : 0.f;  // dL/dCE_mean / N_ce
    const float b = grad_out[1] * tau * aux[1];              // dL/dKL_mean * T^2 / T / N
    // T = 2: softmax(s) = softmax(s/2)^2 e^(2 lse_q - lse_s)
    const float square = LT == TWO_T ? fexp(2.0f * lse_q - lse_s) : 0.f;
    const int64_t step = THREADS * 8;
    int64_t i = (int64_t)threadIdx.x * 8;
    u32x4 qs, qt;
    if (i < V) {
        qs = load_logits<STREAM>(s + i);
        qt = load_logits<STREAM>(t + i);
    }
    for (; i < V; i += step) {
        float sv[8], tv[8], g[8];
        unpack8(qs, sv);
        unpack8(qt, tv);
        if (i + step < V) {
            qs = load_logits<STREAM>(s + i + step);
            qt = load_logits<STREAM>(t + i + step);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float eq = LT == UNIT_T ? 0.f : fexp(sv[j] * inv_tau - lse_q);
            const float es = LT == TWO_T ? eq * eq * square : fexp(sv[j] - lse_s);
            const float ps = es - ((i + j) == y ? 1.f : 0.f);
            const float dq = LT == UNIT_T ? es - fexp(tv[j] - lse_t) : eq - fexp(tv[j] * inv_tau - lse_t);
            g[j] = a * ps + b * dq;
        }
        u32x4 q;
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = f2bf2(g[2 * j], g[2 * j + 1]);
        if constexpr (STREAM)
            __builtin_nontemporal_store(q, reinterpret_cast<u32x4*>(d + i));
        else
            *reinterpret_cast<u32x4*>(d + i) = q;
    }
}

// The instantiation of a pass for these sizes and this temperature.
template <class Launch>
static void loss_dispatch(int64_t rows, int64_t V, float temperature, Launch launch) {
    auto with_threads = [&](auto lt, auto stream) {
        if (rows < kLossFewRows && V >= kLossFewVocab)
            launch(lt, stream, std::integral_constant<int, kLossFewThreads>{});
        else
            launch(lt, stream, std::integral_constant<int, kLossThreads>{});
    };
    auto with_stream = [&](auto lt) {
        if (2 * rows * V >= kLossStreamBytes)
            with_threads(lt, std::true_type{});
        else
            with_threads(lt, std::false_type{});
    };
    if (temperature == 1.0f)
        with_stream(std::integral_constant<LossT, UNIT_T>{});
    else if (temperature == 2.0f)
        with_stream(std::integral_constant<LossT, TWO_T>{});
    else
        with_stream(std::integral_constant<LossT, ANY_T>{});
}

hipError_t launch_distill_fwd(const bf16_t* S, const bf16_t* T, const int64_t* labels, int64_t rows, int64_t V,
                              float temperature, float* out, float* ws, hipStream_t s) {
    float* stats = ws;
    float* row_loss = ws + 3 * rows;
    float* aux = ws + 5 * rows;
    loss_dispatch(rows, V, temperature, [&](auto lt, auto stream, auto threads) {
        distill_fwd_kernel<decltype(lt)::value, decltype(stream)::value, decltype(threads)::value>
            <<<dim3((unsigned)rows), decltype(threads)::value, 0, s>>>(S, T, labels, V, 1.0f / temperature,
                                                                       temperature * temperature, stats, row_loss);
    });
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    distill_reduce_kernel<<<1, 256, 0, s>>>(row_loss, labels, rows, out, aux);
    return hipGetLastError();
}

hipError_t launch_distill_bwd(const bf16_t* S, const bf16_t* T, const int64_t* labels, int64_t rows, int64_t V,
                              float temperature, const float* grad_out, bf16_t* dS, const float* ws, hipStream_t s) {
    loss_dispatch(rows, V, temperature, [&](auto lt, auto stream, auto threads) {
        distill_bwd_kernel<decltype(lt)::value, decltype(stream)::value, decltype(threads)::value>
            <<<dim3((unsigned)rows), decltype(threads)::value, 0, s>>>(S, T, labels, V, 1.0f / temperature, temperature,
                                                                       ws, ws + 5 * rows, grad_out, dS);
    });
    return hipGetLastError();
}

}  // namespace vq
