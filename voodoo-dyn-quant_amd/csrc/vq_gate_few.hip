// Gate gradient of at most kFewGateTokens tokens:
//   partials[block][k] = sum over the block's weights of dW[n][d] * W_k[n][d],
//   dW[n][d] = sum_m dY[m][n] X[m][d].
// With so few tokens the product is a few MFMAs per 1024 weights and the time
// is the candidates': their packed bytes and their decode.  A small tensor has
// too few 256 x 256 tiles to fill the chip (16 at 1024 x 1024); here a workgroup
// takes 16 weight rows of one 256-weight group at a time, six of them share a
// CU, and one's copies run beside another's decode.
//
// A wave forms dW^T for 64 columns x 16 rows by 16x16x32 MFMAs: A holds
// columns of X, B rows of dY^T, both from token-contiguous copies
// (transpose_tokens_kernel) so a lane's 8 tokens are one 16-byte load.  The
// columns are dealt to A's rows so that four MFMAs leave each lane 16
// consecutive weights of one row, the run the decoders read under one scale.
#include "vq_internal.h"

namespace vq {

namespace {

constexpr int kRows = 16;  // weight rows per step

// 16-byte chunks that hold any span of gb bytes, whatever its start mod 16; an
// odd count, so the 16 rows of a step fall on distinct bank groups.
__host__ __device__ constexpr int span_chunks(int gb) { return ((gb + 15 + 15) / 16) | 1; }

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct GateFewPlan {
    CandSet cs;
    const bf16_t* xt;   // [G * 256][MT]
    const bf16_t* dyt;  // [16 * row blocks][MT]
    float* partials;    // [grid][ncand]
    int N, D, G, splits, per;  // per: row blocks of a split
    int chunks[kMaxCand], lds_off[kMaxCand], red_off;
    uint32_t inv[kMaxCand];  // floor(L / chunks) = (L * inv) >> 16 for L < 16 chunks
};

}  // namespace

// out[c][0 .. MT) = in[0 .. M)[c], zeros past the M tokens and the C columns.
// Blocks [0, bx) take X's columns, the rest dY's; 64 columns each.
template <int MT>
__global__ __launch_bounds__(256) void transpose_tokens_kernel(const bf16_t* __restrict__ x, int D,
                                                               const bf16_t* __restrict__ dy, int N, int M, int bx,
                                                               bf16_t* __restrict__ xt, bf16_t* __restrict__ dyt,
                                                               int xrows, int yrows) {
    __shared__ __attribute__((aligned(16))) bf16_t tile[64][MT + 8];
    const bool isx = (int)blockIdx.x < bx;
    const bf16_t* in = isx ? x : dy;
    bf16_t* out = isx ? xt : dyt;
    const int C = isx ? D : N, rows = isx ? xrows : yrows;
    const int c0 = 64 * ((int)blockIdx.x - (isx ? 0 : bx));
    const int t = threadIdx.x, cc = 8 * (t & 7);
#pragma unroll
    for (int m0 = 0; m0 < MT; m0 += 32) {
        const int m = m0 + (t >> 3);
        uint4 v = make_uint4(0, 0, 0, 0);
        if (m < M && c0 + cc < C) v = *reinterpret_cast<const uint4*>(in + (int64_t)m * C + c0 + cc);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) tile[cc + e][m] = (bf16_t)(w[e >> 1] >> (16 * (e & 1)));
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 64 * MT / 8; i += 256) {
        const int row = (i + t) / (MT / 8), part = (i + t) % (MT / 8);
        if (c0 + row < rows)
            *reinterpret_cast<uint4*>(out + (int64_t)(c0 + row) * MT + 8 * part) =
                *reinterpret_cast<const uint4*>(&tile[row][8 * part]);
    }
}

template <bool IQ, int KS>
__global__ __launch_bounds__(kStreamThreads) void gate_few_kernel(GateFewPlan gp) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    float(*red)[kStreamThreads] = reinterpret_cast<float(*)[kStreamThreads]>(lds + gp.red_off);  // [ncand]
    typedef __attribute__((address_space(3))) void lds_void;
    constexpr int MT = 32 * KS;
    const CandSet& cs = gp.cs;
    const int t = threadIdx.x, lane = t & 63, h = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    for (int k = 0; k < cs.ncand; ++k) red[k][t] = 0.0f;
    // neighbouring groups of the same rows run on one XCD: their spans share cache lines
    const int per_xcd = (int)gridDim.x / 8;
    const int idx = ((int)blockIdx.x % 8) * per_xcd + (int)blockIdx.x / 8;
    const int split = idx / gp.G, grp = idx - split * gp.G;
    const int blocks = (gp.N + kRows - 1) / kRows;
    const int b0 = split < gp.splits ? split * gp.per : blocks, b1 = min(blocks, b0 + gp.per);
    const int p = 64 * wave + 16 * h;  // this lane's 16 weights within the group
    const bool live = 256 * grp + p < gp.D;
    // A: row i of MFMA q is column 16 (i / 4) + 4 q + i % 4 of the wave's 64
    bf16x8 a[4][KS];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int i = lane & 15;
        const int64_t col = 256 * (int64_t)grp + 64 * wave + 16 * (i >> 2) + 4 * q + (i & 3);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            a[q][ks] = *reinterpret_cast<const bf16x8*>(gp.xt + col * MT + 32 * ks + 8 * h);
    }
    for (int nb = b0; nb < b1; ++nb) {
        const int n = kRows * nb + (lane & 15);
        bf16x8 b[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            b[ks] = *reinterpret_cast<const bf16x8*>(gp.dyt + (int64_t)n * MT + 32 * ks + 8 * h);
        // the 16 rows' spans of every candidate, each from its 16-byte
        // boundary; bytes past the buffer's end (rounded up to the 4 the
        // bounds check works in) come as zeros
        const int64_t g0 = (int64_t)kRows * nb * cs.row_groups + grp;
        for (int k = 0; k < cs.ncand; ++k) {
            const int gb = group_bytes(cs.qtype[k]), nch = gp.chunks[k];
            const int64_t off0 = g0 * gb, base = off0 & ~int64_t(15);
            const int64_t left = (((int64_t)gp.N * cs.row_groups * gb + 3) & ~int64_t(3)) - base;
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint8_t*>(cs.qbytes[k] + base), (short)0, (int)min<int64_t>(left, 0x7fffffff), 0x00020000);
            const int pitch = (int)cs.row_groups * gb, head0 = (int)(off0 - base);
            for (int l0 = 64 * wave; l0 < kRows * nch; l0 += kStreamThreads) {
                const int l = l0 + lane;
                const int row = (int)(((uint32_t)l * gp.inv[k]) >> 16);
                const int at = ((head0 + row * pitch) & ~15) + 16 * (l - row * nch);
                if (l < kRows * nch)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(lds + gp.lds_off[k] + 16 * l0), 16, at, 0,
                                                             0, 0);
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        float v[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q][ks], b[ks], c, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[4 * q + r] = c[r];
        }
        float sv = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) sv += v[r];
        const uint32_t gi = (uint32_t)n * (uint32_t)cs.row_groups + (uint32_t)grp;  // its low bits count
        for (int k = 0; k < cs.ncand; ++k) {
            const int qt = cs.qtype[k], gb = group_bytes(qt);
            const uint8_t* g =
                lds + gp.lds_off[k] + (lane & 15) * 16 * gp.chunks[k] + (int)((gi * (uint32_t)gb) & 15u);
            float dot;
            switch (qt) {
            case Q8_0: dot = dot_sub16<Q8_0>(g, p, v, sv); break;
            case Q2_K: dot = dot_sub16<Q2_K>(g, p, v, sv); break;
            case Q3_K: dot = dot_sub16<Q3_K>(g, p, v, sv); break;
            case Q4_K: dot = dot_sub16<Q4_K>(g, p, v, sv); break;
            case Q5_K: dot = dot_sub16<Q5_K>(g, p, v, sv); break;
            case Q6_K: dot = dot_sub16<Q6_K>(g, p, v, sv); break;
            default:
                if constexpr (IQ)
                    dot = dot_sub16_iq(qt, g, p, v, sv);
                else
                    dot = dot_sub16<Q6_K>(g, p, v, sv);
                break;
            }
            // weights past D or N have no gradient, whatever their bytes hold
            if (live && n < gp.N) red[k][t] += dot;
        }
        __syncthreads();  // the next step's copies reuse the spans' LDS
    }
    // each wave sums its share of the candidates over the workgroup, in order
    for (int k = wave; k < cs.ncand; k += kStreamThreads / 64) {
        float s = (red[k][lane] + red[k][64 + lane]) + (red[k][128 + lane] + red[k][192 + lane]);
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
        if (lane == 0) gp.partials[(int64_t)blockIdx.x * cs.ncand + k] = s;
    }
}

namespace {

int few_mt(int64_t M) { return M <= 32 ? 32 : 64; }

// Row blocks are dealt so that about six workgroups per CU run: one round.
void gate_few_split(int64_t N, int64_t D, int& G, int& splits, int& per, int& grid) {
    G = (int)((D + 255) / 256);
    const int blocks = (int)((N + kRows - 1) / kRows);
    const int want = (6 * device_cus() + G - 1) / G;
    per = (blocks + want - 1) / want;
    splits = (blocks + per - 1) / per;
    grid = (G * splits + 7) / 8 * 8;
}

}  // namespace

// Taken for a gate product by itself (the fused few-token backward).  Measured
// on MI355X, K = 6, 1 / 64 tokens, with its reduction, against eight-wave
// tiles: 1024 x 1024 12.9 / 13.3 against 31.5 us, 1032 x 2056 15.4 / 17.8
// against 31.5, 4096 x 2048 25.8 / 28.9 against 33; K = 8 with code books
// 15.8 / 16.3 against 48 at 1024 x 1024; at 6144 x 5120 77.6 / 83 against 69,
// for the tiles fill the chip there and copy each span's chunks once.  With dX
// beside it the tiles' one launch is the faster one at every size.
bool gate_few(int64_t M, int64_t N, int64_t D) {
    return M >= 1 && M <= kFewGateTokens && N * D <= ((int64_t)1 << 23);
}

int64_t gate_few_blocks(int64_t N, int64_t D) {
    int G, splits, per, grid;
    gate_few_split(N, D, G, splits, per, grid);
    return grid;
}

int64_t gate_few_bytes(int64_t M, int64_t N, int64_t D) {
    if (!gate_few(M, N, D)) return 0;
    return ((D + 255) / 256 * 256 + (N + kRows - 1) / kRows * kRows) * few_mt(M) * 2;
}

template <bool IQ>
static hipError_t launch_gate_few_t(const GateFewPlan& gp, int ks, int grid, size_t lds, hipStream_t s) {
    const void* kern = ks == 1 ? (const void*)gate_few_kernel<IQ, 1> : (const void*)gate_few_kernel<IQ, 2>;
    const hipError_t e = allow_dynamic_lds(kern, lds);  // 16 Q8_0 candidates: 92 KiB
    if (e != hipSuccess) return e;
    if (ks == 1)
        gate_few_kernel<IQ, 1><<<grid, kStreamThreads, lds, s>>>(gp);
    else
        gate_few_kernel<IQ, 2><<<grid, kStreamThreads, lds, s>>>(gp);
    return hipGetLastError();
}

hipError_t launch_gate_few(const bf16_t* dY, const bf16_t* X, const CandSet& cs, float* partials, int M, int N, int D,
                           void* ws, hipStream_t s) {
    if (!gate_few(M, N, D) || !ws || D % 8 != 0 || N % 8 != 0 || (int64_t)(D + 255) / 256 > cs.row_groups)
        return hipErrorInvalidValue;
    const int mt = few_mt(M), ks = mt / 32;
    GateFewPlan gp{};
    int grid;
    gate_few_split(N, D, gp.G, gp.splits, gp.per, grid);
    const int xrows = 256 * gp.G, yrows = (N + kRows - 1) / kRows * kRows;
    bf16_t* xt = static_cast<bf16_t*>(ws);
    bf16_t* dyt = xt + (int64_t)xrows * mt;
    const int bx = xrows / 64, by = (yrows + 63) / 64;
    if (ks == 1)
        transpose_tokens_kernel<32><<<bx + by, 256, 0, s>>>(X, D, dY, N, M, bx, xt, dyt, xrows, yrows);
    else
        transpose_tokens_kernel<64><<<bx + by, 256, 0, s>>>(X, D, dY, N, M, bx, xt, dyt, xrows, yrows);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    gp.cs = cs;
    gp.xt = xt;
    gp.dyt = dyt;
    gp.partials = partials;
    gp.N = N;
    gp.D = D;
    size_t lds = 0;
    for (int k = 0; k < cs.ncand; ++k) {
        gp.chunks[k] = span_chunks(group_bytes(cs.qtype[k]));
        gp.inv[k] = (uint32_t)(65536 / gp.chunks[k] + 1);
        gp.lds_off[k] = (int)lds;
        lds += (size_t)kRows * gp.chunks[k] * 16;
    }
    gp.red_off = (int)lds;
    lds += (size_t)cs.ncand * kStreamThreads * sizeof(float);
    return any_iq(cs) ? launch_gate_few_t<true>(gp, ks, grid, lds, s) : launch_gate_few_t<false>(gp, ks, grid, lds, s);
}

}  // namespace vq
