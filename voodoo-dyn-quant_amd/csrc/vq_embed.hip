// Embedding rows straight from the packed candidates: the row-select lookup of
// a gated embedding (reference layers.py:670-750, 753-790) and the Q8_0
// teacher's embedding (training/q8_teacher.py:131-173).
//
// Every supported format stores a weight row as row_groups consecutive
// 256-weight groups, so row `id` of candidate k is the byte span
// [id * row_groups * gb_k, (id + 1) * row_groups * gb_k).  A workgroup takes as
// many requested rows as fit its 16 groups (4 rows of 1024 weights; a row of
// more than 16 groups is cut into segments, one per workgroup), copies each
// row's span of every candidate it needs into LDS, a wave per span, and
// decodes runs of 16 weights per thread as the full-matrix kernels do:
//   mixture:  out = ((0 + p0 W0) + p1 W1) + ..., the mix kernel's arithmetic
//             (fp32, products and sums rounded separately), stored as bf16
//             (the same row of W_eff bit for bit) or as fp32;
//   routed:   out = W_k(r), ggml's exact value, as bf16 or fp32;
//   backward: part[b][k] = <G rows of block b, W_k rows> for a bf16 or fp32 G,
//             reduced over blocks in a fixed order in fp64 (dL/dp_k).
// Row ids (and routes) outside their range give a zero row and a zero
// contribution; the kernels never read outside the candidate buffers.
//
// Bound: memory latency.  A workgroup's chain is id -> row bytes -> decode ->
// store, so what counts is that every span's copies are in flight together
// (whole 16-byte chunks only: a byte-wise tail would wait for the copies before
// it) and that no lane idles.  Measured on MI355X, 8192 ids of 1024 weights,
// K = 6: with one row per workgroup, byte-wise tails and 8 weights per thread
// the forward took 41 us and the backward with its reduction 76; as here 25
// and 32.  16384 ids of 5120 weights: 218 -> 175 and 382 -> 270.
#include "vq_internal.h"

namespace vq {

namespace {

// LDS bytes reserved for one candidate's span of `seg` groups: up to 15 bytes
// ahead of it (kept so every field sits at the same address mod 16 as in
// global memory) and the rest of its last 16-byte chunk.
__host__ __device__ constexpr int span_cap(int gb, int seg) { return (seg * gb + 15 + 15) & ~15; }

// Copy [src, src + len) to dst + (src mod 16), dst 16-byte aligned in LDS, by
// one wave's direct-to-LDS loads (buffer_load_dwordx4 ... lds: lane l lands at
// M0 + 16 l) of the 16-byte chunks that hold it, so every candidate's copies
// are in flight together.  The first chunk starts at or above the 16-byte
// aligned buffer that holds src; the last one is cut at `left`, the bytes from
// src to that buffer's end, rounded up to the 4 bytes a bounds check works in
// (the check fills the rest with zeros).
__device__ __forceinline__ void stage_span(uint8_t* __restrict__ dst, const uint8_t* __restrict__ src, int len,
                                           int64_t left) {
    typedef __attribute__((address_space(3))) void lds_void;
    const int head = (int)(reinterpret_cast<uintptr_t>(src) & 15u);
    const int nvec = (head + len + 15) >> 4;
    const int64_t room = (head + left + 3) & ~int64_t(3);
    const int bytes = (int)min<int64_t>(16 * nvec, room);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(src - head), (short)0, bytes, 0x00020000);
    const int lane = threadIdx.x & 63;
    for (int b = 0; b < nvec; b += 64)
        if (b + lane < nvec)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(dst + 16 * b), 16, 16 * (b + lane), 0, 0, 0);
}

// Address mod 16 of group `at` of the candidate at q: where its span starts in LDS.
__device__ __forceinline__ int span_head(const uint8_t* q, uint32_t at, int gb) {
    return (int)(((uint32_t)reinterpret_cast<uintptr_t>(q) + at * (uint32_t)gb) & 15u);
}

__device__ __forceinline__ void span_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Item i (a requested row's segment) of this workgroup's `per`.
struct Item {
    int64_t r;   // requested row (output row)
    int s0;      // first group of the segment
    int ng;      // groups in the segment; 0 past the last item
};

__device__ __forceinline__ Item item_at(int i, int64_t nids, const EmbedPlan& pl) {
    Item it;
    const uint32_t b = blockIdx.x * (uint32_t)pl.per + (uint32_t)i;  // nids * nseg < 2^31
    const uint32_t r = b / (uint32_t)pl.nseg;
    it.r = r;
    it.s0 = (int)(b - r * (uint32_t)pl.nseg) * pl.seg;
    it.ng = it.r < nids ? min(pl.seg, pl.gused - it.s0) : 0;
    return it;
}

// Where candidate k's span of item i starts in LDS, without its head.
struct Spans {
    int off[kMaxCand];  // of item 0
    int item;           // bytes per item
};

// This wave's share of the workgroup's (item, candidate) spans.  ROUTED: only
// each item's routed candidate is copied.
template <bool ROUTED>
__device__ __forceinline__ void stage_items(const CandSet& cs, const Spans& sp, const EmbedPlan& pl,
                                            const int64_t* __restrict__ ids, const int64_t* __restrict__ routing,
                                            int64_t nids, int64_t vocab, uint8_t* lds) {
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int ncopy = ROUTED ? pl.per : pl.per * cs.ncand;
    for (int c = wave; c < ncopy; c += kStreamThreads / 64) {
        const int i = ROUTED ? c : c / cs.ncand;
        const Item it = item_at(i, nids, pl);
        if (it.ng <= 0) continue;
        const int64_t id = ids[it.r];
        if (id < 0 || id >= vocab) continue;
        int k = c - i * cs.ncand;
        if constexpr (ROUTED) {
            const int64_t kr = routing[it.r];
            if (kr < 0 || kr >= cs.ncand) continue;
            k = (int)kr;
        }
        const int gb = group_bytes(cs.qtype[k]);
        const int64_t at = (id * cs.row_groups + it.s0) * gb;
        stage_span(lds + i * sp.item + (ROUTED ? 0 : sp.off[k]), cs.qbytes[k] + at, it.ng * gb,
                   vocab * cs.row_groups * gb - at);
    }
}

__device__ __forceinline__ void decode16_mix_rt(int qt, const uint8_t* g, int p, float (&w)[16]) {
    switch (qt) {
    case Q8_0: decode_mix<Q8_0, 16>(g, p, w); break;
    case Q2_K: decode_mix<Q2_K, 16>(g, p, w); break;
    case Q3_K: decode_mix<Q3_K, 16>(g, p, w); break;
    case Q4_K: decode_mix<Q4_K, 16>(g, p, w); break;
    case Q5_K: decode_mix<Q5_K, 16>(g, p, w); break;
    case Q6_K: decode_mix<Q6_K, 16>(g, p, w); break;
    default: decode_mix_iq<16>(qt, g, p, w); break;
    }
}

__device__ __forceinline__ float dot16_rt(int qt, const uint8_t* g, int p, const float* v) {
    switch (qt) {
    case Q8_0: return dot_run<Q8_0, 16>(g, p, v);
    case Q2_K: return dot_run<Q2_K, 16>(g, p, v);
    case Q3_K: return dot_run<Q3_K, 16>(g, p, v);
    case Q4_K: return dot_run<Q4_K, 16>(g, p, v);
    case Q5_K: return dot_run<Q5_K, 16>(g, p, v);
    case Q6_K: return dot_run<Q6_K, 16>(g, p, v);
    default: return dot_run_iq<16>(qt, g, p, v);
    }
}

__device__ __forceinline__ void store8(bf16_t* o, const float* v) {
    uint4 q;
    q.x = f2bf2(v[0], v[1]);
    q.y = f2bf2(v[2], v[3]);
    q.z = f2bf2(v[4], v[5]);
    q.w = f2bf2(v[6], v[7]);
    *reinterpret_cast<uint4*>(o) = q;
}

__device__ __forceinline__ void store8(float* o, const float* v) {
    float4* o4 = reinterpret_cast<float4*>(o);
    o4[0] = make_float4(v[0], v[1], v[2], v[3]);
    o4[1] = make_float4(v[4], v[5], v[6], v[7]);
}

__device__ __forceinline__ void load8(const bf16_t* g, float* v) {
    const uint4 q = *reinterpret_cast<const uint4*>(g);
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        v[2 * r] = __uint_as_float(w[r] << 16);
        v[2 * r + 1] = __uint_as_float(w[r] & 0xffff0000u);
    }
}

__device__ __forceinline__ void load8(const float* g, float* v) {
    const float4 a = reinterpret_cast<const float4*>(g)[0];
    const float4 b = reinterpret_cast<const float4*>(g)[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

}  // namespace

// The thread's place: the 16 weights 16 (t mod 16) .. of its item's group j.
struct Place {
    Item it;
    int64_t id, col;  // first of its columns
    int j, p, item;
    bool lo, hi;      // its first and second 8 columns exist (dim is a multiple of 8)
};

__device__ __forceinline__ Place place_of(const EmbedPlan& pl, const int64_t* __restrict__ ids, int64_t nids,
                                          int64_t dim) {
    Place q;
    const int slot = (int)threadIdx.x >> 4;
    q.p = 16 * (threadIdx.x & 15);
    q.item = slot / pl.seg;
    q.j = slot - q.item * pl.seg;
    q.it = item_at(q.item, nids, pl);
    const bool live = q.item < pl.per && q.j < q.it.ng;
    q.id = live ? ids[q.it.r] : -1;
    q.col = (int64_t)(q.it.s0 + q.j) * 256 + q.p;
    q.lo = live && q.col < dim;
    q.hi = live && q.col + 8 < dim;
    return q;
}

template <bool ROUTED, class OUT>
__global__ __launch_bounds__(kStreamThreads) void embed_rows_kernel(CandSet cs, Spans sp, EmbedPlan pl,
                                                                    const float* __restrict__ probs,
                                                                    const int64_t* __restrict__ routing,
                                                                    const int64_t* __restrict__ ids, int64_t nids,
                                                                    int64_t vocab, int64_t dim,
                                                                    OUT* __restrict__ out) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ float pr[kMaxCand];  // the probabilities, read once per workgroup
    stage_items<ROUTED>(cs, sp, pl, ids, routing, nids, vocab, lds);
    if (!ROUTED && (int)threadIdx.x < cs.ncand) pr[threadIdx.x] = probs[threadIdx.x];
    const Place q = place_of(pl, ids, nids, dim);
    bool valid = q.id >= 0 && q.id < vocab;
    int kr = 0;
    if constexpr (ROUTED) {
        const int64_t k = q.lo ? routing[q.it.r] : 0;
        valid = valid && k >= 0 && k < cs.ncand;
        kr = valid ? (int)k : 0;
    }
    span_wait();
    __syncthreads();
    if (!q.lo) return;
    float val[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) val[r] = 0.0f;
    if (valid) {
        const uint32_t at = (uint32_t)q.id * (uint32_t)cs.row_groups + (uint32_t)q.it.s0;  // its low bits count
        const uint8_t* base = lds + q.item * sp.item;
        if constexpr (ROUTED) {
            const int qt = cs.qtype[kr], gb = group_bytes(qt);
            const int head = span_head(cs.qbytes[kr], at, gb);
            decode_run_rt<8>(qt, base + head + q.j * gb, q.p, val);
            decode_run_rt<8>(qt, base + head + q.j * gb, q.p + 8, val + 8);
        } else {
            for (int k = 0; k < cs.ncand; ++k) {
                const int qt = cs.qtype[k], gb = group_bytes(qt);
                const int head = span_head(cs.qbytes[k], at, gb);
                float w[16];
                decode16_mix_rt(qt, base + sp.off[k] + head + q.j * gb, q.p, w);
                const float pk = pr[k];
                {
                    // product and sum rounded separately, as in the mix kernel
#pragma clang fp contract(off)
#pragma unroll
                    for (int r = 0; r < 16; ++r) val[r] = val[r] + pk * w[r];
                }
            }
        }
    }
    OUT* o = out + q.it.r * dim + q.col;
    store8(o, val);
    if (q.hi) store8(o + 8, val + 8);
}

// part[b][k] = sum over block b's weights of G[r][c] * W_k[id][c].
template <class GT>
__global__ __launch_bounds__(kStreamThreads) void embed_rows_bwd_kernel(CandSet cs, Spans sp, EmbedPlan pl,
                                                                        const int64_t* __restrict__ ids, int64_t nids,
                                                                        int64_t vocab, int64_t dim,
                                                                        const GT* __restrict__ grad,
                                                                        float* __restrict__ partials) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ float red[kMaxCand][kStreamThreads / 64];
    stage_items<false>(cs, sp, pl, ids, nullptr, nids, vocab, lds);
    // this thread's gradient values, kept across the candidates
    const int t = threadIdx.x;
    const Place q = place_of(pl, ids, nids, dim);
    const bool live = q.lo && q.id >= 0 && q.id < vocab;
    float v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = 0.0f;
    if (live) {
        const GT* g = grad + q.it.r * dim + q.col;
        load8(g, v);
        if (q.hi) load8(g + 8, v + 8);
    }
    span_wait();
    __syncthreads();
    const int wave = t >> 6;
    const uint32_t at = (uint32_t)q.id * (uint32_t)cs.row_groups + (uint32_t)q.it.s0;  // its low bits count
    const uint8_t* base = lds + q.item * sp.item;
    for (int k = 0; k < cs.ncand; ++k) {
        const int qt = cs.qtype[k], gb = group_bytes(qt);
        float a = 0.0f;
        if (live) {
            const int head = span_head(cs.qbytes[k], at, gb);
            a = dot16_rt(qt, base + sp.off[k] + head + q.j * gb, q.p, v);
        }
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) a += __shfl_xor(a, m, 64);
        if ((t & 63) == 0) red[k][wave] = a;
    }
    __syncthreads();
    if (t < cs.ncand) {
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < kStreamThreads / 64; ++w) s += red[t][w];
        partials[(int64_t)blockIdx.x * cs.ncand + t] = s;
    }
}

// One workgroup, so that the answer needs no cleared flag and no second launch;
// a thread keeps 8 ids in flight.  Launches bound the check it serves: as torch
// comparisons and an any() it took five.
__global__ __launch_bounds__(1024) void ids_out_of_range_kernel(const int64_t* __restrict__ ids, int nids,
                                                                int64_t vocab, uint8_t* __restrict__ bad) {
    bool mine = false;
    for (int64_t i0 = threadIdx.x; i0 < nids; i0 += 8 * 1024) {
        int64_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int64_t i = i0 + 1024 * u;
            v[u] = ids[i < nids ? i : nids - 1];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) mine = mine || v[u] < 0 || v[u] >= vocab;
    }
    const int any = __syncthreads_or(mine);
    if (threadIdx.x == 0) *bad = any ? 1 : 0;
}

hipError_t launch_ids_out_of_range(const int64_t* ids, int nids, int64_t vocab, uint8_t* bad, hipStream_t s) {
    ids_out_of_range_kernel<<<1, 1024, 0, s>>>(ids, nids, vocab, bad);
    return hipGetLastError();
}

EmbedPlan embed_plan(int64_t nids, int64_t dim) {
    EmbedPlan pl;
    pl.gused = (int)((dim + 255) / 256);
    pl.nseg = (pl.gused + kGroupsPerBlock - 1) / kGroupsPerBlock;
    pl.seg = pl.nseg > 0 ? (pl.gused + pl.nseg - 1) / pl.nseg : 0;
    pl.per = pl.nseg == 1 ? kGroupsPerBlock / pl.seg : 1;
    pl.blocks = (nids * pl.nseg + pl.per - 1) / pl.per;
    return pl;
}

static size_t embed_spans(const CandSet& cs, const EmbedPlan& pl, bool routed, Spans& sp) {
    sp = Spans{};
    for (int k = 0; k < cs.ncand; ++k) {
        const int c = span_cap(group_bytes(cs.qtype[k]), pl.seg);
        sp.off[k] = routed ? 0 : sp.item;
        sp.item = routed ? (c > sp.item ? c : sp.item) : sp.item + c;
    }
    return (size_t)sp.item * pl.per;
}

template <class OUT>
static hipError_t embed_rows_t(const CandSet& cs, const float* probs, const int64_t* routing, const int64_t* ids,
                               int64_t nids, int64_t vocab, int64_t dim, const EmbedPlan& pl, OUT* out,
                               hipStream_t s) {
    const dim3 grid((unsigned)pl.blocks);
    Spans sp;
    const size_t lds = embed_spans(cs, pl, routing != nullptr, sp);
    const hipError_t e = allow_dynamic_lds(
        routing ? (const void*)embed_rows_kernel<true, OUT> : (const void*)embed_rows_kernel<false, OUT>, lds);
    if (e != hipSuccess) return e;
    if (routing)
        embed_rows_kernel<true, OUT><<<grid, kStreamThreads, lds, s>>>(cs, sp, pl, probs, routing, ids, nids, vocab,
                                                                       dim, out);
    else
        embed_rows_kernel<false, OUT><<<grid, kStreamThreads, lds, s>>>(cs, sp, pl, probs, nullptr, ids, nids, vocab,
                                                                        dim, out);
    return hipSuccess;
}

hipError_t launch_embed_rows(const CandSet& cs, const float* probs, const int64_t* routing, const int64_t* ids,
                             int64_t nids, int64_t vocab, int64_t dim, void* out, bool out_f32, hipStream_t s) {
    const EmbedPlan pl = embed_plan(nids, dim);
    if (pl.blocks <= 0) return hipSuccess;
    const hipError_t e =
        out_f32 ? embed_rows_t(cs, probs, routing, ids, nids, vocab, dim, pl, static_cast<float*>(out), s)
                : embed_rows_t(cs, probs, routing, ids, nids, vocab, dim, pl, static_cast<bf16_t*>(out), s);
    if (e != hipSuccess) return e;
    return hipGetLastError();
}

hipError_t launch_embed_rows_bwd(const CandSet& cs, const int64_t* ids, int64_t nids, int64_t vocab, int64_t dim,
                                 const void* grad, bool grad_f32, float* partials, float* dprobs, hipStream_t s) {
    const EmbedPlan pl = embed_plan(nids, dim);
    if (pl.blocks <= 0) {
        // no rows: dL/dp is zero (written by a kernel, not a memset, so the call can be captured)
        return launch_gate_reduce(partials, 0, cs.ncand, dprobs, s);
    }
    const dim3 grid((unsigned)pl.blocks);
    Spans sp;
    const size_t lds = embed_spans(cs, pl, false, sp);
    const hipError_t ea = allow_dynamic_lds(
        grad_f32 ? (const void*)embed_rows_bwd_kernel<float> : (const void*)embed_rows_bwd_kernel<bf16_t>, lds);
    if (ea != hipSuccess) return ea;
    if (grad_f32)
        embed_rows_bwd_kernel<float><<<grid, kStreamThreads, lds, s>>>(
            cs, sp, pl, ids, nids, vocab, dim, static_cast<const float*>(grad), partials);
    else
        embed_rows_bwd_kernel<bf16_t><<<grid, kStreamThreads, lds, s>>>(
            cs, sp, pl, ids, nids, vocab, dim, static_cast<const bf16_t*>(grad), partials);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_gate_reduce(partials, pl.blocks, cs.ncand, dprobs, s);
}

}  // namespace vq
