// The 256x256 bf16 products on gfx950: C[i][j] = sum_k A[i][k] B[j][k] with
// four waves of 128x128 (v_mfma_f32_16x16x32_bf16, 256 fp32 accumulators per
// lane in AGPRs), one wave per SIMD, the operands streamed through LDS by
// direct-to-LDS copies in stages of 64 k.
//
// What bounds it: the card's power while the matrix pipes work, and what keeps
// them from working.  Against eight waves of 64x128 on 32x32x16 (two waves per
// SIMD hiding each other's fragment reads), this layout reads a third less
// from LDS per MFMA, moves half the accumulator bytes per FLOP and leaves no
// address arithmetic in the loop, so the chip holds a higher clock; nothing
// hides a stall of the single wave, so the loop is written as instruction text
// (vq_gemm_loop.inc) with every read and copy placed behind a given MFMA.
// Measured on MI355X, 8192 tokens, forward: 5120 -> 17408 1127-1146 -> 928-968
// us, 5120 -> 6144 401 -> 329 us, 1024 -> 6144 99 -> 81 us.
//
// Operands are K-major ("KS": [rows][K], fragments by ds_read_b128) or
// [K][rows] ("NS": fragments by ds_read_b64_tr_b16).  A's rows are permuted
// within each 64: MFMA row m of fragment a reads tile row
// 64 (a / 4) + 16 (m / 4) + 4 (a % 4) + m % 4, so that the four accumulators of
// fragments 4 q .. 4 q + 3 hold 16 consecutive rows i for one j per lane:
//   acc(a, b)[r] of lane l = C[64 (a / 4) + 16 (l / 16) + 4 (a % 4) + r][16 b + l % 16]
// relative to the wave's 128x128 tile.
//
// MFMA 16x16x32 operand/result layout (64 lanes):
//   A: lane l holds A[i = l%16][k = 8*(l/16) .. +7]
//   B: lane l holds B[k = 8*(l/16) .. +7][j = l%16]
//   D: register r of lane l is D[i = 4*(l/16) + r][j = l%16]
#pragma once

#include "vq_gemm_impl.h"
#include "vq_gemm_loop.inc"

namespace vq {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x32 __attribute__((ext_vector_type(32)));

enum OperandLayout : int { KS = 0, NS = 1 };

constexpr int kStThreads = 256;
constexpr int kStTile = 256;                    // rows i and columns j of a workgroup's tile
constexpr int kStBK = 64;                       // k per stage
constexpr int kStOperand = 32 * 1024;           // bytes of one operand's stage
constexpr int kStStage = 2 * kStOperand;        // A's 32 KiB, then B's; buffer 1 starts at kStStage
constexpr int kStTurn = 8 * 1024;               // a wave's 32 x 128 bf16 block of a store epilogue
constexpr size_t kStStoreLds = 2 * kStStage + 4 * kStTurn;
constexpr int kStStores = 32;                   // 16-byte stores per lane and stored tile
static_assert(kStStage == 0x10000, "the loop text moves between the buffers by xor");
static_assert(kStStoreLds <= 160 * 1024, "exceeds the 160 KiB of LDS per workgroup");

// The swizzles: the 16-byte chunk c of a row (KS) or k-row (NS) sits in slot
// c ^ swz.  A lane group of a read then touches distinct bank groups:
//   KS, A: rows of one pass differ in bits 0, 1, 4, 5 (permuted fragments);
//   KS, B: in bits 0..3;
//   NS, A: 4 k-rows x 4 granules two chunks apart; NS, B: 4 k-rows x 4
//   granules in two neighbouring chunks.
// None depends on the bits a fragment's index moves, so one address register
// and immediate offsets reach every fragment (NS: a register per xor pattern).
template <OperandLayout L, bool PERM>
__device__ __forceinline__ int st_swz(int r) {
    if constexpr (L == KS)
        return PERM ? (((r ^ (r >> 5)) & 1) | (r & 2) | ((r >> 2) & 4)) : ((r & 7) ^ ((r >> 3) & 1));
    else
        return PERM ? ((r & 1) | ((r & 2) << 2)) : ((r & 3) << 1);
}

// One operand of a tile: where its stages' copies read.
template <OperandLayout L, bool PERM>
struct StOperand {
    // byte offsets of this lane's 8 copies of a stage from the stage's base;
    // kOOB (zeros) for rows past `rows` and k past `kvalid`
    static __device__ __forceinline__ void offsets(int* vo, int64_t ld, int r0, int rows, int kvalid, int tid) {
        const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if constexpr (L == KS) {
                const int row = (i * 4 + wave) * 8 + (lane >> 3);
                const int c = (lane & 7) ^ st_swz<L, PERM>(row);
                vo[i] = ((r0 + row < rows) & (8 * c + 8 <= kvalid)) ? (int)((row * ld + 8 * c) * 2) : (int)kOOB;
            } else {
                const int kr = (i * 4 + wave) * 2 + (lane >> 5);
                const int c = (lane & 31) ^ st_swz<L, PERM>(kr);
                vo[i] = ((r0 + 8 * c < rows) & (kr < kvalid)) ? (int)((kr * ld + 8 * c) * 2) : (int)kOOB;
            }
        }
    }
    // the base of the stage at k of the tile at row r0, and the step to the next stage's
    static __device__ __forceinline__ uint64_t base(const bf16_t* src, int64_t ld, int r0, int k) {
        return reinterpret_cast<uint64_t>(L == KS ? src + (int64_t)r0 * ld + k : src + (int64_t)k * ld + r0);
    }
    static __device__ __forceinline__ int64_t step(int64_t ld) { return L == KS ? 2 * kStBK : 2 * kStBK * ld; }
    // LDS addresses of this lane's fragment reads in the stage at `lds`; w: the wave's 128-row half
    static __device__ __forceinline__ void read_addrs(int (&a)[4], uint32_t lds, int w, int lane) {
        const int m = lane & 15, g = lane >> 4;
        if constexpr (L == KS) {
            const int row = 128 * w + (PERM ? 16 * (m >> 2) + (m & 3) : m);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) a[ks] = (int)(lds + 128 * row + 16 * ((4 * ks + g) ^ st_swz<L, PERM>(row)));
            a[2] = a[3] = 0;
        } else {
            const int k = 8 * g + (m >> 2), q = m & 3;
            const int chunk = (16 * w + (PERM ? 2 * q : q >> 1)) ^ st_swz<L, PERM>(k);
            const int at = (int)(lds + 512 * k + 16 * chunk + (PERM ? 0 : 8 * (q & 1)));
#pragma unroll
            for (int x = 0; x < 4; ++x) a[x] = at ^ (PERM ? 16 * (x & 1) + 128 * (x >> 1) : 32 * x);
        }
    }
};

// A tile's share of a stream of stages.
struct StTile {
    int i0, j0, kbeg, kend;
    int nk;                    // stages: at least 3 (those past kend are zeros)
    int split, ns, tail_slot;  // as WorkItem
    bool live;
};

__device__ __forceinline__ StTile st_tile(int i0, int j0, int kbeg, int kend, bool live) {
    StTile t;
    t.live = live;
    t.i0 = live ? i0 : 0;
    t.j0 = live ? j0 : 0;
    t.kbeg = live ? kbeg : 0;
    t.kend = live ? kend : 0;
    const int nk = (t.kend - t.kbeg + kStBK - 1) / kStBK;
    t.nk = nk < 3 ? 3 : nk;
    t.split = 0;
    t.ns = 1;
    t.tail_slot = -1;
    return t;
}

// The thread index as a value of its own: what a tile boundary computes from
// it is then computed there again instead of being kept in registers through
// the main loop, which has none to spare.
__device__ __forceinline__ int fresh_tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

#if defined(__HIP_DEVICE_COMPILE__)
#define VQ_R10(p, n) p #n "0", p #n "1", p #n "2", p #n "3", p #n "4", p #n "5", p #n "6", p #n "7", p #n "8", p #n "9"
#define VQ_ST_VGPRS                                                                                                  \
    "v128", "v129", VQ_R10("v", 13), VQ_R10("v", 14), VQ_R10("v", 15), VQ_R10("v", 16), VQ_R10("v", 17),              \
        VQ_R10("v", 18), "v190", "v191"
#define VQ_ST_AGPRS                                                                                                  \
    "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", VQ_R10("a", 1), VQ_R10("a", 2), VQ_R10("a", 3),       \
        VQ_R10("a", 4), VQ_R10("a", 5), VQ_R10("a", 6), VQ_R10("a", 7), VQ_R10("a", 8), VQ_R10("a", 9),               \
        VQ_R10("a", 10), VQ_R10("a", 11), VQ_R10("a", 12), VQ_R10("a", 13), VQ_R10("a", 14), VQ_R10("a", 15),         \
        VQ_R10("a", 16), VQ_R10("a", 17), VQ_R10("a", 18), VQ_R10("a", 19), VQ_R10("a", 20), VQ_R10("a", 21),         \
        VQ_R10("a", 22), VQ_R10("a", 23), VQ_R10("a", 24), "a250", "a251", "a252", "a253", "a254", "a255"
// One run of the loop text.  The accumulators live in a[0:255] from one run to
// the next (the compiler keeps nothing there: every run clobbers them), the
// fragments of the next k-step in v[64:127].  The text advances the copies'
// base addresses and destination itself; the members track them.
#define VQ_ST_RUN(TEXT, COUNT)                                                                                       \
    do {                                                                                                             \
        i32x4 ra_out, rb_out;                                                                                        \
        int fill_out, n_out, m0_save;                                                                                \
        asm volatile(TEXT                                                                                            \
                     : "+{v[64:95]}"(fa), "+{v[96:127]}"(fb), [a0] "+v"(aa[0]), [a1] "+v"(aa[1]), [a2] "+v"(aa[2]),   \
                       [a3] "+v"(aa[3]), [b0] "+v"(ab[0]), [b1] "+v"(ab[1]), [b2] "+v"(ab[2]), [b3] "+v"(ab[3]),      \
                       "={s[84:87]}"(ra_out), "={s[88:91]}"(rb_out), [fill] "=s"(fill_out), [n] "=s"(n_out),          \
                       [m0save] "=&s"(m0_save)                                                                       \
                     : "{s[84:87]}"(rsrc(ka)), "{s[88:91]}"(rsrc(kb)), "[fill]"(fill), "[n]"(COUNT), [da] "s"(da),    \
                       [db] "s"(db), [v0] "v"(vo[0]), [v1] "v"(vo[1]), [v2] "v"(vo[2]), [v3] "v"(vo[3]),              \
                       [v4] "v"(vo[4]), [v5] "v"(vo[5]), [v6] "v"(vo[6]), [v7] "v"(vo[7]), [v8] "v"(vo[8]),           \
                       [v9] "v"(vo[9]), [v10] "v"(vo[10]), [v11] "v"(vo[11]), [v12] "v"(vo[12]), [v13] "v"(vo[13]),   \
                       [v14] "v"(vo[14]), [v15] "v"(vo[15])                                                          \
                     : VQ_ST_VGPRS, VQ_ST_AGPRS, "memory", "scc");                                                   \
    } while (0)

// The stream of one workgroup: copies run two stages ahead of the MFMAs.
template <OperandLayout LA_, OperandLayout LB_>
struct Stream {
    using OA = StOperand<LA_, true>;
    using OB = StOperand<LB_, false>;
    static constexpr bool kStoresInFlight = LB_ == KS;  // products whose stream goes on past a tile's stores
    int vo[16];        // A's, then B's copy offsets
    uint64_t ka, kb;   // the next stage to copy
    int da, db;        // bytes from one stage to the next (below 2^31: 128 bytes per k-row column)
    int fill;          // LDS address of this wave's first copy of the next stage
    int aa[4], ab[4];  // fragment read addresses
    i32x32 fa, fb;     // fragments of the next k-step
    int s;             // the next stage to copy, within its tile
    bool full;         // vo holds the offsets of whole stages

    static __device__ __forceinline__ i32x4 rsrc(uint64_t base) {
        return i32x4{__builtin_amdgcn_readfirstlane((int)base), __builtin_amdgcn_readfirstlane((int)((base >> 32) & 0xffff)),
                     (int)kRange, 0x00020000};
    }
    // Offsets of the stage `s` of tile t; B's rows through p.rowmap when GATHER.
    template <bool GATHER>
    __device__ __forceinline__ void offsets(const GemmParams& p, const StTile& t) {
        const int left = t.kend - t.kbeg - kStBK * s;
        const int kvalid = left < 0 ? 0 : left < kStBK ? left : kStBK;
        const int tid = fresh_tid();
        OA::offsets(vo, p.lda, t.i0, p.I, kvalid, tid);
        if constexpr (GATHER) {
            const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int row = (i * 4 + wave) * 8 + (lane >> 3);
                const int c = (lane & 7) ^ st_swz<KS, false>(row);
                const int src = t.j0 + row < p.J ? p.rowmap[t.j0 + row] : -1;
                vo[8 + i] = (((unsigned)src < (unsigned)p.map_rows) & (8 * c + 8 <= kvalid))
                                ? (int)(((int64_t)src * p.ldb + 8 * c) * 2)
                                : (int)kOOB;
            }
        } else {
            OB::offsets(vo + 8, p.ldb, t.j0, p.J, kvalid, tid);
        }
        full = kvalid == kStBK;
    }
    // Points the copies at tile t's first stage.
    template <bool GATHER>
    __device__ __forceinline__ void enter(const GemmParams& p, const StTile& t) {
        s = 0;
        ka = OA::base(p.A, p.lda, t.i0, t.kbeg);
        kb = GATHER ? reinterpret_cast<uint64_t>(p.B + t.kbeg) : OB::base(p.B, p.ldb, t.j0, t.kbeg);
        offsets<GATHER>(p, t);
    }
    __device__ __forceinline__ void advance(int n) {
        s += n;
        ka += (int64_t)n * OA::step(lda_);
        kb += (int64_t)n * OB::step(ldb_);
    }
    // Copies of the first two stages of tile t, then the first fragments.
    template <bool GATHER>
    __device__ __forceinline__ void start(const GemmParams& p, const StTile& t, u32x4* __restrict__ smem) {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const uint32_t lds = (uint32_t)(uintptr_t)(lds_void_t*)smem;  // 0: the kernels have no static LDS
        lda_ = p.lda;
        ldb_ = p.ldb;
        da = (int)OA::step(p.lda);
        db = (int)OB::step(p.ldb);
        enter<GATHER>(p, t);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            if (b == 1 && !(full && t.kend - t.kbeg >= 2 * kStBK)) offsets<GATHER>(p, t);
#pragma unroll
            for (int i = 0; i < 16; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(reinterpret_cast<const void*>(i < 8 ? ka : kb)),
                                                         (lds_void_t*)(smem + (b * kStStage + i * 4096) / 16 + 64 * wave),
                                                         16, vo[i], 0, 0, 0);
            advance(1);
        }
        fill = (int)lds + 1024 * wave;
        OA::read_addrs(aa, lds, wave >> 1, lane);
        OB::read_addrs(ab, lds + kStOperand, wave & 1, lane);
        asm volatile("s_waitcnt vmcnt(16)\n\ts_barrier" ::: "memory");
#define VQ_ST_READ(TEXT)                                                                                             \
    asm volatile(TEXT                                                                                                \
                 : "=&{v[64:95]}"(fa), "=&{v[96:127]}"(fb)                                                           \
                 : [a0] "v"(aa[0]), [a1] "v"(aa[1]), [a2] "v"(aa[2]), [a3] "v"(aa[3]), [b0] "v"(ab[0]),               \
                   [b1] "v"(ab[1]), [b2] "v"(ab[2]), [b3] "v"(ab[3])                                                 \
                 : "memory")
        if constexpr (LA_ == KS && LB_ == KS)
            VQ_ST_READ(VQ_STREAM_KSKS_READ);
        else if constexpr (LB_ == KS)
            VQ_ST_READ(VQ_STREAM_NSKS_READ);
        else
            VQ_ST_READ(VQ_STREAM_NSNS_READ);
#undef VQ_ST_READ
    }
    // Multiplies the nk stages of tile `cur` into fresh accumulators while the
    // copies move on to tile `nxt`.  stores: `cur`'s first stage runs with the
    // last tile's kStStores stores still in flight.
    template <bool GATHER>
    __device__ __forceinline__ void tile(const GemmParams& p, const StTile& cur, const StTile& nxt, bool stores) {
        int rem = cur.nk;
        bool in_cur = true, first = true;
        while (rem > 0) {
            if (in_cur && s == cur.nk) {
                in_cur = false;
                enter<GATHER>(p, nxt);
            }
            const StTile& t = in_cur ? cur : nxt;
            const int left = t.kend - t.kbeg - kStBK * s;  // k from the next stage on
            if ((left >= kStBK) != full || !full) offsets<GATHER>(p, t);
            // one run per kind of stage: whole stages together, the others singly
            int n = left >= kStBK ? left / kStBK : 1;
            n = n < rem ? n : rem;
            if (first) {
                n = 1;
                if constexpr (LA_ == KS && LB_ == KS) {
                    if (stores)
                        VQ_ST_RUN(VQ_STREAM_KSKS_FIRST_STORES, 1);
                    else
                        VQ_ST_RUN(VQ_STREAM_KSKS_FIRST, 1);
                } else if constexpr (LB_ == KS) {
                    if (stores)
                        VQ_ST_RUN(VQ_STREAM_NSKS_FIRST_STORES, 1);
                    else
                        VQ_ST_RUN(VQ_STREAM_NSKS_FIRST, 1);
                } else {
                    VQ_ST_RUN(VQ_STREAM_NSNS_FIRST, 1);
                }
                first = false;
            } else {
                if constexpr (LA_ == KS && LB_ == KS)
                    VQ_ST_RUN(VQ_STREAM_KSKS_LOOP, n);
                else if constexpr (LB_ == KS)
                    VQ_ST_RUN(VQ_STREAM_NSKS_LOOP, n);
                else
                    VQ_ST_RUN(VQ_STREAM_NSNS_LOOP, n);
            }
            fill ^= (n & 1) << 16;
            advance(n);
            rem -= n;
        }
    }

private:
    int64_t lda_, ldb_;
};

#endif  // __HIP_DEVICE_COMPILE__

// The accumulators after a tile's last stage.  They stay in a[0:255], where the
// loop text leaves them, and are read one register at a time: as C++ values
// the compiler would copy all 256 around.  It keeps nothing of its own there
// (the runs clobber every AGPR, and the epilogues fit the VGPRs).
// The token orders the reads: st_acc depends on it and on nothing else, so
// loads move freely across the reads, and a read moves no further up than the
// token's last st_pin.
__device__ __forceinline__ int st_accumulators_ready() {
    int token = 0;
    asm volatile("s_nop 15\n\ts_nop 3" : "+v"(token) : : "memory");  // an MFMA's result reaches VALU reads after 11 wait states
    return token;
}
// Element r of accumulator (a, b).
__device__ __forceinline__ float st_acc(int token, int a, int b, int r) {
    float x = 0.0f;
#if defined(__HIP_DEVICE_COMPILE__)
    asm("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x) : "n"(32 * a + 4 * b + r), "v"(token));
#endif
    return x;
}

// Later reads come after x: without such points the compiler reads all 256
// accumulators first.
__device__ __forceinline__ void st_pin(int& token, float& x) { asm("" : "+v"(token), "+v"(x)); }

// Store epilogue: C[j][i] in bf16.  A wave turns 32 j x 128 i at a time through
// 8 KiB of LDS of its own (no barrier, and the stage buffers stay free for the
// next tile's copies) and stores 256-byte row pieces, 32 stores per lane in
// all, always issued: rows and columns past the matrix go out of the
// descriptor's range.  Nothing waits for them until two stages later.
// Non-temporal: every CU writes its tile at about the same moment, and the
// burst would push operand lines out of L2.
__device__ __forceinline__ void st_store_tile(const GemmParams& p, const StTile& t, u32x4* __restrict__ smem, int token,
                                              bool scatter) {
    const int tid = fresh_tid();
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wi = wave >> 1, wj = wave & 1, h = lane >> 4;
    u32x4* const turn = smem + (2 * kStStage + wave * kStTurn) / 16;
    const int ib = t.i0 + 128 * wi;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        __builtin_amdgcn_sched_barrier(0);  // one block's accumulators in VGPRs at a time
#pragma unroll
        for (int b2 = 0; b2 < 2; ++b2) {
            const int j = 16 * b2 + (lane & 15);
#pragma unroll
            for (int c = 0; c < 4; ++c) {  // 8 consecutive i: fragments 2 c, 2 c + 1
                u32x4 w;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    w[e] = pk_bf16(st_acc(token, 2 * c + (e >> 1), 2 * q + b2, 2 * (e & 1)),
                                   st_acc(token, 2 * c + (e >> 1), 2 * q + b2, 2 * (e & 1) + 1));
                turn[16 * j + ((8 * (c >> 1) + 2 * h + (c & 1)) ^ (j & 15))] = w;
            }
        }
        const int jb = t.j0 + 128 * wj + 32 * q;
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.C + (scatter ? 0 : (int64_t)jb * p.ldc) + ib);
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            const int row = 4 * x + (lane >> 4), c = lane & 15;
            const u32x4 w = turn[16 * row + (c ^ (row & 15))];
            bool ok = (jb + row < p.J) & (ib + 8 * c < p.I);
            if (scatter) {  // 64-bit row addresses: C may pass 2^31 bytes
                const int dest = jb + row < p.J ? p.rowmap[jb + row] : -1;
                ok = ok && (unsigned)dest < (unsigned)p.map_rows;
                if (ok) __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(p.C + (int64_t)dest * p.ldc + ib + 8 * c));
            } else {
                __builtin_amdgcn_raw_buffer_store_b128(w, rs, ok ? (int)((row * p.ldc + 8 * c) * 2) : (int)kOOB, 0, 2);
            }
        }
    }
}

// K part of a split tile: fp32, [element 32 a + 4 b + r][thread].
__device__ __forceinline__ void st_store_part(float* __restrict__ slot, int token) {
#pragma unroll
    for (int a = 0; a < 8; ++a) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 32; ++e) slot[(32 * a + e) * kStThreads + threadIdx.x] = st_acc(token, a, e >> 2, e & 3);
    }
}

// Measured on MI355X, split against whole: 8 rounds, a part saving 40 of 80
// steps (8192 x 5120 -> 17408 forward) 1009 against 970-987 us; 1 round, 40 of
// 80 (4096 x 5120 -> 6144 forward) 185 against 198 us, 72 of 96 (its dX) 183
// against 227 us; 2 rounds, 136 of 272 (8192 x 17408 -> 5120 forward) 1028
// against 1179 us.
constexpr int kMinSavedPerRound = 12;

// A tile configuration: layouts, and how the tiles become work items.
// C[j][i] products (STORE) may split their last tiles along K when the caller
// gives workspace; gate products split without any (each part has its own
// partial sums); parts products run every tile in p.parts parts.
template <OperandLayout LA_, OperandLayout LB_, int EPI_>
struct StCfg {
    static constexpr OperandLayout LA = LA_, LB = LB_;
    static constexpr int EPI = EPI_;
    static constexpr int BI = kStTile, BJ = kStTile, BK = kStBK, THREADS = kStThreads;
    static constexpr size_t lds() {
        constexpr size_t gate = (size_t)2 * BJ * kGateMaxChunks * 16 + 4 * kMaxCand * 4;  // two candidate buffers, wave sums
        return EPI == EPI_STORE ? kStStoreLds : EPI == EPI_GATE && gate > 2 * kStStage ? gate : 2 * kStStage;
    }
    static int tiles_i(const GemmParams& p) { return (p.I + BI - 1) / BI; }
    static int tiles_j(const GemmParams& p) { return (p.J + BJ - 1) / BJ; }
    static __host__ __device__ int ksteps(const GemmParams& p) { return (p.K + BK - 1) / BK; }
    // Fill in the work decomposition; returns the grid size (8 * items per XCD).
    // per_round: kMinSavedPerRound applies (without it the plan bounds the workspace).
    static int plan(GemmParams& p, int cus, bool split_ok, bool per_round = true) {
        if (p.I <= 0 || p.J <= 0) return 0;
        p.cus_per_xcd = cus / 8 > 0 ? cus / 8 : 1;
        p.tail_max = 0;
        p.s_max = 1;
        const int tiles = tiles_i(p) * tiles_j(p);
        int items = 0;
        if constexpr (EPI == EPI_PARTS) {
            // every tile in p.parts parts, the XCDs' tile ranges as for whole tiles
            p.split_ok = 0;
            for (int x = 0; x < 8; ++x) {
                const XcdPlan pl = xcd_plan(x, tiles, p.cus_per_xcd, ksteps(p), false);
                items = pl.tiles * p.parts > items ? pl.tiles * p.parts : items;
            }
            return 8 * items;
        }
        // A split store tile pays for its partial writes and a fixup launch, so
        // a part has to save kMinSavedSplitSteps K steps, and kMinSavedPerRound
        // more for every whole round of tiles before it: behind many rounds a
        // half-empty last one costs less than its time, since the card is at
        // its power limit and the fewer CUs run it at a higher clock.
        const int rounds = per_round ? tiles / (8 * p.cus_per_xcd) : 0;
        p.split_min_saved = EPI == EPI_STORE ? kMinSavedSplitSteps + kMinSavedPerRound * rounds : 0;
        p.split_max = 8;
        p.split_ok = split_ok ? 1 : 0;
        for (int x = 0; x < 8; ++x) {
            const XcdPlan pl = xcd_plan(x, tiles, p.cus_per_xcd, ksteps(p), split_ok, p.split_min_saved, p.split_max);
            items = pl.items() > items ? pl.items() : items;
            p.tail_max = pl.tail > p.tail_max ? pl.tail : p.tail_max;
            p.s_max = pl.s > p.s_max ? pl.s : p.s_max;
        }
        return 8 * items;
    }
    // fp32 workspace the split tails of a store product need
    static int64_t tail_bytes(const GemmParams& p) {
        return p.tail_max > 0 ? (int64_t)8 * p.tail_max * p.s_max * BI * BJ * 4 : 0;
    }
    // Work item `block` (of an XCD's: block / 8).  Tile-rows of the grouped
    // order are the activation rows: j of a store product, i of a gate one.
    static __device__ __forceinline__ StTile item(const GemmParams& p, int block) {
        const int ti = (p.I + BI - 1) / BI, tj = (p.J + BJ - 1) / BJ;
        const int steps = (p.K + BK - 1) / BK;
        if constexpr (EPI == EPI_PARTS) {
            const int local = block / 8;
            const XcdPlan pl = xcd_plan(block % 8, ti * tj, p.cus_per_xcd, steps, false);
            const bool live = local < pl.tiles * p.parts;
            int tm, tn;
            tile_coords(live ? pl.t0 + local / p.parts : 0, ti, tj, kGroupM, tm, tn);
            const int chunk = (steps + p.parts - 1) / p.parts * BK, part = local % p.parts;
            const int kbeg = min(p.K, part * chunk);
            StTile t = st_tile(tm * BI, tn * BJ, kbeg, min(p.K, kbeg + chunk), live);
            t.split = part;
            return t;
        }
        const WorkItem w = map_work(block, EPI == EPI_STORE ? tj : ti, EPI == EPI_STORE ? ti : tj, steps, p.cus_per_xcd,
                                    p.split_ok != 0, p.tail_max, kGroupM, p.split_min_saved, p.split_max);
        int kbeg = 0, kend = p.K;
        if (w.ns > 1) {
            const int chunk = (steps + w.ns - 1) / w.ns * BK;
            kbeg = min(p.K, w.split * chunk);
            kend = min(p.K, kbeg + chunk);
        }
        StTile t = st_tile((EPI == EPI_STORE ? w.tn : w.tm) * BI, (EPI == EPI_STORE ? w.tm : w.tn) * BJ, kbeg, kend,
                           !w.idle);
        t.split = w.split;
        t.ns = w.ns;
        t.tail_slot = w.tail_slot;
        return t;
    }
};

// ---------------------------------------------------------------- gate epilogue
// As described at gate_span_chunks: the tile's candidates stream through LDS, two
// in turn, and every lane decodes exactly the weights its accumulators hold:
// for column j (row n of the candidate) 16 b + l % 16, the 16 consecutive
// weights 64 a4 + 16 (l / 16) .. + 15, a4 = 0, 1.
//
// A candidate's rows of the tile, in 32-bit offsets from the 16-byte boundary
// at or below the tile's first row: row r's span of the group starts at
// head + r * stride (a row past the tensor takes row 0's).
struct StGateRows {
    int64_t origin;
    int stride, head, gb, rows;
    __device__ __forceinline__ StGateRows(int qt, int64_t row_groups, int j0, int group, int J) {
        gb = group_bytes(qt);
        stride = (int)(row_groups * gb);
        const int64_t first = (int64_t)j0 * row_groups * gb;
        origin = first & ~int64_t(15);
        head = (int)(first & 15) + group * gb;
        rows = J - j0;
    }
    __device__ __forceinline__ int span(int r) const { return head + (r < rows ? r : 0) * stride; }
};

// Copies of a candidate's 256 row spans: a lane's (row, chunk) moves on by 256
// chunks at a time, without a division per copy.
__device__ __forceinline__ void st_gate_stage(u32x4* __restrict__ buf, const uint8_t* __restrict__ qbytes, int qt,
                                              int64_t row_groups, int j0, int group, int J) {
    const StGateRows rw(qt, row_groups, j0, group, J);
    const int nch = gate_row_chunks(qt);
    const int64_t bytes = (int64_t)J * row_groups * rw.gb - rw.origin;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(qbytes + rw.origin), (short)0, (int)(bytes < (int64_t)kRange ? bytes : (int64_t)kRange),
        0x00020000);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int q = 256 / nch, rem = 256 - q * nch;
    int row = (int)threadIdx.x / nch, c = (int)threadIdx.x - row * nch;
    u32x4* dst = buf + 64 * wave;  // lanes land at dst + 16 lane
    if (rw.rows >= kStTile) {
        int at = rw.span(row);
        const int step = q * rw.stride;
        for (int i = 0; i < nch; ++i) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t*)dst, 16, (at & ~15) + 16 * c, 0, 0, 0);
            dst += 256;
            c += rem;
            at += step;
            if (c >= nch) {
                c -= nch;
                at += rw.stride;
            }
        }
        return;
    }
    for (int i = 0; i < nch; ++i) {  // the last rows' tile: rows past the tensor read row 0's span
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t*)dst, 16, (rw.span(row) & ~15) + 16 * c, 0, 0, 0);
        dst += 256;
        row += q;
        c += rem;
        if (c >= nch) {
            c -= nch;
            ++row;
        }
    }
}

// <acc, W_k> over the lane's accumulators.
template <int QT>
__device__ __forceinline__ float st_gate_dot(int& token, const float (&sv)[2][8], const float (&kept)[4][16],
                                             const uint8_t* __restrict__ buf, int64_t row_groups, int j0, int group,
                                             int wi, int wj, int lane, int J) {
    const StGateRows rw(QT, row_groups, j0, group, J);
    const int pitch = 16 * gate_span_chunks(rw.gb);  // bytes per staged row span
    asm("" : "+v"(lane) : "v"(token));  // row addresses computed here, per candidate, not kept for all of them
    const int p = 128 * wi + 16 * (lane >> 4);
    float s = 0.0f;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const int nl = 128 * wj + 16 * b + (lane & 15);
        const uint8_t* g = buf + nl * pitch + (rw.span(nl) & 15);
#pragma unroll
        for (int a4 = 0; a4 < 2; ++a4) {
            float v[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = a4 == 0 && b < 4 ? kept[b & 3][r] : st_acc(token, 4 * a4 + (r >> 2), b, r & 3);
            if constexpr (is_iq(QT))
                s += dot_sub16_iq(QT, g, p + 64 * a4, v, sv[a4][b]);
            else
                s += dot_sub16<QT>(g, p + 64 * a4, v, sv[a4][b]);
        }
        if (is_iq(QT) || (b & 1)) st_pin(token, s);  // four blocks' accumulators at a time (IQ: two)
    }
    return s;
}

// IQ: the candidate set may hold IQ formats (their table-lookup decode needs
// registers the K-quant-only instantiation keeps for itself).
template <bool IQ>
__device__ __forceinline__ void st_gate_epilogue(const GemmParams& p, int block, int i0, int j0,
                                                 u32x4* __restrict__ smem, int token) {
    constexpr int BUF_CH = kStTile * kGateMaxChunks;  // 16-byte chunks per candidate buffer
    float(*red)[kMaxCand] = reinterpret_cast<float(*)[kMaxCand]>(smem + 2 * BUF_CH);  // per-wave candidate sums
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: scale fields index by it
    const int wi = wave >> 1, wj = wave & 1;
    const int group = i0 / 256;
    // the gated tensor this tile's rows belong to (uniform per block)
    int g = 0;
#pragma unroll
    for (int q = 1; q < kMaxSets; ++q)
        if (q < p.cg.nsets && j0 >= p.cg.set_j0[q]) g = q;
    const CandSet& cs = p.cg.sets[g];
    const int jl0 = j0 - p.cg.set_j0[g];                 // first row within the tensor
    const int jn = p.cg.set_j0[g + 1] - p.cg.set_j0[g];  // the tensor's rows
    const int64_t rg = cs.row_groups;
    // candidate-independent sums of each 16 values; a quarter of the values stays in
    // the VGPRs the main loop's fragments had, the rest are read per candidate
    float sv[2][8], kept[4][16];
#pragma unroll
    for (int a4 = 0; a4 < 2; ++a4)
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            float t = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float x = st_acc(token, 4 * a4 + (r >> 2), b, r & 3);
                t += x;
                if (a4 == 0 && b < 4) kept[b & 3][r] = x;
            }
            st_pin(token, t);
            sv[a4][b] = t;
        }
    st_gate_stage(smem, cs.qbytes[0], cs.qtype[0], rg, jl0, group, jn);
    for (int k = 0; k < cs.ncand; ++k) {
        // this wave's direct-to-LDS copies of candidate k have landed, then
        // everyone's have; buffer (k+1) % 2 is no longer read
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
        if (k + 1 < cs.ncand)
            st_gate_stage(smem + ((k + 1) & 1) * BUF_CH, cs.qbytes[k + 1], cs.qtype[k + 1], rg,
                                                jl0, group, jn);
        const uint8_t* buf = reinterpret_cast<const uint8_t*>(smem + (k & 1) * BUF_CH);
        const int qt = cs.qtype[k];
        float sum;
        switch (qt) {
        case Q8_0: sum = st_gate_dot<Q8_0>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
        case Q2_K: sum = st_gate_dot<Q2_K>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
        case Q3_K: sum = st_gate_dot<Q3_K>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
        case Q4_K: sum = st_gate_dot<Q4_K>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
        case Q5_K: sum = st_gate_dot<Q5_K>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
        case Q6_K: sum = st_gate_dot<Q6_K>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
        default:
            sum = 0.0f;
            if constexpr (IQ) {
                switch (qt) {
                case IQ2_XXS: sum = st_gate_dot<IQ2_XXS>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
                case IQ2_XS: sum = st_gate_dot<IQ2_XS>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
                case IQ2_S: sum = st_gate_dot<IQ2_S>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
                case IQ3_XXS: sum = st_gate_dot<IQ3_XXS>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
                case IQ3_S: sum = st_gate_dot<IQ3_S>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
                case IQ1_S: sum = st_gate_dot<IQ1_S>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
                case IQ1_M: sum = st_gate_dot<IQ1_M>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
                case IQ4_XS: sum = st_gate_dot<IQ4_XS>(token, sv, kept, buf, rg, jl0, group, wi, wj, lane, jn); break;
                default: break;
                }
            }
            break;
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off);
        if (lane == 0) red[wave][k] = sum;
    }
    __syncthreads();
    // this block's slots of every tensor: its own sums, zeros for the others
    const int nslot = p.cg.nsets * p.cg.kstride;
    if ((int)threadIdx.x < nslot) {
        const int k = (int)threadIdx.x - g * p.cg.kstride;
        float s = 0.0f;
        if (k >= 0 && k < cs.ncand)
            for (int wv = 0; wv < 4; ++wv) s += red[wv][k];
        p.partials[(int64_t)block * nslot + threadIdx.x] = s;
    }
}

// ---------------------------------------------------------------- kernels
// Work item `block`, alone: the copies past its end are zeros.
template <class C, bool IQ = false>
__device__ __forceinline__ void st_body(const GemmParams& p, int block, u32x4* __restrict__ smem) {
#if defined(__HIP_DEVICE_COMPILE__)
    const StTile t = C::item(p, block);
    if (!t.live) {
        if constexpr (C::EPI == EPI_GATE) {
            const int nslot = p.cg.nsets * p.cg.kstride;
            if ((int)threadIdx.x < nslot) p.partials[(int64_t)block * nslot + threadIdx.x] = 0.0f;
        }
        return;
    }
    Stream<C::LA, C::LB> st;
    st.template start<false>(p, t, smem);
    st.template tile<false>(p, t, st_tile(0, 0, 0, 0, false), false);
    int token = st_accumulators_ready();
    if constexpr (C::EPI == EPI_STORE) {
        if (t.ns > 1)
            st_store_part(p.partials + ((int64_t)t.tail_slot * p.s_max + t.split) * (kStTile * kStTile), token);
        else
            st_store_tile(p, t, smem, token, false);
        wait_vmcnt_barrier<0>();  // the zero copies have landed before the LDS is given back
    } else if constexpr (C::EPI == EPI_PARTS) {
        // 16 consecutive i per lane: four 16-byte stores, four lanes per 256-byte row piece
        const int tid = fresh_tid();
        const int lane = tid & 63, wave = tid >> 6;
        const int ti = t.i0 / kStTile, tj = t.j0 / kStTile, tiles_j = (p.J + kStTile - 1) / kStTile;
        float* slot = p.dwp + ((int64_t)(ti * tiles_j + tj) * p.parts + t.split) * (kStTile * kStTile);
#pragma unroll
        for (int b = 0; b < 8; ++b)
#pragma unroll
            for (int a4 = 0; a4 < 2; ++a4) {
                __builtin_amdgcn_sched_barrier(0);
                float4* o = reinterpret_cast<float4*>(slot + (128 * (wave & 1) + 16 * b + (lane & 15)) * kStTile +
                                                      128 * (wave >> 1) + 64 * a4 + 16 * (lane >> 4));
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    o[q] = make_float4(st_acc(token, 4 * a4 + q, b, 0), st_acc(token, 4 * a4 + q, b, 1),
                                       st_acc(token, 4 * a4 + q, b, 2), st_acc(token, 4 * a4 + q, b, 3));
            }
        wait_vmcnt_barrier<0>();
    } else {
        wait_vmcnt_barrier<0>();  // the zero copies have landed and no wave reads the stages any more
        st_gate_epilogue<IQ>(p, block, t.i0, t.j0, smem, token);
    }
#endif
}

template <class C, bool IQ = false>
__global__ __launch_bounds__(kStThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
void st_gemm_kernel(GemmParams p) {
    extern __shared__ u32x4 smem[];
    st_body<C, IQ>(p, blockIdx.x, smem);
}

// A store product as one stream per workgroup: `wgs` workgroups per XCD walk
// its work items (block, block + 8 wgs, ...), each tile's last stages already
// copying the next tile's first ones and its stores left behind in flight.
// The K-split parts, if any, come last (one per workgroup).
template <class C>
__global__ __launch_bounds__(kStThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
void st_persist_kernel(GemmParams p, int wgs) {
#if defined(__HIP_DEVICE_COMPILE__)
    extern __shared__ u32x4 smem[];
    int block = blockIdx.x;
    StTile cur = C::item(p, block);
    if (!cur.live) return;
    Stream<C::LA, C::LB> st;
    st.template start<false>(p, cur, smem);
    bool stores = false;
    for (;;) {
        block += 8 * wgs;
        const StTile nxt = C::item(p, block);
        st.template tile<false>(p, cur, nxt, stores);
        int token = st_accumulators_ready();
        if (cur.ns > 1) {
            st_store_part(p.partials + ((int64_t)cur.tail_slot * p.s_max + cur.split) * (kStTile * kStTile), token);
            break;
        }
        st_store_tile(p, cur, smem, token, false);
        if (!nxt.live) break;
        __builtin_amdgcn_sched_barrier(0);
        stores = true;
        cur = nxt;
    }
    wait_vmcnt_barrier<0>();  // the copies past the end have landed before the LDS is given back
#endif
}

// Two independent products in one launch: blocks [0, n1) run problem 1,
// blocks [n1, ...) problem 2 (n1 is a multiple of 8, so both keep the XCD
// mapping of map_work).  One grid lets the second product's work items fill the
// last, partial round of the first instead of each launch idling CUs in its
// own tail.
template <class C1, class C2, bool IQ1>
__global__ __launch_bounds__(kStThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
void st_dual_kernel(GemmParams p1, int n1, GemmParams p2) {
    extern __shared__ u32x4 smem[];
    const int b = blockIdx.x;
    if (b < n1)
        st_body<C1, IQ1>(p1, b, smem);
    else
        st_body<C2, false>(p2, b - n1, smem);
}

// Sum of the K parts of each split tail tile, in part order, rounded to bf16
// into C.  One block per (XCD tail slot, accumulator row a): a thread takes
// fragment row a's 32 values.
template <class C>
__global__ __launch_bounds__(kStThreads) void st_fixup_kernel(GemmParams p) {
    constexpr int TILE = kStTile * kStTile;
    const int slot = blockIdx.x / 16, a4 = (blockIdx.x / 8) % 2, b = blockIdx.x % 8;
    const int x = slot / p.tail_max, tt = slot % p.tail_max;
    const int ti = (p.I + kStTile - 1) / kStTile, tj = (p.J + kStTile - 1) / kStTile;
    const XcdPlan pl = xcd_plan(x, ti * tj, p.cus_per_xcd, C::ksteps(p), p.split_ok != 0, p.split_min_saved, p.split_max);
    if (tt >= pl.tail) return;
    int tm, tn;
    tile_coords(pl.t0 + pl.full + tt, tj, ti, kGroupM, tm, tn);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float* base = p.partials + (int64_t)slot * p.s_max * TILE + threadIdx.x;
    // elements 32 (4 a4 + q) + 4 b + r: 16 consecutive i
    auto at = [&](int sp, int e) { return base[(int64_t)sp * TILE + (32 * (4 * a4 + (e >> 2)) + 4 * b + (e & 3)) * kStThreads]; };
    float v[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = at(0, e);
#pragma unroll
    for (int sp = 1; sp < 8; ++sp) {
        if (sp < pl.s) {
            float t[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) t[e] = at(sp, e);
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] += t[e];
        }
    }
    const int gj = tm * kStTile + 128 * (wave & 1) + 16 * b + (lane & 15);
    const int gi = tn * kStTile + 128 * (wave >> 1) + 64 * a4 + 16 * (lane >> 4);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        if (gj < p.J && gi + 8 * c < p.I) {
            u32x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = f2bf2(v[8 * c + 2 * e], v[8 * c + 2 * e + 1]);
            *reinterpret_cast<u32x4*>(p.C + (int64_t)gj * p.ldc + gi + 8 * c) = w;
        }
    }
}

template <class C>
static hipError_t launch_st_fixup(const GemmParams& p, hipStream_t s) {
    st_fixup_kernel<C><<<dim3(8 * p.tail_max * 16), dim3(kStThreads), 0, s>>>(p);
    return hipGetLastError();
}

// A store product.  `cus` is the device's CU count; tail tiles are split only
// when `tail_ws` (tail_bytes of the plan) is given.
template <class C>
static hipError_t launch_st_store(GemmParams p, int cus, float* tail_ws, hipStream_t s) {
    static_assert(C::EPI == EPI_STORE, "a store product");
    const int grid = C::plan(p, cus, tail_ws != nullptr);
    if (grid == 0) return hipSuccess;
    p.partials = tail_ws;
    static bool attr_set = false;  // per instantiation
    auto kern = st_persist_kernel<C>;
    hipError_t e = set_lds_attr<C>((const void*)kern, C::lds(), attr_set);
    if (e != hipSuccess) return e;
    const int wgs = grid / 8 < p.cus_per_xcd ? grid / 8 : p.cus_per_xcd;
    kern<<<dim3(8 * wgs), dim3(kStThreads), C::lds(), s>>>(p, wgs);
    e = hipGetLastError();
    if (e != hipSuccess || p.tail_max == 0) return e;
    return launch_st_fixup<C>(p, s);
}

// A gate product alone.
template <class C, bool IQ>
static hipError_t launch_st_gate(GemmParams p, int cus, hipStream_t s) {
    const int grid = C::plan(p, cus, true);
    if (grid == 0) return hipSuccess;
    static bool attr_set = false;
    auto kern = st_gemm_kernel<C, IQ>;
    hipError_t e = set_lds_attr<C>((const void*)kern, C::lds(), attr_set);
    if (e != hipSuccess) return e;
    kern<<<dim3(grid), dim3(kStThreads), C::lds(), s>>>(p);
    return hipGetLastError();
}

// Two products in one launch (see st_dual_kernel): problem 1, a store product
// with split tails (tail_ws1), and problem 2, a gate product.  The gate
// product's work items come first and the store product's fill the tail (its
// split parts are fixed up after the launch).
template <class C1, class C2, bool IQ2>
static hipError_t launch_st_dual(GemmParams p1, GemmParams p2, int cus, float* tail_ws1, hipStream_t s) {
    static_assert(C1::EPI == EPI_STORE && C2::EPI != EPI_STORE, "a store product and a gate product");
    const int grid1 = C1::plan(p1, cus, tail_ws1 != nullptr);
    const int grid2 = C2::plan(p2, cus, true);
    p1.partials = tail_ws1;
    if (grid1 == 0) return launch_st_gate<C2, IQ2>(p2, cus, s);
    if (grid2 == 0) return launch_st_store<C1>(p1, cus, tail_ws1, s);
    constexpr size_t lds = C1::lds() > C2::lds() ? C1::lds() : C2::lds();
    static bool attr_set = false;
    auto kern = st_dual_kernel<C2, C1, IQ2>;
    hipError_t e = set_lds_attr<C2>((const void*)kern, lds, attr_set);
    if (e != hipSuccess) return e;
    kern<<<dim3(grid2 + grid1), dim3(kStThreads), lds, s>>>(p2, grid2, p1);
    e = hipGetLastError();
    if (e != hipSuccess || p1.tail_max == 0) return e;
    return launch_st_fixup<C1>(p1, s);
}

// ---------------------------------------------------------------- routed product
// Grouped GEMM: C[rowmap[r]] = B[rowmap[r]] . bk[g]^T for the rows r of each
// group g (group_off on the device, so the host never waits for the counts).
// The grid covers ceil(m / 256) + ngroups - 1 tile-rows, the most the groups can
// need; every block counts the tile-rows the groups do need, takes its tile of
// those (the XCDs get even contiguous ranges, the spare blocks spread over all
// of them) and finds the tile's group by walking the group sizes.
__global__ __launch_bounds__(kStThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
void st_routed_kernel(GemmParams p, int tile_rows) {
#if defined(__HIP_DEVICE_COMPILE__)
    extern __shared__ u32x4 smem[];
    const int tiles_i = (p.I + kStTile - 1) / kStTile;
    // group bounds clamped to [0, map_rows] and made monotonic, so bad
    // offsets cannot index rowmap out of range; the work is spread over the
    // tile-rows the groups actually have (the grid covers the most they can)
    int used_rows = 0;
    for (int g = 0, h = 0; g < p.ngroups; ++g) {
        const int l = min(max(p.group_off[g], h), p.map_rows);
        h = min(max(p.group_off[g + 1], l), p.map_rows);
        used_rows += (h - l + kStTile - 1) / kStTile;
    }
    used_rows = min(used_rows, tile_rows);
    // the XCDs take contiguous ranges of the tiles (as in map_work); the tiles
    // run group by group, each group's tile-rows in blocks of kGroupM with the
    // tile-rows fastest, so the tiles an XCD runs at once read one candidate's
    // weight panels and share them in its L2
    const int x = blockIdx.x % 8, local = blockIdx.x / 8;
    const XcdPlan pl = xcd_plan(x, used_rows * tiles_i, p.cus_per_xcd, 0, false);
    if (local >= pl.items()) return;
    int tile = pl.t0 + local, tm = 0, tn = 0, g = 0, lo = 0, hi = 0;
    for (; g < p.ngroups; ++g) {
        lo = min(max(p.group_off[g], hi), p.map_rows);
        hi = min(max(p.group_off[g + 1], lo), p.map_rows);
        const int nt = (hi - lo + kStTile - 1) / kStTile;
        if (tile < nt * tiles_i) {
            tile_coords(tile, nt, tiles_i, kGroupM, tm, tn);
            break;
        }
        tile -= nt * tiles_i;
    }
    if (g >= p.ngroups) return;
    GemmParams q = p;
    q.A = p.bk[g];
    q.J = hi;  // end of the group's rows in rowmap
    const StTile t = st_tile(tn * kStTile, lo + tm * kStTile, 0, q.K, true);
    Stream<KS, KS> st;
    st.template start<true>(q, t, smem);
    st.template tile<true>(q, t, st_tile(0, 0, 0, 0, false), false);
    int token = st_accumulators_ready();
    st_store_tile(q, t, smem, token, true);
    wait_vmcnt_barrier<0>();  // the zero copies have landed before the LDS is given back
#endif
}

static hipError_t launch_st_routed(GemmParams p, int m, int cus, hipStream_t s) {
    if (m <= 0 || p.I <= 0 || p.ngroups <= 0) return hipSuccess;
    const int tile_rows = (m + kStTile - 1) / kStTile + p.ngroups - 1;
    const int tiles = tile_rows * ((p.I + kStTile - 1) / kStTile);
    p.cus_per_xcd = cus / 8 > 0 ? cus / 8 : 1;
    p.split_ok = 0;
    int items = 0;
    for (int x = 0; x < 8; ++x) {
        const XcdPlan pl = xcd_plan(x, tiles, p.cus_per_xcd, 0, false);
        items = pl.items() > items ? pl.items() : items;
    }
    static bool attr_set = false;
    hipError_t e = set_lds_attr<StCfg<KS, KS, EPI_STORE>>((const void*)st_routed_kernel, kStStoreLds, attr_set);
    if (e != hipSuccess) return e;
    st_routed_kernel<<<dim3(8 * items), dim3(kStThreads), kStStoreLds, s>>>(p, tile_rows);
    return hipGetLastError();
}

}  // namespace vq
