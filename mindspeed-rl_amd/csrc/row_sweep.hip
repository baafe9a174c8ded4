// Row-in-registers vocabulary sweeps for gfx950.
//
// A workgroup owns one logits row (of the shortest rows, up to four side by side) and keeps ALL of it in registers:
// 256 threads for the shortest rows, several workgroups per CU, up to 1024 threads with 19 16-byte vectors each = 311 296 bytes, one per CU,
// enough for a 152 064-entry bf16 row.  The softmax statistics are taken vector by vector as the data
// arrives, the token's loss gradient follows from them, and dlogits are written from the same registers -
// one HBM read and one HBM write per element for the whole forward + backward of the log-prob /
// policy-loss path.  The requests of a row are issued together (the HBM system serves a row best
// that way) and all accesses are range-checked buffer accesses, so the unrolled bodies contain no
// branch (see mrl_internal.h for why that matters).
//
// fused_sweep_persistent_kernel launches as many workgroups as the chip holds; they take rows in ticket
// order and request the next row while they write the current one.  bwd_chunk_kernel is the split path's
// backward (upstream gradients and the log-sum-exp are inputs, so there is no statistics pass and nothing
// has to stay on chip): a plain stream of one vector per thread.
#include <atomic>

#include "lane_ops.h"
#include "mrl_internal.h"
#include "policy_terms.h"
#include "row_sweep.h"
#include "vocab_common.h"

namespace {

using namespace mrl_vocab;
using namespace mrl_loss;
using mrl::lane_value;
using mrl::lanes_max;
using mrl::lanes_sum;

// Vectors of the next row that are requested early (see fused_sweep_persistent_kernel); build-time
// tuning constants, measured on the 152064-entry bf16 row.  The fused sweep gains 4 % from an early
// burst of 4: its statistics pass then starts without waiting for memory.
#ifndef MRL_SWEEP_HEAD
#define MRL_SWEEP_HEAD 4
#endif
// Workgroup size of the streaming backward (bwd_chunk_kernel): 256 measured best (64: +2 %, 128:
// +14 %, 1024: +8 % in time).
#ifndef MRL_BWD_CHUNK_THREADS
#define MRL_BWD_CHUNK_THREADS 256
#endif

// Two-level reduction for the BLK / 64 wavefronts that hold a row: the largest reference first, so that a part is
// rescaled once and the rest is sums; inside a wavefront over its 4 rows of 16 lanes and these through scalar
// registers, then every wavefront combines the BLK / 64 partials for itself.  It is a serial chain in which the
// workgroup neither computes on its row nor writes it; before, it went through shuffles with a rescale in every step
// and a second barrier.  us a sweep, before -> now, where memory does not hide it: 12 926 x 32 003 bf16 300 ->
// 291, 2 367 x 32 000 fp32 109.5 -> 107.7 (108.3 -> 104.9 without entropy), 16 384 x 72 608 bf16 847 -> 835, x
// 100 352 1 114 -> 1 099; the other shapes are at what memory gives (129 280 and 152 064 bf16, short rows) and
// within 0.6 %.
// lds: BLK / 64 entries of this row that nothing else touches until the workgroup has passed another barrier.  Every
// wavefront of the workgroup comes here.
template <int BLK, bool kEntropy>
__device__ __forceinline__ Stats reduce_row(Stats st, float k, Stats* lds, int tid) {
    constexpr int kWaves = BLK / 64;
    constexpr int kSteps = kWaves == 16 ? 4 : (kWaves == 8 ? 3 : 2);
    static_assert(kWaves == 4 || kWaves == 8 || kWaves == 16, "partials of 4, 8 or 16 wavefronts");
    const float m16 = lanes_max<4>(st.m);
    Stats t;
    t.m = fmaxf(fmaxf(lane_value(m16, 0), lane_value(m16, 16)), fmaxf(lane_value(m16, 32), lane_value(m16, 48)));
    const float f = fast_exp2((st.m - t.m) * k);
    const float s16 = lanes_sum<4>(st.s * f);
    t.s = (lane_value(s16, 0) + lane_value(s16, 16)) + (lane_value(s16, 32) + lane_value(s16, 48));
    t.u = 0.f;
    if (kEntropy) {
        const float u16 = lanes_sum<4>(st.u * f);
        t.u = (lane_value(u16, 0) + lane_value(u16, 16)) + (lane_value(u16, 32) + lane_value(u16, 48));
    }
    const int wave = tid >> 6, lane = tid & 63;
    if (lane == 0) lds[wave] = t;
    // LDS accesses only, as in broadcast_ticket
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    const Stats x = lds[lane & (kWaves - 1)];
    const float m = lanes_max<kSteps>(x.m);
    const float fx = fast_exp2((x.m - m) * k);
    // the same in every lane, which the branches and addresses that follow from it have to be known to be
    Stats r;
    r.m = lane_value(m, 0);
    r.s = lane_value(lanes_sum<kSteps>(x.s * fx), 0);
    r.u = kEntropy ? lane_value(lanes_sum<kSteps>(x.u * fx), 0) : 0.f;
    return r;
}

__device__ __forceinline__ int64_t load_label(const void* labels, int dtype, int64_t r) {
    return dtype == MRL_I32 ? (int64_t) reinterpret_cast<const int32_t*>(labels)[r]
                            : reinterpret_cast<const int64_t*>(labels)[r];
}

struct RowGrad {
    float k;        // inv_t * log2(e)
    float lse2;     // lse * log2(e)
    float c0, c1;   // dlogit = 2^(z k - lse2) * (c0 + c1 z)
    float onehot;   // added at the label
};

template <bool kEntropy>
__device__ __forceinline__ float grad_elem(const RowGrad& g, float z) {
    const float e = fast_exp2(__builtin_fmaf(z, g.k, -g.lse2));
    const float w = kEntropy ? __builtin_fmaf(g.c1, z, g.c0) : g.c0;
    return e * w;
}

// The shapes of a workgroup that holds a row, shortest rows first: threads, vectors a thread, and the longest row
// that it is taken for in vectors of fp32 and of 16-bit logits (0: none).  Why the lines lie there: see pick_shape.
struct RowShape {
    int threads, vectors;
    int64_t most_f32, most_16;
    constexpr int64_t most(int dtype) const { return dtype == MRL_F32 ? most_f32 : most_16; }
};
constexpr int64_t kMaxVec = 19 * 1024;              // vectors of the widest row that one workgroup holds
constexpr int64_t kMinHalf = (kMaxVec + 1) / 2;     // of the shorter half of a wider one
constexpr RowShape kRowShapes[] = {
    {256, 4, 1024, 1024},      {256, 8, 2048, 2048},      {256, 12, 2496, 3072},     {512, 8, 4096, 4096},
    {512, 12, 0, 6144},        {512, 16, 0, 8192},        {1024, 8, 8192, 0},        {1024, 10, 10240, 10240},
    {1024, 12, 12288, 12288},  {1024, 14, 14336, 14336},  {1024, 16, 16384, 16384},  {1024, 19, kMaxVec, kMaxVec},
};
constexpr int kShapes = sizeof(kRowShapes) / sizeof(kRowShapes[0]);

// Rows that are held side by side (see pick_rows), each by 256 threads: how many, vectors a thread, and the row lengths in
// vectors, longer than `above` and up to `most` (0: none).
struct SideShape {
    int rows, vectors;
    int64_t above_f32, most_f32, above_16, most_16;
    constexpr int64_t above(int dtype) const { return dtype == MRL_F32 ? above_f32 : above_16; }
    constexpr int64_t most(int dtype) const { return dtype == MRL_F32 ? most_f32 : most_16; }
};
constexpr int kSideThreads = 256;
constexpr SideShape kSideShapes[] = {
    {4, 4, 512, 1024, 928, 1024}, {2, 7, 0, 0, 1312, 1792},  {4, 8, 1024, 2048, 0, 0},
    {2, 8, 0, 0, 1792, 2048},     {2, 10, 0, 0, 2048, 2560}, {4, 12, 2048, 2496, 0, 0},
};
constexpr int kSides = sizeof(kSideShapes) / sizeof(kSideShapes[0]);

// Vectors of a thread that are complete in every row that the tables give to a workgroup of BLK threads with NV vectors
// each; the later ones may be partly or wholly past the end of the row.  A row with edges has up to 8 vectors less than
// its length suggests.
constexpr int complete_vectors(int threads, int vectors, bool edge) {
    int64_t least = kMaxVec + 1;
    for (int dtype : {MRL_F32, MRL_BF16}) {
        int64_t before = 0;                         // the longest row of a smaller shape
        for (const RowShape& s : kRowShapes) {
            const int64_t most = s.most(dtype);
            if (most == 0) continue;
            if (s.threads == threads && s.vectors == vectors) {
                if (before + 1 < least) least = before + 1;
                // halves of wide rows: the shorter one may be a vector less than the one that the shape follows from
                const int64_t half = before > kMinHalf ? before : kMinHalf;
                if (most > kMinHalf && half < least) least = half;
            }
            before = most;
        }
        for (const SideShape& s : kSideShapes)
            if (threads == kSideThreads && s.vectors == vectors && s.most(dtype) != 0 && s.above(dtype) + 1 < least)
                least = s.above(dtype) + 1;
    }
    if (edge) least -= 8;
    return least < threads ? 0 : (int)(least / threads);
}

template <int BLK, int NV, bool kEdge>
struct Tail {
    static constexpr int kFull = complete_vectors(BLK, NV, kEdge);
    static_assert(kFull <= NV, "no row of this many threads and vectors is in the tables");
};

// Vector q of a row is addressed through a descriptor of its own (the row from byte q * 16 * BLK on,
// clamped to empty) with the same per-thread byte offset for every q: the descriptors live in
// scalar registers and cost scalar instructions, where one vector offset per q would cost 19
// vector registers that the row itself needs.
struct RowRef {
    const char* base;   // uniform over the workgroup
    uint32_t bytes;     // 0: nothing is read (loads return zeros) or written
};

__device__ __forceinline__ RowRef row_ref(const void* base, uint32_t bytes) {
    RowRef r = {reinterpret_cast<const char*>(base), bytes};
    return r;
}

template <int BLK>
__device__ __forceinline__ mrl::rsrc_t vec_rsrc(const RowRef& row, int q) {
    // signed arithmetic on purpose: an unsigned saturating subtraction is selected as a VECTOR
    // instruction, which would make the descriptor non-uniform
    const int skip = q * (BLK * 16);
    const int rest = (int)row.bytes - skip;
    return mrl::make_rsrc(row.base + skip, (uint32_t)(rest > 0 ? rest : 0));
}

// Keeps the instruction scheduler from moving work of one vector across the work of the next: in
// a fully unrolled, branch-free body it would otherwise unpack many vectors ahead of their use and
// spill the row.
__device__ __forceinline__ void vector_fence() { __builtin_amdgcn_sched_barrier(0); }

__device__ __forceinline__ uint32_t lane_offset(int tid) { return (uint32_t)tid * 16u; }

// Vectors [A, B) of a row: loads (back to back and without a branch: vectors past the end of the row come
// back as zeros from the range check of the buffer access), zero stores.
template <int BLK, int A, int B, int NV>
__device__ __forceinline__ void load_part(u32x4 (&v)[NV], const RowRef& src, int tid) {
#pragma unroll
    for (int q = A; q < B; ++q) {
        v[q] = mrl::buf_load_nt(vec_rsrc<BLK>(src, q), lane_offset(tid));
        vector_fence();     // keeps the requests in this order wherever a row is loaded
    }
}

template <int BLK, int A, int B>
__device__ __forceinline__ void zero_part(const RowRef& dst, int tid) {
    const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int q = A; q < B; ++q) {
        mrl::buf_store_nt(zero, vec_rsrc<BLK>(dst, q), lane_offset(tid));
        vector_fence();
    }
}

// Online-softmax statistics of the vectors one thread holds, the careful way: the running maximum is
// brought up to date before every vector, so the exponentials never exceed 1 whatever the logits are
// (infinities and NaN included).  A vector past the end of the row (zeros from the range-checked load)
// is processed like any other and its result discarded, which costs three selects on the few vectors
// that can be affected and keeps the pass free of branches.
template <int DT, int BLK, int NV, bool kEntropy, bool kEdge>
__device__ __forceinline__ Stats thread_stats_careful(const u32x4 (&v)[NV], int n_vec, float k, int tid) {
    using E = Elem<DT>;
    constexpr int kVec = E::kVec;
    Stats st = {kMaxInit, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        // through an empty asm statement, as in grad_vec: entries that another pass has unpacked
        // must not be kept for this one
        u32x4 x = v[q];
        asm volatile("" : "+v"(x));
        float z[kVec];
        E::unpack(x, z);
        Stats nx = st;
        float vmax = nx.m;
#pragma unroll
        for (int i = 0; i < kVec; ++i) vmax = fmaxf(vmax, z[i]);
        grow_max<kEntropy>(nx, vmax, k);
        const float mk = nx.m * k;
#pragma unroll
        for (int i = 0; i < kVec; ++i) add_one<kEntropy>(nx, z[i], k, mk);
        if (q >= Tail<BLK, NV, kEdge>::kFull) {
            const bool valid = q * BLK + tid < n_vec;
            st.m = valid ? nx.m : st.m;
            st.s = valid ? nx.s : st.s;
            st.u = valid ? nx.u : st.u;
        } else {
            st = nx;
        }
        // pins the running statistics here: without it the scheduler splits the whole unrolled pass
        // into one chain per statistic and parks every exponential in scratch memory in between
        asm volatile("" : "+v"(st.m), "+v"(st.s), "+v"(st.u));
    }
    return st;
}

// A thread's sums may be taken against any reference value in place of the running maximum, as long
// as no exponential overflows: the result (m, s, u) then simply carries that reference as its m, and
// every later merge treats it like a maximum.  An entry of the row is a safe reference from below
// (the largest entry then contributes at least 1), and for ordinary logits it is within a few units
// of the maximum, so nothing comes near the 2^127 an fp32 holds.  Taking the largest entry of the
// thread's first vector saves the maximum over every vector and the rescale that follows it - a
// quarter of the arithmetic of the pass.  If a sum does end up beyond 2^90, infinite or NaN (logits
// that climb by more than 62 above that entry, infinities, NaN), the thread takes its statistics
// once more, carefully.  Which way a thread went depends only on its own entries.
//
// The limit is what the reduction below can bring to another reference.  A reference that lies 126 or
// more powers of two under the largest one is scaled by a flushed zero, and with it goes up to 2^90 x
// 2^-126 of the row's weight (which is 1 at least) a thread: 2^-26 from all 1024 threads, below half
// an ulp.  (With 2^120 it was up to 2^-6 a thread: a logsumexp of 0.003 for 1.336.)  Sums of 1024
// threads against one reference stay below 2^100.  What it costs: rows that climb by 62 to 83, us a
// sweep, 430 -> 447 (4 096 x 152 064 bf16), 175 -> 179 (4 096 x 32 000 fp32), 185 -> 216 (8 192 x 32 000
// bf16), as rows that climb further always did; the others are as before.
constexpr float kSumLimit = 1.2379400392853803e27f;     // 2^90

template <int DT, bool kEntropy>
__device__ __forceinline__ void add_vector(const u32x4& vec, float k, float rk, float& s, float& u) {
    using E = Elem<DT>;
    constexpr int kVec = E::kVec;
    float z[kVec];
    E::unpack(vec, z);
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
        const float e = fast_exp2(__builtin_fmaf(z[i], k, -rk));
        s += e;
        if (kEntropy) u = __builtin_fmaf(e, z[i], u);
    }
}

template <int DT>
__device__ __forceinline__ float vector_max(const u32x4& vec) {
    using E = Elem<DT>;
    constexpr int kVec = E::kVec;
    float z[kVec];
    E::unpack(vec, z);
    float r = z[0];
#pragma unroll
    for (int i = 1; i < kVec; ++i) r = fmaxf(r, z[i]);
    return r;
}

// want_max (uniform over the workgroup): the caller needs the true maximum of the row in m (a label
// outside the vocabulary scores the row maximum), which only the careful pass delivers.
// kEdge: the thread also holds one entry of the row outside its vectors, z_edge, if has_edge.
template <int DT, int BLK, int NV, bool kEntropy, bool kEdge>
__device__ __forceinline__ Stats thread_stats(const u32x4 (&v)[NV], int n_vec, float k, bool want_max, bool has_edge,
                                              float z_edge, int tid) {
    Stats st = {kMaxInit, 0.f, 0.f};
    // in a row so short that a thread may hold no complete vector there is no reference to take
    bool careful = (Tail<BLK, NV, kEdge>::kFull == 0 && n_vec < BLK) || want_max;
    if (!careful) {
        st.m = vector_max<DT>(v[0]);
        const float rk = st.m * k;
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            if (q < Tail<BLK, NV, kEdge>::kFull) {
                add_vector<DT, kEntropy>(v[q], k, rk, st.s, st.u);
            } else if (q * BLK < n_vec) {               // uniform: nothing to compute past the end of the row
                float s = st.s, u = st.u;
                add_vector<DT, kEntropy>(v[q], k, rk, s, u);
                const bool valid = q * BLK + tid < n_vec;
                st.s = valid ? s : st.s;
                st.u = valid ? u : st.u;
            }
            asm volatile("" : "+v"(st.s), "+v"(st.u));       // as in the careful pass
            // nothing but the two sums links one vector to the next here, so the scheduler would
            // unpack many vectors ahead of their use; keep each vector's work together
            vector_fence();
        }
        if (kEdge) {
            const float e = fast_exp2(__builtin_fmaf(z_edge, k, -rk));
            st.s = has_edge ? st.s + e : st.s;
            if (kEntropy) st.u = has_edge ? __builtin_fmaf(e, z_edge, st.u) : st.u;
        }
        careful = !(st.s < kSumLimit);
    }
    if (careful) {
        st = thread_stats_careful<DT, BLK, NV, kEntropy, kEdge>(v, n_vec, k, tid);
        if (kEdge && has_edge) {
            grow_max<kEntropy>(st, z_edge, k);
            add_one<kEntropy>(st, z_edge, k, st.m * k);
        }
    }
    return st;
}

template <int DT, bool kEntropy>
__device__ __forceinline__ u32x4 grad_vec(const u32x4& v, const RowGrad& g) {
    using E = Elem<DT>;
    constexpr int kVec = E::kVec;
    // The packed vector is passed through an empty asm statement so that the compiler cannot reuse
    // the unpacked values of the statistics pass: kept alive across both passes they would be a
    // second, four times larger copy of the row, and spill.
    u32x4 x = v;
    asm volatile("" : "+v"(x));
    float z[kVec], d[kVec];
    E::unpack(x, z);
#pragma unroll
    for (int i = 0; i < kVec; ++i) d[i] = grad_elem<kEntropy>(g, z[i]);
    return E::pack(d);
}

// dlogits of vectors [A, B) of the row in registers, stored as they are computed.
template <int DT, int BLK, bool kEntropy, int A, int B, int NV>
__device__ __forceinline__ void grad_part(const u32x4 (&v)[NV], const RowGrad& g, const RowRef& dst, int tid) {
#pragma unroll
    for (int q = A; q < B; ++q) {
        mrl::buf_store_nt(grad_vec<DT, kEntropy>(v[q], g), vec_rsrc<BLK>(dst, q), lane_offset(tid));
        vector_fence();
    }
}

// Rows that do not all start on a 128-byte line: `head` entries before the first line, n_vec 16-byte vectors
// from there, the rest behind them.  The entries outside the vectors ("edge": at most 63 + 7) go to the first
// threads, one each, through accesses of a single entry; the vectors are accessed like those of an aligned
// row.  16-byte alignment would do for the accesses, but then every wavefront's 1 KiB cuts two lines in
// half: 32 003 bf16 logits 4 958 GB/s, on lines 5 433; 129 288 5 334 -> 5 901; 50 260 fp32 5 580 -> 6 095
// (what rows of 32 000, 129 280 and 50 304 reach).
struct RowSpan {
    int head, n_vec;
};
constexpr int kEdgeAlign = 128;

template <int DT>
__device__ __forceinline__ RowSpan row_span(const typename Elem<DT>::T* row, int vocab) {
    constexpr int kVec = Elem<DT>::kVec;
    const int mis = (int)((reinterpret_cast<uintptr_t>(row) % kEdgeAlign) / sizeof(typename Elem<DT>::T));
    RowSpan s;
    s.head = mis ? kEdgeAlign / (int)sizeof(typename Elem<DT>::T) - mis : 0;
    s.n_vec = (vocab - s.head) / kVec;
    return s;
}

// Byte offset inside the row of this thread's edge entry, out of range for a thread without one.
template <int DT>
__device__ __forceinline__ uint32_t edge_offset(const RowSpan& s, int vocab, int tid) {
    constexpr int kVec = Elem<DT>::kVec;
    const int j = tid < s.head ? tid : tid + s.n_vec * kVec;
    return j < vocab ? (uint32_t)j * (uint32_t)sizeof(typename Elem<DT>::T) : 0x80000000u;
}

// The label's entry gets the one-hot term on top of the softmax term.  The thread that has just
// stored the entry re-stores it; for every other thread the byte offset is out of range and the hardware
// drops the store, so there is no branch here either.  Two stores of one thread to the same address stay
// in program order.  y and dst (of `bytes` bytes) are relative to the unit; span: its vectors.
template <int DT, int BLK, bool kEntropy, bool kEdge>
__device__ __forceinline__ void store_label_grad(const typename Elem<DT>::T* dst, uint32_t bytes, const RowSpan& span,
                                                 const RowGrad& g, bool y_ok, int64_t y, float z_y, int tid) {
    using E = Elem<DT>;
    int writer;
    if (kEdge) {
        const int body = (int)y - span.head, n_body = span.n_vec * E::kVec;
        const bool inside = body >= 0 && body < n_body;
        writer = inside ? (body / E::kVec) % BLK : (body < 0 ? (int)y : (int)y - n_body);
    } else {
        writer = (int)((y / E::kVec) % BLK);
    }
    const bool owner = y_ok && writer == tid;
    const uint32_t off = owner ? (uint32_t)y * (uint32_t)sizeof(typename E::T) : 0x80000000u;
    // product and sum in one operation by name, so that every instance of the kernel rounds alike
    const float e = fast_exp2(__builtin_fmaf(z_y, g.k, -g.lse2));
    const float w = kEntropy ? __builtin_fmaf(g.c1, z_y, g.c0) : g.c0;
    E::buf_store(mrl::make_rsrc(dst, bytes), off, __builtin_fmaf(e, w, g.onehot));
}

struct RowScalars {
    float lp, ent;
    Token t;
    float g_lp, g_h;
};

template <bool kEntropy>
__device__ __forceinline__ RowScalars row_scalars(const Stats& tot, float k, float inv_t, bool y_ok, float z_y,
                                                  const float* __restrict__ ops, int has_old, const Params& p,
                                                  float grad_scale, float m, float& lse) {
    RowScalars s;
    lse = (tot.m * k + fast_log2(tot.s)) * kLn2;
    s.lp = (y_ok ? z_y * inv_t : tot.m * inv_t) - lse;
    s.ent = kEntropy ? lse - (tot.u / tot.s) * inv_t : 0.f;
    s.t = token_terms<true>(s.lp, ops[MRL_OP_OLD], has_old != 0, ops[MRL_OP_REF], ops[MRL_OP_ADV], p);
    const float inv_tok = ops[MRL_OP_INVTOK];
    s.g_lp = grad_scale * m * (ops[MRL_OP_WPG] * s.t.d_pg + p.kl_coef * inv_tok * s.t.d_kl);
    s.g_h = kEntropy ? grad_scale * m * (-p.entropy_coeff * inv_tok) : 0.f;
    return s;
}

template <bool kEntropy>
__device__ __forceinline__ RowGrad row_grad(const RowScalars& s, float k, float inv_t, float lse) {
    RowGrad g;
    g.k = k;
    g.lse2 = lse * kLog2e;
    g.c0 = kEntropy ? inv_t * (-s.g_lp + s.g_h * (lse - s.ent)) : -s.g_lp * inv_t;
    g.c1 = kEntropy ? -s.g_h * inv_t * inv_t : 0.f;
    g.onehot = s.g_lp * inv_t;
    return g;
}

__device__ __forceinline__ void write_row_outputs(int64_t r, const RowScalars& s, float m, float* __restrict__ logp,
                                                  float* __restrict__ entropy, float* __restrict__ row_terms) {
    if (logp) logp[r] = s.lp;
    if (entropy) entropy[r] = s.ent;
    float* out = row_terms + r * S_N;
    out[S_PG] = s.t.pg * m;
    out[S_CLIP] = s.t.clipped * m;
    out[S_PPOKL] = s.t.neg_logr * m;
    out[S_KL] = s.t.kl * m;
    out[S_ENT] = s.ent * m;
    out[S_MASK] = m;
    out[6] = 0.f;
    out[7] = 0.f;
}

__device__ __forceinline__ void write_masked_row_outputs(int64_t r, float* __restrict__ logp,
                                                         float* __restrict__ entropy, float* __restrict__ row_terms) {
    if (logp) logp[r] = 0.f;
    if (entropy) entropy[r] = 0.f;
#pragma unroll
    for (int q = 0; q < S_N; ++q) row_terms[r * S_N + q] = 0.f;
}

// Book-keeping of a backward: applied[0], the scale that the gradients carry, becomes u, and u the scale that
// the next sweep starts from (learned, nullable) if it can be one: finite and not zero.
__device__ __forceinline__ void note_scale(float u, float* applied, float* learned) {
    applied[0] = u;
    if (learned && u != 0.f && __builtin_isfinite(u)) *learned = u;
}

// The same by the workgroup that comes here last (one thread of each does): applied[1] counts them and is zero
// again afterwards.  Every workgroup has read applied[0] before it counts itself.
__device__ __forceinline__ void note_scale_last(float u, float* applied, float* learned, uint32_t* rescales) {
    uint32_t* done = reinterpret_cast<uint32_t*>(applied) + 1;
    const uint32_t before = __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (before == gridDim.x - 1) {
        if (rescales) *rescales += 1u;
        note_scale(u, applied, learned);
        __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ------------------------------------------------------------------------------ row tickets
// The persistent kernel hands out rows through a counter: a workgroup that has finished a row takes
// the next unclaimed one.  With a fixed stride (row r, r + grid, ...) the workgroups drift apart and
// the rows in flight spread over a wide stretch of memory; with tickets the rows in flight are always
// the most recent `grid` consecutive ones, which the HBM system serves about a tenth faster.
// The counter is the first four bytes of the caller's workspace and starts at ZERO: a ticket stands for
// `group` consecutive units, workgroup b begins with units b * group .. + group - 1, and the value t that
// the fetch-and-add (of group) returns stands for units t + gridDim.x * group .. + group - 1.  So "reset" means "clear": the workspace is zeroed by whoever prepares the sweep
// (the prepare kernel of the loss, or clear_words_kernel below).
__global__ void clear_words_kernel(unsigned long long* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

// Thread 0 passes its ticket to the workgroup through LDS.  The fences order LDS accesses only and
// the barrier is the bare instruction: __syncthreads() carries a fence over global memory as well,
// which would wait for every outstanding store of the row that was just written.
__device__ __forceinline__ uint32_t broadcast_ticket(uint32_t mine, uint32_t* slot) {
    // every wavefront picks its (unused) result up here, not only the one that passes it on: a
    // result left pending on the other path would make the next fetch-and-add wait for everything
    asm volatile("" : "+v"(mine));
    if (threadIdx.x == 0) *slot = mine;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)*slot);
}

// Every wavefront loads the logit at the label for itself, and in place a wavefront that is through the reduction
// overwrites it with a gradient: so it has arrived in each of them before the reduction's barrier.  It is the youngest
// request of a row, right behind the row's own, and the wait has no cost that shows (152 064 bf16 346.3 and 345.9 us
// per GB without and with it, 32 000 fp32 322.7 and 322.4, 8 000 bf16 344.2 and 344.3).
__device__ __forceinline__ void wait_for_label_logit() { __builtin_amdgcn_s_waitcnt(0x0F70); }     // vmcnt(0)

// ------------------------------------------------------------------------------ wide rows
// A row that does not fit the registers of one CU is cut into two halves that two workgroups hold at
// the same time (units 2 r and 2 r + 1 of the ticket order, so the halves of a row are taken by
// workgroups that ask for work one after the other).  Each workgroup publishes a record of its half
// - its statistics and, if the label lies in it, the logit at the label: 16 bytes in the caller's
// workspace, written and read with device-scope atomics only, so that no cache has to be flushed -
// and picks up the other half's before it computes the row's gradient.  A workgroup publishes BEFORE
// it waits, and nothing it does before publishing depends on another workgroup, so waits cannot form
// a cycle; the wait is bounded all the same: when the limit is reached the workgroup reads the other
// half from memory and computes its statistics itself, with the partner's assignment of vectors to
// threads and the same order of operations, so the result is the partner's to the last bit.
//
// In place (dlogits over the logits) the other half may be overwritten by its owner at any time
// AFTER the owner has published: a workgroup waits until its record has reached memory before any of
// its threads stores a gradient.  A workgroup that had to read the other half therefore looks at the
// record once more afterwards: if it is there now, the record is used and what was read is thrown
// away; if it still is not, the owner had not begun to write, and everything read was logits.
struct HalfRecord {
    unsigned long long ms;      // (m, s): never 0, s >= 1 or NaN
    unsigned long long uz;      // (u, logit at the label if it lies in this half, else 1): never 0
};

__device__ __forceinline__ unsigned long long pack2f(float lo, float hi) {
    return (unsigned long long)__float_as_uint(lo) | ((unsigned long long)__float_as_uint(hi) << 32);
}

// Statistics of a stretch of a row streamed from memory by the whole workgroup (the fallback above):
// thread t takes vectors t, t + 1024, ... in this order, as thread_stats does with the vectors a
// thread holds - the same reference, the same sums, the same second attempt - and the reduction is
// the same.  `whole`: every thread has at least one vector and the row maximum is not asked for (what
// makes thread_stats take the short way).
constexpr int kWideBlock = 1024;        // threads of a workgroup that holds half a row

template <int DT, bool kEntropy>
__device__ __forceinline__ Stats stream_stats(const typename Elem<DT>::T* base, int n_vec, float k, bool whole,
                                              Stats* lds) {
    using E = Elem<DT>;
    constexpr int kVec = E::kVec;
    const u32x4* vec = reinterpret_cast<const u32x4*>(base);
    Stats st = {kMaxInit, 0.f, 0.f};
    bool careful = !whole;
    if (whole) {
        st.m = vector_max<DT>(__builtin_nontemporal_load(vec + threadIdx.x));
        const float rk = st.m * k;
        for (int idx = threadIdx.x; idx < n_vec; idx += kWideBlock)
            add_vector<DT, kEntropy>(__builtin_nontemporal_load(vec + idx), k, rk, st.s, st.u);
        careful = !(st.s < kSumLimit);
    }
    if (careful) {
        st = {kMaxInit, 0.f, 0.f};
        for (int idx = threadIdx.x; idx < n_vec; idx += kWideBlock) {
            float z[kVec];
            E::unpack(__builtin_nontemporal_load(vec + idx), z);
            float vmax = st.m;
#pragma unroll
            for (int i = 0; i < kVec; ++i) vmax = fmaxf(vmax, z[i]);
            grow_max<kEntropy>(st, vmax, k);
            const float mk = st.m * k;
#pragma unroll
            for (int i = 0; i < kVec; ++i) add_one<kEntropy>(st, z[i], k, mk);
        }
    }
    __syncthreads();            // lds may still be read by a slow wavefront of the previous reduction
    return reduce_row<kWideBlock, kEntropy>(st, k, lds, (int)threadIdx.x);
}

// What thread 0 found in the other half's record.
struct Inbox {
    Stats st;
    uint32_t zy_bits;           // fp32 bits of the logit at the label, if the other half holds it
    uint32_t arrived;
};

__device__ __forceinline__ bool read_record(const HalfRecord* rec, unsigned long long& a, unsigned long long& b) {
    if (a == 0) a = __hip_atomic_load(&rec->ms, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (b == 0) b = __hip_atomic_load(&rec->uz, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return a != 0 && b != 0;
}

__device__ __forceinline__ void fill_inbox(Inbox* in, unsigned long long a, unsigned long long b, bool ok) {
    in->st.m = __uint_as_float((uint32_t)a);
    in->st.s = __uint_as_float((uint32_t)(a >> 32));
    in->st.u = __uint_as_float((uint32_t)b);
    in->zy_bits = (uint32_t)(b >> 32);
    in->arrived = ok ? 1u : 0u;
}

// Publishes `mine` (and z_y, the logit at the label, if this half holds it) as half `half` of a row,
// waits (bounded) for the other half and returns the statistics of the whole row, merged in the order
// (first half, second half) by both workgroups; z_y becomes the other half's where that half holds
// the label (zy_there).  rec: the row's two records.  other_base / other_vec: where the other half's
// logits lie; zy_ptr: where the logit at the label lies.
template <int DT, bool kEntropy>
__device__ __forceinline__ Stats exchange_halves(const Stats& mine, int half, HalfRecord* rec, uint32_t spin_limit,
                                                 const typename Elem<DT>::T* other_base, int other_vec, float k,
                                                 bool other_whole, Stats* lds, Inbox* inbox, bool zy_here, bool zy_there,
                                                 const typename Elem<DT>::T* zy_ptr, float& z_y) {
    using E = Elem<DT>;
    if (threadIdx.x == 0) {
        // +0 would make an empty word of (u, z_y) = (0, 0): -0 is the same logit
        const uint32_t zy_word = zy_here ? (__float_as_uint(z_y) == 0u ? 0x80000000u : __float_as_uint(z_y)) : 1u;
        __hip_atomic_store(&rec[half].ms, pack2f(mine.m, mine.s), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&rec[half].uz, pack2f(kEntropy ? mine.u : 0.f, __uint_as_float(zy_word)), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        // at most spin_limit polls; with a limit of 0 the record is not looked at here at all, so that
        // the fallback can be exercised deterministically
        unsigned long long a = 0, b = 0;
        bool ok = false;
        for (uint32_t polls = 0; polls < spin_limit && !ok; ++polls) {
            ok = read_record(&rec[half ^ 1], a, b);
            if (!ok) __builtin_amdgcn_s_sleep(4);
        }
        fill_inbox(inbox, a, b, ok);
        // the record has reached memory before any thread of this workgroup stores a gradient
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();
    Stats other = inbox->st;
    if (inbox->arrived == 0u) {                                  // uniform branch
        other = stream_stats<DT, kEntropy>(other_base, other_vec, k, other_whole, lds);
        if (threadIdx.x == 0) {
            // the logit at the label from the other half, then - once it has arrived - the record again
            uint32_t zy_mem = zy_there ? __float_as_uint(E::load(zy_ptr)) : 0u;
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(zy_mem)::"memory");
            unsigned long long a = 0, b = 0;
            const bool ok = read_record(&rec[half ^ 1], a, b);
            fill_inbox(inbox, a, b, ok);
            if (!ok) inbox->zy_bits = zy_mem;
        }
        __syncthreads();
        if (inbox->arrived != 0u) other = inbox->st;
    }
    if (zy_there) z_y = __uint_as_float(inbox->zy_bits);
    return half == 0 ? merge<kEntropy>(mine, other, k) : merge<kEntropy>(other, mine, k);
}

// The fused sweep: persistent workgroups walk rows and, as one turns the
// registers of a row into dlogits, refills them with its NEXT row, so the statistics pass of the next
// row starts on its first vectors while the last are still arriving - the register file never has to
// hold two rows.  The next row is the next unclaimed one (see "row tickets" above), taken while the
// row is being written.
// row_ticket NULL: a workgroup per row, each ends with its first.
// Wavefronts per SIMD that the register allocator leaves room for: 4 hold the widest rows (76 registers of
// row), short rows leave more of the register file to further workgroups.
constexpr int waves_per_simd(int nv, int rows) { return nv <= 4 ? 8 : (nv <= 8 && rows == 1 ? 6 : 4); }

// kEdge: rows of any element alignment (see RowSpan); dlogits rows are misaligned alike.  Only these rows are
// ever swept a second time (mrl_fused_logprob_regrad): again.carried is then given and row_terms NULL.
// kWide: the units of work are half rows (see "wide rows" above): unit 2 r is the first
// half_elems entries of row r, unit 2 r + 1 the rest; n_rows then counts units.
// kRows: consecutive rows that a workgroup holds side by side, each by BLK of its threads (see pick_rows).
template <int DT, int BLK, int NV, int kRows, bool kEntropy, bool kWide, bool kEdge>
__global__ __launch_bounds__(BLK * kRows, waves_per_simd(NV, kRows)) void fused_sweep_persistent_kernel(
    const typename Elem<DT>::T* logits, int64_t row_stride, int vocab, uint32_t n_rows,
    const void* __restrict__ labels, int labels_dtype, float inv_t, const float* __restrict__ row_ops, int has_old,
    Params p, float grad_scale, const float* __restrict__ grad_scale_dev, mrl::Again again,
    typename Elem<DT>::T* dlogits, int64_t d_stride, float* __restrict__ logp, float* __restrict__ entropy, float* __restrict__ row_terms,
    unsigned int* row_ticket, int group, int half_elems, HalfRecord* half_records, uint32_t spin_limit) {
    using E = Elem<DT>;
    using T = typename E::T;
    static_assert(!kWide || BLK == kWideBlock, "halves of a row are held by workgroups of kWideBlock threads");
    static_assert(!(kWide && kEdge), "a row that two workgroups hold is aligned");
    static_assert(kRows == 1 || (!kWide && (BLK & (BLK - 1)) == 0), "whole rows side by side");
    // two sets of partials used in turn: a slow wavefront may still read the last row's
    __shared__ Stats lds[2][kRows * BLK / 64];
    int parts = 0;
    // Two slots used in turn, one per BROADCAST: thread 0 may write the next ticket while a slow wavefront
    // has yet to read this one's, and the barrier of the broadcast in between separates a slot's reuse.
    // (Between two broadcasts there may be no other: rows without a mask are not reduced.)
    __shared__ uint32_t next_row[2];
    int slot = 0;
    __shared__ Inbox inbox;                 // the other half's record (wide rows)

    // this thread within its row, and the row within the workgroup's unit (the same for a whole wavefront)
    const int tid = kRows == 1 ? (int)threadIdx.x : (int)threadIdx.x & (BLK - 1);
    const int lane_row = kRows == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / BLK);
    const bool outputs = tid == 0 && (!kEdge || row_terms != nullptr);
    // as in scale_rows_note_kernel: equal scales are noted by workgroup 0 at once, others by whoever ends last
    bool moved = false;
    if (kEdge && again.carried) {
        const float u = *grad_scale_dev;
        moved = u / again.carried[0] != 1.f;
        if (!moved && !again.always) {
            if (blockIdx.x == 0 && threadIdx.x == 0) note_scale(u, again.carried, again.learned);
            return;
        }
    }
    // bytes and vectors of a unit: the whole row, or its first / second half
    const uint32_t unit_bytes[2] = {(uint32_t)(kWide ? half_elems : vocab) * (uint32_t)sizeof(T),
                                    (uint32_t)(kWide ? vocab - half_elems : 0) * (uint32_t)sizeof(T)};
    const float k = inv_t * kLog2e;
    if (grad_scale_dev) grad_scale *= *grad_scale_dev;
    // the counter as a 4-byte buffer: only the lane with offset 0 (thread 0) is inside it
    const mrl::rsrc_t ticket = mrl::make_rsrc(row_ticket, row_ticket ? 4u : 0u);
    const mrl::rsrc_t no_ticket = mrl::make_rsrc(row_ticket, 0u);

    // What a workgroup needs to know of the row it fetches next.  A row that is not a response token
    // is never read: its descriptor gets zero bytes, so the (unconditional) loads return zeros
    // without touching memory; the same happens past the last row.
    struct Next {
        uint32_t r;             // unit; behind the last: none
        int64_t y;
        const T* zy_ptr;
        RowRef row;
        uint32_t edge_off;      // where this thread's edge entry lies in the row (kEdge)
        const T* edge_base;
        uint32_t edge_bytes;    // 0: not read
    };
    // 32 bits: at most 2^31 - 2 units, and what tickets add behind them stays far below 2^32 as well
    uint32_t r = blockIdx.x * (uint32_t)group;
    int left = group - 1;                   // units of the current ticket behind r
    // the unit behind r: the next of the ticket, or the first of a new ticket (asked for in `mine`)
    auto following = [&](uint32_t mine) {
        if (left > 0) {
            --left;
            return r + 1;
        }
        left = group - 1;
        const uint32_t t = broadcast_ticket(mine, &next_row[slot]);
        slot ^= 1;
        return row_ticket ? t + gridDim.x * (uint32_t)group : n_rows;
    };
    auto plan = [&](uint32_t r2) {
        Next n;
        n.r = r2;
        bool has = r2 * kRows < n_rows;
        const uint32_t un = has ? r2 : r;                   // unit
        uint32_t rn = kWide ? (un >> 1) : un * kRows + lane_row;    // row
        if (kRows > 1 && rn >= n_rows) {                    // the last unit may be short of rows
            has = false;
            rn = n_rows - 1;
        }
        const int hn = kWide ? (int)(un & 1) : 0;
        const bool live = has && (row_ops[(int64_t)rn * MRL_ROW_OPS + MRL_OP_MASK] != 0.f);
        const T* nrow = logits + (int64_t)rn * row_stride;
        if (kEdge) {
            const RowSpan span = row_span<DT>(nrow, vocab);
            n.row = row_ref(nrow + span.head, live ? (uint32_t)span.n_vec * 16u : 0u);
            n.edge_base = nrow;
            n.edge_bytes = live ? unit_bytes[0] : 0u;
            n.edge_off = edge_offset<DT>(span, vocab, tid);
        } else {
            n.row = row_ref(nrow + (hn ? half_elems : 0), live ? unit_bytes[hn] : 0u);
        }
        n.y = load_label(labels, labels_dtype, rn);
        n.zy_ptr = nrow + ((n.y >= 0 && n.y < (int64_t)vocab) ? n.y : 0);
        return n;
    };

    // The next row is requested in two bursts: its first H vectors once the first H vectors of the
    // current row have been written (they arrive while the rest of the gradient is computed, so the
    // statistics pass of the next row starts without waiting for memory), the others behind the last
    // store.  A larger H costs bandwidth: a row's requests are served best when they are issued
    // together.  The logit at the label comes last; it is not needed before the row is reduced.
    constexpr int H = NV >= 8 ? MRL_SWEEP_HEAD : NV / 2;
    u32x4 v[NV];
    int64_t y = 0;
    uint32_t zy_bits = 0;                   // the logit at the label as loaded; converted where it is used
    uint32_t edge_bits = 0;                 // the thread's edge entry, likewise
    auto load_edge = [&](const Next& n) {
        return kEdge ? E::buf_load_bits(mrl::make_rsrc(n.edge_base, n.edge_bytes), n.edge_off) : 0u;
    };
    if (r * kRows < n_rows) {
        const Next first = plan(r);
        y = first.y;
        // the same sequence of operations as one turn of the loop leaves behind (with stores that
        // write nothing), so that the number of operations outstanding at the top of the loop - which
        // the compiler has to assume when it places the waits of the statistics pass - is the same
        // on every path into it
        const RowRef none = row_ref(dlogits, 0u);
        mrl::buf_atomic_add_u32(mrl::make_rsrc(dlogits, 0u), lane_offset(tid), 0u);
        zero_part<BLK, 0, H>(none, tid);
        load_part<BLK, 0, H>(v, first.row, tid);
        zero_part<BLK, H, NV>(none, tid);
        if (kEdge) E::buf_store(mrl::make_rsrc(dlogits, 0u), 0u, 0.f);
        mrl::buf_store_b32(0u, mrl::make_rsrc(dlogits, 0u), 0u);
        load_part<BLK, H, NV>(v, first.row, tid);
        edge_bits = load_edge(first);
        zy_bits = E::load_bits(first.zy_ptr);
    }
    while (r * kRows < n_rows) {
        const uint32_t place = kWide ? (r >> 1) : r * kRows + lane_row;
        const bool mine_to_do = kRows == 1 || place < n_rows;   // else a place behind the last row: nothing is written
        const int64_t row = mine_to_do ? place : n_rows - 1;
        const int half = kWide ? (int)(r & 1) : 0;
        const int my_first = half ? half_elems : 0;         // first entry of this unit within the row
        RowSpan span = {0, (int)(unit_bytes[half] / 16u)};
        if (kEdge) span = row_span<DT>(logits + row * row_stride, vocab);
        const int n_vec = span.n_vec;
        T* const drow = dlogits + row * d_stride + my_first;
        const RowRef dst = row_ref(drow + span.head, !mine_to_do ? 0u : (kEdge ? (uint32_t)n_vec * 16u : unit_bytes[half]));
        const uint32_t edge_off = kEdge ? edge_offset<DT>(span, vocab, tid) : 0u;
        const uint32_t edge_bytes = mine_to_do ? unit_bytes[0] : 0u;
        const float* ops = row_ops + row * MRL_ROW_OPS;
        const float m = mine_to_do ? ops[MRL_OP_MASK] : 0.f;
        // the reduction's barrier is for the whole workgroup: it comes where any of its rows counts
        bool reduced = false;
#pragma unroll
        for (int i = 0; i < (kRows > 1 ? kRows : 0); ++i) {
            const uint32_t ri = r * kRows + i;
            reduced = reduced || (ri < n_rows && row_ops[(int64_t)ri * MRL_ROW_OPS + MRL_OP_MASK] != 0.f);
        }
        const bool y_ok = (y >= 0) && (y < (int64_t)vocab);
        // the label's entry gets its one-hot term from the unit that holds it
        const int64_t y_here = y - my_first;
        const bool y_mine = y_ok && (!kWide || (y_here >= 0 && y_here < (int64_t)(unit_bytes[half] / sizeof(T))));
        Next nx;
        uint32_t zy_next = 0, edge_next = 0;

        if constexpr (kRows > 1) {
            // Rows of all kinds share one path: two paths that load the next rows would leave them in different
            // registers, and the copies where the paths meet wait for every load.  A row without a gradient is
            // written as the product of zero coefficients and zeros.
            float z_y = E::from_bits(zy_bits), z_edge = kEdge ? E::from_bits(edge_bits) : 0.f;
            RowGrad g = {k, 0.f, 0.f, 0.f, 0.f};
            bool live = false;
            if (reduced) {
                const Stats st = thread_stats<DT, BLK, NV, kEntropy, kEdge>(v, n_vec, k, !y_ok, edge_off != 0x80000000u, z_edge, tid);
                wait_for_label_logit();
                const Stats tot = reduce_row<BLK, kEntropy>(st, k, lds[parts] + lane_row * (BLK / 64), tid);
                parts ^= 1;
                float lse;
                const RowScalars s = row_scalars<kEntropy>(tot, k, inv_t, y_ok, z_y, ops, has_old, p, grad_scale, m, lse);
                if (m != 0.f) {
                    if (outputs) write_row_outputs(row, s, m, logp, entropy, row_terms);
                    live = s.g_lp != 0.f || s.g_h != 0.f;
                    if (live) g = row_grad<kEntropy>(s, k, inv_t, lse);
                }
            }
            if (m == 0.f && outputs && mine_to_do) write_masked_row_outputs(row, logp, entropy, row_terms);
            if (!live) {
#pragma unroll
                for (int q = 0; q < NV; ++q) v[q] = mrl::make_u32x4(0u, 0u, 0u, 0u);
                z_y = z_edge = 0.f;
            }
            const uint32_t mine = mrl::buf_atomic_add_u32(left > 0 ? no_ticket : ticket, lane_offset((int)threadIdx.x), (uint32_t)group);
            grad_part<DT, BLK, kEntropy, 0, H>(v, g, dst, tid);
            nx = plan(following(mine));
            load_part<BLK, 0, H>(v, nx.row, tid);
            grad_part<DT, BLK, kEntropy, H, NV>(v, g, dst, tid);
            if (kEdge) E::buf_store(mrl::make_rsrc(drow, edge_bytes), edge_off, grad_elem<kEntropy>(g, z_edge));
            store_label_grad<DT, BLK, kEntropy, kEdge>(drow, unit_bytes[0], span, g, live && y_ok, y, z_y, tid);
            load_part<BLK, H, NV>(v, nx.row, tid);
            y = nx.y;
            zy_bits = E::load_bits(nx.zy_ptr);
            edge_bits = load_edge(nx);
            r = nx.r;
            continue;
        }
        bool wrote = false;                 // dlogits of row r written and the next row requested
        if (m != 0.f) {
            float z_y = E::from_bits(zy_bits);
            const float z_edge = kEdge ? E::from_bits(edge_bits) : 0.f;
            const Stats st = thread_stats<DT, BLK, NV, kEntropy, kEdge>(v, n_vec, k, !y_ok, edge_off != 0x80000000u, z_edge, tid);
            wait_for_label_logit();
            Stats tot = reduce_row<BLK, kEntropy>(st, k, lds[parts], tid);
            parts ^= 1;
            if (kWide) {
                // the logit at the label as this unit loaded it counts only if the label lies in this
                // half: the other half may already hold gradients when dlogits overwrite the logits
                const int other_first = half ? 0 : half_elems;
                const T* whole = logits + row * row_stride;
                tot = exchange_halves<DT, kEntropy>(tot, half, half_records + row * 2, spin_limit, whole + other_first,
                                                    (int)(unit_bytes[half ^ 1] / 16u), k, Tail<BLK, NV, kEdge>::kFull != 0 && y_ok, lds[parts ^ 1], &inbox, y_mine,
                                                    y_ok && !y_mine, whole + (y_ok ? y : 0), z_y);
            }
            float lse;
            const RowScalars s = row_scalars<kEntropy>(tot, k, inv_t, y_ok, z_y, ops, has_old, p, grad_scale, m, lse);
            if (outputs && half == 0) write_row_outputs(row, s, m, logp, entropy, row_terms);
            if (s.g_lp != 0.f || s.g_h != 0.f) {
                const RowGrad g = row_grad<kEntropy>(s, k, inv_t, lse);
                // the ticket is asked for ahead of the stores and picked up behind the first H of
                // them: it is older than every store, so waiting for it does not wait for them
                const uint32_t mine = mrl::buf_atomic_add_u32(left > 0 ? no_ticket : ticket, lane_offset((int)threadIdx.x), (uint32_t)group);
                grad_part<DT, BLK, kEntropy, 0, H>(v, g, dst, tid);
                nx = plan(following(mine));
                load_part<BLK, 0, H>(v, nx.row, tid);
                grad_part<DT, BLK, kEntropy, H, NV>(v, g, dst, tid);
                if (kEdge) E::buf_store(mrl::make_rsrc(drow, edge_bytes), edge_off, grad_elem<kEntropy>(g, z_edge));
                store_label_grad<DT, BLK, kEntropy, kEdge>(drow, unit_bytes[half], span, g, y_mine, y_here, z_y, tid);
                load_part<BLK, H, NV>(v, nx.row, tid);
                edge_next = load_edge(nx);
                zy_next = E::load_bits(nx.zy_ptr);
                wrote = true;
            }
        } else if (outputs && half == 0) {
            write_masked_row_outputs(row, logp, entropy, row_terms);
        }
        if (!wrote) {                       // no gradient for this row: zeros, same order of operations
            const uint32_t mine = mrl::buf_atomic_add_u32(left > 0 ? no_ticket : ticket, lane_offset((int)threadIdx.x), (uint32_t)group);
            zero_part<BLK, 0, H>(dst, tid);
            nx = plan(following(mine));
            load_part<BLK, 0, H>(v, nx.row, tid);
            zero_part<BLK, H, NV>(dst, tid);
            if (kEdge) E::buf_store(mrl::make_rsrc(drow, edge_bytes), edge_off, 0.f);
            mrl::buf_store_b32(0u, mrl::make_rsrc(dlogits, 0u), 0u);
            load_part<BLK, H, NV>(v, nx.row, tid);
            edge_next = load_edge(nx);
            zy_next = E::load_bits(nx.zy_ptr);
        }
        y = nx.y;
        zy_bits = zy_next;
        edge_bits = edge_next;
        r = nx.r;
    }
    // Every wavefront of a workgroup with rows has read the old scale by now: it has passed the barrier of at
    // least one ticket.  One without rows has nothing to do whatever it reads.
    if (kEdge && again.carried && threadIdx.x == 0)
        note_scale_last(*grad_scale_dev, again.carried, again.learned, moved ? again.rescales : nullptr);
}

// Backward of the split path as a plain stream: one 16-byte vector per thread, small workgroups that
// retire at once.  The backward needs no whole-row state (the log-sum-exp is an input), so nothing
// has to stay on chip, and this is the access pattern the HBM system serves best: the requests in
// flight always cover one compact, advancing stretch of the logits and of dlogits.  Grid: x walks
// the row in chunks of kThreads vectors, (y, z) number the rows; x is dispatched fastest, so the
// workgroups in flight are neighbours in memory.  A row with no incoming gradient is zero-filled
// without being read; a vector past the end of the row is neither read nor written (range checks).
constexpr int kChunkRowsY = 32768;      // rows per grid.y; grid.z carries the rest

template <int DT, bool kEntropy, int kThreads>
__global__ __launch_bounds__(kThreads) void bwd_chunk_kernel(
    const typename Elem<DT>::T* logits, int64_t row_stride, int vocab, int64_t n_rows,
    const void* __restrict__ labels, int labels_dtype, float inv_t, const float* __restrict__ lse_in,
    const float* __restrict__ ent_in, const float* __restrict__ g_logp, const float* __restrict__ g_entropy,
    typename Elem<DT>::T* dlogits, int64_t d_stride) {
    using E = Elem<DT>;
    using T = typename E::T;
    constexpr int kVec = E::kVec;
    const int64_t r = (int64_t)blockIdx.z * kChunkRowsY + blockIdx.y;
    if (r >= n_rows) return;
    const uint32_t row_bytes = (uint32_t)vocab * (uint32_t)sizeof(T);
    const uint32_t first = blockIdx.x * (uint32_t)kThreads;           // first vector of this workgroup
    const uint32_t off = (first + threadIdx.x) * 16u;
    const mrl::rsrc_t dst = mrl::make_rsrc(dlogits + r * d_stride, row_bytes);
    const float g_lp = g_logp ? g_logp[r] : 0.f;
    const float g_h = (kEntropy && g_entropy) ? g_entropy[r] : 0.f;
    if (g_lp == 0.f && g_h == 0.f) {
        const u32x4 zero = {0u, 0u, 0u, 0u};
        mrl::buf_store_nt(zero, dst, off);
        return;
    }
    const u32x4 v = mrl::buf_load_nt(mrl::make_rsrc(logits + r * row_stride, row_bytes), off);
    const float lse = lse_in[r];
    RowGrad g;
    g.k = inv_t * kLog2e;
    g.lse2 = lse * kLog2e;
    g.c0 = kEntropy ? inv_t * (-g_lp + g_h * (lse - ent_in[r])) : -g_lp * inv_t;
    g.c1 = kEntropy ? -g_h * inv_t * inv_t : 0.f;
    g.onehot = g_lp * inv_t;
    mrl::buf_store_nt(grad_vec<DT, kEntropy>(v, g), dst, off);
    // the entry at the label: written once more, with the one-hot term, by the thread that holds it
    // (stores of one thread to the same address stay in program order)
    const int64_t y = load_label(labels, labels_dtype, r);
    if (y >= 0 && y < (int64_t)vocab) {
        const uint32_t yv = (uint32_t)y / (uint32_t)kVec;
        if (yv >= first && yv < first + (uint32_t)kThreads) {        // uniform over the workgroup
            float z[kVec];
            E::unpack(v, z);
            const int e = (int)((uint32_t)y % (uint32_t)kVec);
            float z_y = z[0];
#pragma unroll
            for (int i = 1; i < kVec; ++i) z_y = (e == i) ? z[i] : z_y;
            const uint32_t y_off = (yv - first == threadIdx.x) ? (uint32_t)y * (uint32_t)sizeof(T) : 0x80000000u;
            E::buf_store(dst, y_off, grad_elem<kEntropy>(g, z_y) + g.onehot);
        }
    }
}

// Conditional in-place rescale: multiplies every row by upstream/applied unless that ratio is 1
// (then every workgroup exits at once; the grid is kept small so that this costs microseconds).
template <int DT>
__device__ __forceinline__ void scale_rows(typename Elem<DT>::T* x, int64_t row_stride, int vocab, int64_t n_rows, int tail,
                                           float ratio) {
    using E = Elem<DT>;
    constexpr int kVec = E::kVec;
    const int n_vec = vocab / kVec;
    for (int64_t r = blockIdx.x; r < n_rows; r += gridDim.x) {
        u32x4* vec = reinterpret_cast<u32x4*>(x + r * row_stride);
        for (int idx = threadIdx.x; idx < n_vec; idx += 256) {
            float z[kVec];
            E::unpack(vec[idx], z);
#pragma unroll
            for (int i = 0; i < kVec; ++i) z[i] *= ratio;
            vec[idx] = E::pack(z);
        }
    }
    // entries behind the last row (see flat_rows)
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < tail) {
        typename E::T* p = x + n_rows * row_stride + i;
        E::store(p, E::load(p) * ratio);
    }
}

template <int DT>
__global__ __launch_bounds__(256) void scale_rows_kernel(typename Elem<DT>::T* x, int64_t row_stride, int vocab,
                                                         int64_t n_rows, int tail, const float* __restrict__ upstream,
                                                         const float* __restrict__ applied) {
    const float ratio = *upstream / *applied;
    if (ratio == 1.f) return;
    scale_rows<DT>(x, row_stride, vocab, n_rows, tail, ratio);
}

// One backward of one buffer in a single launch: the conditional rescale above, then the book-keeping
// of grad_scale_note_kernel.  When nothing is to be moved (the ratio is 1, i.e. the new scale equals
// the old one) workgroup 0 does the book-keeping at once - what it stores over the scale is the value
// every other workgroup reads there anyway - and the others leave.  Otherwise the workgroup that
// finishes last does it (a counter next to the scale tells; every workgroup has read the scale before
// it counts itself, so the last one may overwrite it).
template <int DT>
__global__ __launch_bounds__(256) void scale_rows_note_kernel(typename Elem<DT>::T* x, int64_t row_stride, int vocab,
                                                              int64_t n_rows, int tail,
                                                              const float* __restrict__ upstream, float* applied,
                                                              float* learned, uint32_t* rescales) {
    const float u = *upstream;
    const float was = applied[0];
    const float ratio = u / was;
    if (ratio == 1.f) {
        if (blockIdx.x == 0 && threadIdx.x == 0) note_scale(u, applied, learned);
        return;
    }
    scale_rows<DT>(x, row_stride, vocab, n_rows, tail, ratio);
    __syncthreads();
    if (threadIdx.x == 0) note_scale_last(u, applied, learned, rescales);
}

// Book-keeping behind one or more scale_rows_kernel launches: the buffers now carry `upstream`.
__global__ void grad_scale_note_kernel(const float* __restrict__ upstream, float* applied, float* learned,
                                       uint32_t* rescales) {
    if (threadIdx.x != 0) return;
    const float u = *upstream;
    const float was = *applied;
    if (rescales && u / was != 1.f) *rescales += 1u;
    note_scale(u, applied, learned);
}

// ----------------------------------------------------------------------------- host dispatch
// Workgroup size and vectors per thread.  A row shorter than the 1024 x 12 that the register files were
// laid out for leaves lanes and registers of a lone workgroup idle, and nothing computes while it waits for
// its loads; several smaller workgroups per CU overlap each other.  Upper ends by measurement (forward +
// backward of a row, 2.5 GB of logits, GB/s; 1024 threads with the fewest vectors before):
//   bf16:  16 KB 1 517 -> 5 467, 32 KB 2 980 -> 5 595, 48 KB 4 197 -> 5 731, 64 KB 5 144 -> 6 139,
//          80 KB 4 417 -> 5 906, 100 KB 5 199 -> 5 879 (512 x 16; 512 x 12 where both fit within 2 %)
//   fp32 (half the entries per byte to compute): 32 KB 3 802 -> 5 599, 48 KB 4 859 -> 6 205, 64 KB 5 832 -> 6 083;
//          96 and 128 KB stay with 1024 x 8 (6 190 and 6 250 against 5 800 and 5 700 with 512 x 16);
//          34 and 39 KB 5 354 and 5 934 with 512 x 8, up to there 256 x 12, which takes rows side by side (5 833 and
//          5 963; 600 of them 16.3 and 16.7 -> 12.6 and 12.9 us; fewer than 512, a row to a workgroup, within 5 %).  That
//          one is not as in the larger shape: half the threads add up twice the vectors, which rounds differently
// 16-bit rows of 40 to 48 KB, 256 x 12 and with 512 x 8: 24 576 entries 5 576 and 6 115 GB/s, 600 of them 15.6 and 17.2 us.
// Vectors of a thread that lie past the row are computed on all the same, so that a shape with fewer is the faster one,
// the more so with the entropy's sum and with few rows, which wait for a single row's chain; which thread holds what is
// as in the larger shape, and with it every bit.  512 x 12 -> 512 x 8, without and with entropy, GB/s of 1 GB of logits
// and us of 600 rows: 24 640 bf16 5 680 -> 5 985 and 5 232 -> 5 743, 19.6 -> 17.5 and 20.4 -> 15.9; 32 000 5 910 ->
// 5 927 and 5 843 -> 5 874, 20.4 -> 19.4; 12 000 fp32 6 090 -> 6 195, 18.0 -> 17.1.  Its registers leave room for three
// workgroups per CU, which pays where all rows start at once; with more rows three move less than two (32 000 bf16
// 5 624, 12 000 fp32 5 815), hence the limit in launch_sweep.  1024 x 12 -> 1024 x 10 with entropy: 66 000 bf16 5 427 ->
// 5 561, 42.2 -> 40.3; 1024 x 16 -> 1024 x 14: 100 352 5 853 -> 5 916, 55.6 -> 53.1.  512 x 10 and 512 x 14 changed
// nothing but 2 to 3 % of few rows.
// The choice depends on the row's length alone, so a row's result does not depend on the other rows' contents.
// Its place does enter for rows that are not whole 128-byte lines (see RowSpan): which thread adds which entry
// follows from the row's address modulo 128, so the fp32 sums round differently at another place in the batch.
inline int pick_shape(int dtype, int64_t n_vec) {
    for (int i = 0; i < kShapes; ++i)
        if (n_vec <= kRowShapes[i].most(dtype)) return i;
    return kShapes;                                 // too long: two halves
}

// Number of CUs of the current device (one persistent workgroup each); 0 if the query fails.
int cu_count() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    return n;
}

// Rows of 256 threads that a workgroup holds side by side (and with how many vectors a thread: fewer than the row's
// shape has where that leaves no lane idle; which thread holds what is the same, and with it every bit of the
// results).  A CU holds four to eight such rows either way (six of 256 x 8 alone, four side by side), but alone they are
// as many separate bursts of 16 to 48 KiB: the rows of a unit are requested, and written, together.  1 GB of logits, GB/s
// of a row alone -> side by side (16 bits without and with the entropy's sum; fp32 within 1 % of each other):
//   16 bits  8 000 entries 5 227 -> 5 733, 5 247 -> 5 675; 11 776 5 522 -> 6 046, 5 497 -> 5 845; 13 824 5 461 ->
//            6 052, 5 471 -> 5 974; 16 384 5 458 -> 6 116, 5 473 -> 6 069; 17 408 5 399 -> 5 895, 5 383 -> 5 826;
//            20 480 5 683 -> 5 866, 5 665 -> 5 823.  Not 7 168 (4 846 -> 4 824 with entropy), 9 728 (5 516 -> 5 227)
//            and 22 528 (5 616 -> 5 700): there the last of a thread's vectors are mostly past the row, and the
//            arithmetic of a unit, which starts and ends together, shows
//   fp32     3 328 5 405 -> 5 954, 4 096 5 497 -> 5 849, 4 864 5 604 -> 6 053, 5 888 5 588 -> 6 200, 8 192 5 568 -> 6 190,
//            8 704 5 421 -> 5 854, 9 984 5 683 -> 5 973
// Few rows: where all start at once they share tickets and are done sooner, also where four of them leave CUs without any
// (512 rows, us: 8 192 bf16 12.0 -> 9.4, 16 384 12.8 -> 11.2, 2 112 fp32 11.3 -> 8.7, 8 192 12.3 -> 11.1, 8 704 12.6 -> 12.1;
// 1 024 x 8 000 bf16 13.0 -> 10.8, 1 024 x 5 888 fp32 13.9 -> 12.6); in between the last, half empty round of larger units costs more than they gain
// (2 048 x 16 384 bf16 26.6 -> 29.0 us, 4 096 x 8 000 28.9 -> 30.8; 8 192 x 16 384 100.1 -> 97.6), except where rows
// are longer than 32 KiB (1 024 x 17 408 21.8 -> 15.7, 3 072 47.0 -> 45.0).
// Returns the place in kSideShapes; -1: a row to a workgroup.
inline int pick_rows(int dtype, int64_t n_vec, int64_t n_rows) {
    for (int i = 0; i < kSides; ++i) {
        const SideShape& s = kSideShapes[i];
        if (n_vec <= s.above(dtype) || n_vec > s.most(dtype)) continue;
        if (n_rows >= (n_vec <= 1024 ? 16384 : 8192)) return i;
        const int per_cu = waves_per_simd(s.vectors, s.rows);       // a row is a wavefront on each of a CU's four SIMDs
        return n_rows >= 512 && (n_vec > 2048 || n_rows <= (int64_t)per_cu * cu_count()) ? i : -1;
    }
    return -1;
}

// Upper bound of the polls a workgroup spends waiting for the other half of a wide row before it
// computes that half's statistics itself (mrl_set_wide_spin_limit; 0: never look, always compute).
constexpr uint32_t kDefaultSpinLimit = 1u << 18;
std::atomic<uint32_t> g_wide_spin_limit{kDefaultSpinLimit};

constexpr int64_t kWorkspaceHeader = 16;    // the row counter, padded to the alignment of the records
// Unaligned rows below this go to the split kernels: a thread then holds less than half of its 4 vectors.
constexpr int64_t kMinEdgeRowBytes = 8192;

template <int DT, int BLK, int NV, int kRows, bool kEntropy, bool kWide, bool kEdge>
int launch_sweep(const mrl::FusedArgs& a) {
    using T = typename Elem<DT>::T;
    const Params p = {a.clip_lo, a.clip_hi, a.kl_coef, a.entropy_coeff, 1.f, a.kl_penalty, 0};
    unsigned int* counter = reinterpret_cast<unsigned int*>(a.workspace);
    const int64_t rows = kWide ? 2 * a.n_rows : a.n_rows;       // half rows are counted as such
    const int64_t units = (rows + kRows - 1) / kRows;
    int64_t grid = units;
    int group = 1;
    if (counter != nullptr) {
        const int cus = cu_count();
        if (cus < 2) return mrl::fail(MRL_ERR_LAUNCH, "mrl_fused_logprob_loss: cannot query the device");
        // half rows: an even number of workgroups, so that the halves of a row start side by side
        int64_t per_cu = waves_per_simd(NV, kRows) * 4 / (BLK * kRows / 64);
        if (BLK == 512 && NV == 8 && rows > per_cu * cus) per_cu = 2;       // see pick_shape
        const int64_t cap = kWide ? (cus & ~1) : (int64_t)cus * per_cu;
        // Rows per ticket: the counter serves about 85 tickets per microsecond, rows below 32 KiB go faster
        // than that (8 000 bf16 logits, rows per ticket 1 / 2 / 4: 2 728 / 5 085 / 5 276 GB/s for 155 648 rows,
        // 1 819 / 2 537 / 2 479 for 2 048; 16 384: 5 241 / 5 481 / 5 294; 24 576: 5 681 / 5 466 / 5 253).
        if (BLK * kRows == 256 && NV <= 8 && a.n_rows > 512) group = NV <= 4 && a.n_rows >= 4096 ? 4 : 2;
        grid = (units + group - 1) / group;
        if (cap < grid) grid = cap;
        if (!a.workspace_cleared) {
            const int64_t words = (kWorkspaceHeader + (kWide ? a.n_rows * 2 * (int64_t)sizeof(HalfRecord) : 0)) / 8;
            hipLaunchKernelGGL(clear_words_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, a.stream,
                               reinterpret_cast<unsigned long long*>(a.workspace), words);
        }
    }
    HalfRecord* rec = kWide ? reinterpret_cast<HalfRecord*>(reinterpret_cast<char*>(a.workspace) + kWorkspaceHeader) : nullptr;
    hipLaunchKernelGGL((fused_sweep_persistent_kernel<DT, BLK, NV, kRows, kEntropy, kWide, kEdge>), dim3((unsigned)grid),
                       dim3(BLK * kRows), 0, a.stream, (const T*)a.logits, a.row_stride, (int)a.vocab, (uint32_t)rows, a.labels, a.labels_dtype,
                       a.inv_t, a.row_ops, a.has_old, p, a.grad_scale, a.grad_scale_dev, a.again, (T*)a.dlogits, a.d_stride, a.logp,
                       a.entropy, a.row_terms, counter, group, (int)a.half_elems, rec,
                       g_wide_spin_limit.load(std::memory_order_relaxed));
    return mrl::check_launch("mrl_fused_logprob_loss");
}

template <int DT, int BLK, int NV, int kRows = 1>
int launch_narrow(const mrl::FusedArgs& a) {
    if (a.edge)
        return a.with_entropy ? launch_sweep<DT, BLK, NV, kRows, true, false, true>(a)
                              : launch_sweep<DT, BLK, NV, kRows, false, false, true>(a);
    return a.with_entropy ? launch_sweep<DT, BLK, NV, kRows, true, false, false>(a)
                          : launch_sweep<DT, BLK, NV, kRows, false, false, false>(a);
}

template <int DT, int I = 0>
int fused_by_shape(int shape, const mrl::FusedArgs& a) {
    if constexpr (I < kShapes) {
        constexpr RowShape s = kRowShapes[I];
        if (I != shape) return fused_by_shape<DT, I + 1>(shape, a);
        if constexpr (s.most(DT) > 0) {
            if constexpr (s.most(DT) > kMinHalf)
                if (a.wide)
                    return a.with_entropy ? launch_sweep<DT, s.threads, s.vectors, 1, true, true, false>(a)
                                          : launch_sweep<DT, s.threads, s.vectors, 1, false, true, false>(a);
            return launch_narrow<DT, s.threads, s.vectors>(a);
        }
    }
    return mrl::fail(MRL_ERR_LAUNCH, "mrl_fused_logprob_loss: no shape for these rows");
}

template <int DT, int I = 0>
int fused_side_by_side(int side, const mrl::FusedArgs& a) {
    if constexpr (I < kSides) {
        constexpr SideShape s = kSideShapes[I];
        if (I != side) return fused_side_by_side<DT, I + 1>(side, a);
        if constexpr (s.most(DT) > 0) return launch_narrow<DT, kSideThreads, s.vectors, s.rows>(a);
    }
    return mrl::fail(MRL_ERR_LAUNCH, "mrl_fused_logprob_loss: no shape for these rows");
}

template <int DT>
int fused_sweep(int shape, int side, const mrl::FusedArgs& a) {
    return side >= 0 ? fused_side_by_side<DT>(side, a) : fused_by_shape<DT>(shape, a);
}

}  // namespace

namespace mrl {

template <int DT, int kThreads>
static int launch_bwd_chunk_n(const BwdArgs& a) {
    using T = typename Elem<DT>::T;
    const int64_t n_vec = a.vocab / Elem<DT>::kVec;
    const int64_t gy = a.n_rows < kChunkRowsY ? a.n_rows : kChunkRowsY;
    const int64_t gz = (a.n_rows + kChunkRowsY - 1) / kChunkRowsY;
    const dim3 grid((unsigned)((n_vec + kThreads - 1) / kThreads), (unsigned)gy, (unsigned)gz);
#define MRL_BWDC_LAUNCH(ENT)                                                                                     \
    hipLaunchKernelGGL((bwd_chunk_kernel<DT, ENT, kThreads>), grid, dim3(kThreads), 0, a.stream, (const T*)a.logits, \
                       a.row_stride, (int)a.vocab, a.n_rows, a.labels, a.labels_dtype, a.inv_t, a.lse, a.entropy,  \
                       a.g_logp, a.g_entropy, (T*)a.dlogits, a.d_stride)
    if (a.g_entropy != nullptr) MRL_BWDC_LAUNCH(true);
    else MRL_BWDC_LAUNCH(false);
#undef MRL_BWDC_LAUNCH
    return check_launch("mrl_vocab_logprob_bwd");
}

// Workgroups of half the size when that leaves at least 3 % fewer lanes idle in a row's last
// chunk (a 38 KiB row is 9.3 chunks of 256 vectors: 2.30 ms against 2.19 ms for 171 174 such rows).
template <int DT>
static int launch_bwd_chunk(const BwdArgs& a) {
    constexpr int kFull = MRL_BWD_CHUNK_THREADS, kHalf = MRL_BWD_CHUNK_THREADS / 2;
    const int64_t n_vec = a.vocab / Elem<DT>::kVec;
    const int64_t idle_full = (n_vec + kFull - 1) / kFull * kFull - n_vec;
    const int64_t idle_half = (n_vec + kHalf - 1) / kHalf * kHalf - n_vec;
    if ((idle_full - idle_half) * 100 >= 3 * n_vec) return launch_bwd_chunk_n<DT, kHalf>(a);
    return launch_bwd_chunk_n<DT, kFull>(a);
}

int launch_bwd_chunks(const BwdArgs& a) {
    switch (a.dtype) {
        case MRL_F32: return launch_bwd_chunk<MRL_F32>(a);
        case MRL_BF16: return launch_bwd_chunk<MRL_BF16>(a);
        default: return launch_bwd_chunk<MRL_F16>(a);
    }
}

bool bwd_chunks_supported(int dtype, int64_t vocab, const void* in, int64_t in_stride, const void* out,
                          int64_t out_stride, int64_t n_rows) {
    const int eb = float_dtype_bytes(dtype);
    if (eb == 0) return false;
    const int64_t per_vec = 16 / eb;
    // rows of whole vectors, at least 16 KiB (below that the loop kernel with one workgroup per row has
    // less to launch), below 2 GiB (32-bit range checks), and a grid.z within its limit
    if (vocab % per_vec != 0 || vocab * eb < 16 * 1024 || vocab * eb >= (1LL << 31)) return false;
    if (n_rows > (int64_t)kChunkRowsY * 65535) return false;
    if (!aligned(in, 16) || !aligned(out, 16)) return false;
    if (n_rows > 1 && ((in_stride * eb) % 16 != 0 || (out_stride * eb) % 16 != 0)) return false;
    return true;
}

// How rows of this shape and place are swept: as whole 16-byte vectors (also the only way for rows that two
// workgroups hold), or line by line with edges, for which every row of dlogits must be misaligned as its row
// of logits is.
RowLayout row_sweep_layout(int dtype, int64_t vocab, const void* in, int64_t in_stride, const void* out,
                           int64_t out_stride, int64_t n_rows) {
    const int64_t eb = float_dtype_bytes(dtype);
    if (eb == 0) return RowLayout::none;
    const uintptr_t pi = reinterpret_cast<uintptr_t>(in), po = reinterpret_cast<uintptr_t>(out);
    const int64_t n_vec = vocab / (16 / eb);
    const int64_t si = n_rows > 1 ? in_stride * eb : 0, so = n_rows > 1 ? out_stride * eb : 0;
    const bool vectors = vocab % (16 / eb) == 0 && (n_vec + 1) / 2 <= kMaxVec && pi % 16 == 0 && po % 16 == 0 &&
                         si % 16 == 0 && so % 16 == 0;
    if (vectors && (n_vec > kMaxVec || (pi % kEdgeAlign == 0 && si % kEdgeAlign == 0))) return RowLayout::vectors;
    const int64_t alike = vectors ? kEdgeAlign : 16;        // taken from the vectors only if both sides gain
    const bool edges = vocab * eb >= kMinEdgeRowBytes && n_vec <= kMaxVec && pi % eb == 0 && pi % alike == po % alike &&
                       (si - so) % alike == 0;
    return edges ? RowLayout::edges : (vectors ? RowLayout::vectors : RowLayout::none);
}

}  // namespace mrl

extern "C" int64_t mrl_fused_max_vocab(int logits_dtype) {
    const int eb = mrl::float_dtype_bytes(logits_dtype);
    if (eb == 0) return 0;
    return 2 * kMaxVec * (16 / eb);                 // two workgroups hold a wide row
}

extern "C" int64_t mrl_fused_workspace_bytes(int logits_dtype, int64_t n_rows, int64_t vocab) {
    const int eb = mrl::float_dtype_bytes(logits_dtype);
    if (eb == 0 || n_rows < 0 || vocab <= 0) return 0;
    const int64_t n_vec = vocab / (16 / eb);
    if (vocab % (16 / eb) != 0) return vocab * eb >= kMinEdgeRowBytes && n_vec <= kMaxVec ? kWorkspaceHeader : 0;
    if (n_vec <= kMaxVec) return kWorkspaceHeader;
    if ((n_vec + 1) / 2 > kMaxVec) return 0;
    return kWorkspaceHeader + n_rows * (int64_t)sizeof(HalfRecord) * 2;
}

extern "C" int64_t mrl_set_wide_spin_limit(int64_t polls) {
    const uint32_t next = polls < 0 ? kDefaultSpinLimit : (uint32_t)(polls > 0xffffffffLL ? 0xffffffffLL : polls);
    return (int64_t)g_wide_spin_limit.exchange(next, std::memory_order_relaxed);
}

// Checks and launch shared by the two entry points of the sweep.
static int run_sweep(const char* fn, mrl::FusedArgs& a, int64_t workspace_bytes) {
    MRL_REQUIRE(a.n_rows >= 0 && a.vocab > 0 && a.n_rows <= 0x3fffffffLL, MRL_ERR_INVALID_ARG, "%s: n_rows=%lld vocab=%lld",
                fn, (long long)a.n_rows, (long long)a.vocab);
    const int eb = mrl::float_dtype_bytes(a.dtype);
    MRL_REQUIRE(eb != 0, MRL_ERR_UNSUPPORTED, "%s: logits dtype %d (want F32, BF16 or F16)", fn, a.dtype);
    MRL_REQUIRE(mrl::int_dtype_bytes(a.labels_dtype) != 0, MRL_ERR_UNSUPPORTED, "%s: labels dtype %d (want I32 or I64)",
                fn, a.labels_dtype);
    MRL_REQUIRE(a.row_stride >= a.vocab && a.d_stride >= a.vocab, MRL_ERR_INVALID_ARG, "%s: row stride below vocab", fn);
    MRL_REQUIRE(a.kl_penalty >= MRL_KL_NONE && a.kl_penalty <= MRL_KL_LOW_VAR, MRL_ERR_INVALID_ARG, "%s: kl_penalty=%d", fn,
                a.kl_penalty);
    MRL_REQUIRE(a.inv_t > 0.f && a.inv_t < 1.0e6f, MRL_ERR_INVALID_ARG, "%s: inv_temperature=%g must be in (0, 1e6)", fn,
                (double)a.inv_t);
    if (a.n_rows == 0) return MRL_OK;
    const bool again = a.again.carried != nullptr;
    MRL_REQUIRE(a.logits && a.labels && a.row_ops && a.dlogits && (a.row_terms || again), MRL_ERR_INVALID_ARG,
                "%s: NULL pointer", fn);
    MRL_REQUIRE(mrl::aligned(a.workspace, 16) && mrl::aligned(a.grad_scale_dev, 4) &&
                    mrl::aligned(a.again.carried, 8) && mrl::aligned(a.again.learned, 4) && mrl::aligned(a.again.rescales, 4),
                MRL_ERR_MISALIGNED, "%s: workspace must be 16-byte, a scale with its counter 8-byte and the other scalars "
                "4-byte aligned", fn);
    const mrl::RowLayout layout =
        mrl::row_sweep_layout(a.dtype, a.vocab, a.logits, a.row_stride, a.dlogits, a.d_stride, a.n_rows);
    MRL_REQUIRE(layout != mrl::RowLayout::none, MRL_ERR_UNSUPPORTED,
                "%s: needs 16-byte aligned rows, vocab %% %d == 0 and vocab <= %lld for this dtype, or rows of 8 KiB to "
                "half that vocab whose dlogits are misaligned alike (got vocab=%lld)", fn, 16 / eb,
                (long long)mrl_fused_max_vocab(a.dtype), (long long)a.vocab);
    a.edge = layout == mrl::RowLayout::edges;
    MRL_REQUIRE(!again || a.edge, MRL_ERR_UNSUPPORTED, "%s: rows of whole aligned vectors are not swept again", fn);
    if (a.dlogits != a.logits) {
        const char* x = (const char*)a.logits;
        const char* y = (const char*)a.dlogits;
        const int64_t xb = ((a.n_rows - 1) * a.row_stride + a.vocab) * eb, yb = ((a.n_rows - 1) * a.d_stride + a.vocab) * eb;
        MRL_REQUIRE(x + xb <= y || y + yb <= x, MRL_ERR_INVALID_ARG, "%s: dlogits partially overlaps logits", fn);
    } else {
        MRL_REQUIRE(!again, MRL_ERR_INVALID_ARG, "%s: the logits have been overwritten", fn);
        MRL_REQUIRE(a.d_stride == a.row_stride, MRL_ERR_INVALID_ARG, "%s: in-place needs identical strides", fn);
    }
    const int64_t n_vec = a.vocab / (16 / eb);
    int shape = pick_shape(a.dtype, n_vec);
    a.wide = shape == kShapes;
    a.half_elems = 0;
    if (a.wide) {
        a.half_elems = (n_vec + 1) / 2 * (16 / eb);
        shape = pick_shape(a.dtype, (n_vec + 1) / 2);
    }
    // without a counter every row has a workgroup of its own
    const int side = a.workspace != nullptr && !a.wide ? pick_rows(a.dtype, n_vec, a.n_rows) : -1;
    if (a.workspace != nullptr || a.wide) {
        const int64_t need = a.wide ? mrl_fused_workspace_bytes(a.dtype, a.n_rows, a.vocab) : kWorkspaceHeader;
        MRL_REQUIRE(a.workspace != nullptr && workspace_bytes >= need, MRL_ERR_INVALID_ARG,
                    "%s: workspace of %lld bytes, need %lld (rows of this width are cut in two halves that exchange "
                    "their statistics through it)", fn, (long long)(a.workspace ? workspace_bytes : 0), (long long)need);
    }
    switch (a.dtype) {
        case MRL_F32: return fused_sweep<MRL_F32>(shape, side, a);
        case MRL_BF16: return fused_sweep<MRL_BF16>(shape, side, a);
        default: return fused_sweep<MRL_F16>(shape, side, a);
    }
}

extern "C" int mrl_fused_logprob_loss(const void* logits, int logits_dtype, int64_t n_rows, int64_t vocab,
                                      int64_t row_stride, const void* labels, int labels_dtype,
                                      float inv_temperature, const float* row_ops, int has_old, float clip_lo,
                                      float clip_hi, int kl_penalty, float kl_coef, float entropy_coeff,
                                      float grad_scale, const float* grad_scale_dev, void* dlogits,
                                      int64_t dlogits_row_stride, float* logp, float* entropy, float* row_terms,
                                      void* workspace, int64_t workspace_bytes, int workspace_cleared,
                                      void* stream) {
    mrl::FusedArgs a = {};
    a.logits = logits; a.dtype = logits_dtype; a.n_rows = n_rows; a.vocab = vocab; a.row_stride = row_stride;
    a.labels = labels; a.labels_dtype = labels_dtype; a.inv_t = inv_temperature; a.row_ops = row_ops;
    a.has_old = has_old; a.clip_lo = clip_lo; a.clip_hi = clip_hi; a.kl_penalty = kl_penalty; a.kl_coef = kl_coef;
    a.entropy_coeff = entropy_coeff; a.grad_scale = grad_scale; a.grad_scale_dev = grad_scale_dev;
    a.workspace = workspace; a.workspace_cleared = workspace_cleared != 0; a.dlogits = dlogits; a.d_stride = dlogits_row_stride;
    a.logp = logp; a.entropy = entropy; a.row_terms = row_terms; a.with_entropy = (entropy != nullptr);
    a.stream = mrl::as_stream(stream);
    return run_sweep("mrl_fused_logprob_loss", a, workspace_bytes);
}

extern "C" int mrl_fused_logprob_regrad(const void* logits, int logits_dtype, int64_t n_rows, int64_t vocab,
                                        int64_t row_stride, const void* labels, int labels_dtype,
                                        float inv_temperature, const float* row_ops, int has_old, float clip_lo,
                                        float clip_hi, int kl_penalty, float kl_coef, float entropy_coeff,
                                        float grad_scale, const float* upstream, float* carried, float* learned,
                                        uint32_t* rescales, int always, void* dlogits, int64_t dlogits_row_stride, void* workspace, int64_t workspace_bytes,
                                        int workspace_cleared, void* stream) {
    const char* fn = "mrl_fused_logprob_regrad";
    MRL_REQUIRE(n_rows == 0 || (upstream && carried), MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    mrl::FusedArgs a = {};
    a.logits = logits; a.dtype = logits_dtype; a.n_rows = n_rows; a.vocab = vocab; a.row_stride = row_stride;
    a.labels = labels; a.labels_dtype = labels_dtype; a.inv_t = inv_temperature; a.row_ops = row_ops;
    a.has_old = has_old; a.clip_lo = clip_lo; a.clip_hi = clip_hi; a.kl_penalty = kl_penalty; a.kl_coef = kl_coef;
    a.entropy_coeff = entropy_coeff; a.grad_scale = grad_scale; a.grad_scale_dev = upstream;
    a.again = {carried, learned, rescales, always};
    a.workspace = workspace; a.workspace_cleared = workspace_cleared != 0; a.dlogits = dlogits; a.d_stride = dlogits_row_stride;
    a.with_entropy = entropy_coeff != 0.f;
    a.stream = mrl::as_stream(stream);
    return run_sweep(fn, a, workspace_bytes);
}

// Dense rows of an odd vocabulary are one stretch of entries: cut into rows of 2048 (fewer when there are
// fewer) and a tail of less than that, which is returned.  Other rows stay as they are.
static int flat_rows(int eb, int64_t& n_rows, int64_t& vocab, int64_t& row_stride) {
    if (vocab % (16 / eb) == 0 || row_stride != vocab) return 0;
    const int64_t total = n_rows * vocab;
    vocab = row_stride = 2048;
    n_rows = total / vocab;
    return (int)(total % vocab);
}

extern "C" int mrl_scale_rows(void* x, int dtype, int64_t n_rows, int64_t vocab, int64_t row_stride,
                              const float* upstream, const float* applied, void* stream) {
    const char* fn = "mrl_scale_rows";
    const int eb = mrl::float_dtype_bytes(dtype);
    MRL_REQUIRE(eb != 0, MRL_ERR_UNSUPPORTED, "%s: dtype %d (want F32, BF16 or F16)", fn, dtype);
    MRL_REQUIRE(n_rows >= 0 && n_rows <= 0x7fffffffLL && vocab > 0 && row_stride >= vocab, MRL_ERR_INVALID_ARG,
                "%s: n_rows=%lld vocab=%lld row_stride=%lld", fn, (long long)n_rows, (long long)vocab,
                (long long)row_stride);
    if (n_rows == 0) return MRL_OK;
    MRL_REQUIRE(x && upstream && applied, MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    MRL_REQUIRE(mrl::aligned(upstream, 4) && mrl::aligned(applied, 4), MRL_ERR_MISALIGNED,
                "%s: upstream and applied must be 4-byte aligned", fn);
    const int tail = flat_rows(eb, n_rows, vocab, row_stride);
    MRL_REQUIRE(vocab % (16 / eb) == 0 && mrl::aligned(x, 16) && (n_rows == 1 || (row_stride * eb) % 16 == 0),
                MRL_ERR_UNSUPPORTED, "%s: needs 16-byte aligned or dense rows", fn);
    hipStream_t s = mrl::as_stream(stream);
    const dim3 grid((unsigned)(n_rows < 8 ? 8 : (n_rows < 4096 ? n_rows : 4096))), block(256);
    switch (dtype) {
        case MRL_F32:
            hipLaunchKernelGGL(scale_rows_kernel<MRL_F32>, grid, block, 0, s, (float*)x, row_stride, (int)vocab,
                               n_rows, tail, upstream, applied);
            break;
        case MRL_BF16:
            hipLaunchKernelGGL(scale_rows_kernel<MRL_BF16>, grid, block, 0, s, (uint16_t*)x, row_stride, (int)vocab,
                               n_rows, tail, upstream, applied);
            break;
        default:
            hipLaunchKernelGGL(scale_rows_kernel<MRL_F16>, grid, block, 0, s, (uint16_t*)x, row_stride, (int)vocab,
                               n_rows, tail, upstream, applied);
            break;
    }
    return mrl::check_launch(fn);
}

extern "C" int mrl_grad_scale_note(const float* upstream, float* applied, float* learned, uint32_t* rescales,
                                   void* stream) {
    const char* fn = "mrl_grad_scale_note";
    MRL_REQUIRE(upstream && applied, MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    MRL_REQUIRE(mrl::aligned(upstream, 4) && mrl::aligned(applied, 4) && mrl::aligned(learned, 4) &&
                    mrl::aligned(rescales, 4),
                MRL_ERR_MISALIGNED, "%s: pointers must be 4-byte aligned", fn);
    hipLaunchKernelGGL(grad_scale_note_kernel, dim3(1), dim3(64), 0, mrl::as_stream(stream), upstream, applied, learned,
                       rescales);
    return mrl::check_launch(fn);
}

extern "C" int mrl_scale_rows_note(void* x, int dtype, int64_t n_rows, int64_t vocab, int64_t row_stride,
                                   const float* upstream, float* applied, float* learned, uint32_t* rescales,
                                   void* stream) {
    const char* fn = "mrl_scale_rows_note";
    const int eb = mrl::float_dtype_bytes(dtype);
    MRL_REQUIRE(eb != 0, MRL_ERR_UNSUPPORTED, "%s: dtype %d (want F32, BF16 or F16)", fn, dtype);
    MRL_REQUIRE(n_rows > 0 && n_rows <= 0x7fffffffLL && vocab > 0 && row_stride >= vocab, MRL_ERR_INVALID_ARG,
                "%s: n_rows=%lld vocab=%lld row_stride=%lld", fn, (long long)n_rows, (long long)vocab,
                (long long)row_stride);
    MRL_REQUIRE(x && upstream && applied, MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    MRL_REQUIRE(mrl::aligned(upstream, 4) && mrl::aligned(applied, 8) && mrl::aligned(learned, 4) &&
                    mrl::aligned(rescales, 4),
                MRL_ERR_MISALIGNED, "%s: applied must be 8-byte, the other scalars 4-byte aligned", fn);
    const int tail = flat_rows(eb, n_rows, vocab, row_stride);
    MRL_REQUIRE(vocab % (16 / eb) == 0 && mrl::aligned(x, 16) && (n_rows == 1 || (row_stride * eb) % 16 == 0),
                MRL_ERR_UNSUPPORTED, "%s: needs 16-byte aligned or dense rows", fn);
    hipStream_t s = mrl::as_stream(stream);
    const dim3 grid((unsigned)(n_rows < 8 ? 8 : (n_rows < 2048 ? n_rows : 2048))), block(256);
    switch (dtype) {
        case MRL_F32:
            hipLaunchKernelGGL(scale_rows_note_kernel<MRL_F32>, grid, block, 0, s, (float*)x, row_stride, (int)vocab,
                               n_rows, tail, upstream, applied, learned, rescales);
            break;
        case MRL_BF16:
            hipLaunchKernelGGL(scale_rows_note_kernel<MRL_BF16>, grid, block, 0, s, (uint16_t*)x, row_stride,
                               (int)vocab, n_rows, tail, upstream, applied, learned, rescales);
            break;
        default:
            hipLaunchKernelGGL(scale_rows_note_kernel<MRL_F16>, grid, block, 0, s, (uint16_t*)x, row_stride,
                               (int)vocab, n_rows, tail, upstream, applied, learned, rescales);
            break;
    }
    return mrl::check_launch(fn);
}
