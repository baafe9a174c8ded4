// Streaming vocabulary sweeps for gfx950: per-row log-softmax gather + entropy + logsumexp
// (forward, one read of the logits) and the fused dlogits (backward, one read + one write).
//
// Mapping: one workgroup per token row, 256 threads (4 wavefronts) in the backward, 256 to 1024 by the row's
// length in the forward.  A row is addressed as
// a run of 16-byte vectors from its first 128-byte line on; elements in front of it and after the last
// vector (only present for odd vocab sizes or strides) are handled with scalar loads by the first lanes.
// Each thread keeps an online (max, sum exp, sum exp*z) triple in fp32; a rescale happens at
// most once per round of vectors and only when the running maximum grows, so the steady
// state costs one convert, one FMA and one v_exp_f32 per element.  Wavefront reduction uses
// cross-lane shuffles, the wavefronts combine through LDS.
#include <stdlib.h>

#include "mrl_internal.h"
#include "row_sweep.h"
#include "seq_windows.h"
#include "vocab_common.h"

namespace {

using namespace mrl_vocab;

#ifndef MRL_VOCAB_BLOCK
#define MRL_VOCAB_BLOCK 256
#endif
#ifndef MRL_VOCAB_UNROLL
#define MRL_VOCAB_UNROLL 4
#endif
constexpr int kBlock = MRL_VOCAB_BLOCK;
constexpr int kUnroll = MRL_VOCAB_UNROLL;
// Splits a row of `vocab` elements starting at `row` into head scalars up to a 128-byte line (with vectors
// that are 16-byte aligned only, every wavefront's 1 KiB cuts two lines in half: 129 281 bf16 logits forward
// 6 437 GB/s, on lines 6 870), 16-byte vectors and tail scalars.  So the order of the fp32 sums, and their
// last bits, follow from the row's address modulo 128.
template <typename T, int kVec>
struct RowSplit {
    int head;       // scalar elements before the first vector
    int n_vec;      // aligned vectors
    int tail_begin; // element index of the first tail scalar
    __device__ __forceinline__ RowSplit(const T* row, int vocab) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(row);
        const int mis = (int)((a % 128) / sizeof(T));
        head = mis ? 128 / (int)sizeof(T) - mis : 0;
        if (head > vocab) head = vocab;
        n_vec = (vocab - head) / kVec;
        tail_begin = head + n_vec * kVec;
    }
};

// Which rows the forward scores and where their results go.  A workgroup is a row of the logits, or a cell of
// the scored windows' [batch, width] result; `row` is what it reads (-1: nothing, its results are zeros).
//
// The cells take a scoring pass to one launch, where flags for the rows, a sweep and a cut of both results were
// four: the window's three lengths are loaded at once and stand in for the flag, and only rows of a window have
// a workgroup that reads.  505 of 1 208 padded rows x 32 000 bf16 48 -> 19 us a pass, 133 rows x 8 000 45 -> 20;
// 60 779 rows x 8 000 185 -> 175; the sweep itself is bound by memory as before.
struct FlaggedRows {
    static constexpr int kCells = 1;
    const uint8_t* active;          // NULL: all
    __device__ __forceinline__ int64_t row(int64_t out) const { return active != nullptr && active[out] == 0 ? -1 : out; }
};

struct WindowCells {
    static constexpr int kCells = 1;
    mrl::SeqWindows seqs;
    uint32_t width;
    int64_t n_rows;
    __device__ __forceinline__ int64_t row(int64_t out) const {
        const uint32_t i = (uint32_t)out / width, j = (uint32_t)out - i * width;
        int64_t start, n;
        seqs.window(i, start, n);
        const int64_t t = start + j;
        return (int64_t)j < n && t >= 0 && t < n_rows ? t : -1;
    }
};

// Many cells (see launch_fwd_shape).  An empty one keeps a workgroup's registers for the microsecond that the loads of
// its window take, and a CU has room for two workgroups of 1024 threads but eight of 256: a pass over windows with few
// live cells consists of that.  So a workgroup of 512 or 1024 threads takes kCells = 2 or 4 cells of a sequence, a half
// or quarter of the width apart: the live ones are the first, and fall to different workgroups.
template <int kOfUnit>
struct ManyCells {
    static constexpr int kCells = kOfUnit;
    mrl::SeqWindows seqs;
    uint32_t width, step;           // step: units of a sequence, width / kCells rounded up
    int64_t n_rows;
    struct Unit {
        int64_t first, start, n;    // of the sequence: its first cell, its window
        uint32_t j;
    };
    __device__ __forceinline__ Unit unit(uint32_t u) const {
        const uint32_t i = u / step;
        Unit r;
        r.j = u - i * step;
        r.first = (int64_t)i * width;
        seqs.window(i, r.start, r.n);
        return r;
    }
    // whether there is a cell c of the unit; its place and the row that it reads
    __device__ __forceinline__ bool cell(const Unit& u, int c, int64_t& out, int64_t& row) const {
        const uint32_t j = u.j + (uint32_t)c * step;
        const int64_t t = u.start + j;
        out = u.first + j;
        row = (int64_t)j < u.n && t >= 0 && t < n_rows ? t : -1;
        return j < width;
    }
};

// Log-prob, entropy and log-sum-exp of row r, by the whole workgroup.
template <int DT, typename LabelT, bool kEntropy, int kBlk, int kDeep>
__device__ __forceinline__ void score_row(
    const typename Elem<DT>::T* __restrict__ logits, int64_t row_stride, int vocab,
    const LabelT* __restrict__ labels, int64_t r, int64_t out, float inv_t,
    float* __restrict__ logp, float* __restrict__ entropy, float* __restrict__ lse_out, Stats* lds, const int tid) {
    using E = Elem<DT>;
    using T = typename E::T;
    constexpr int kVec = E::kVec;
    const T* row = logits + r * row_stride;
    const float k = inv_t * kLog2e;

    // label logit: issued first so that its latency hides behind the sweep
    const int64_t y = (int64_t)labels[r];
    const bool y_ok = (y >= 0) && (y < (int64_t)vocab);
    float z_y = 0.f;
    if (tid == 0 && y_ok) z_y = E::load(row + y);

    const RowSplit<T, kVec> sp(row, vocab);
    const u32x4* vec = reinterpret_cast<const u32x4*>(row + sp.head);

    Stats st = {kMaxInit, 0.f, 0.f};

    // rounds of kDeep vectors a thread, all requested before any is used
    auto request = [&](u32x4 (&v)[kDeep], int base) {
#pragma unroll
        for (int q = 0; q < kDeep; ++q) v[q] = __builtin_nontemporal_load(vec + base + q * kBlk + tid);
    };
    auto add_round = [&](const u32x4 (&v)[kDeep]) {
        float z[kDeep][kVec];
        float vmax = st.m;
#pragma unroll
        for (int q = 0; q < kDeep; ++q) {
            E::unpack(v[q], z[q]);
#pragma unroll
            for (int i = 0; i < kVec; ++i) vmax = fmaxf(vmax, z[q][i]);
        }
        grow_max<kEntropy>(st, vmax, k);
        const float mk = st.m * k;
#pragma unroll
        for (int q = 0; q < kDeep; ++q) {
#pragma unroll
            for (int i = 0; i < kVec; ++i) add_one<kEntropy>(st, z[q][i], k, mk);
        }
    };
    constexpr int kRound = kBlk * kDeep;
    const int n_full = sp.n_vec / kRound * kRound;
    for (int base = 0; base < n_full - kRound; base += kRound) {
        u32x4 v[kDeep];
        request(v, base);
        add_round(v);
    }
    // The last whole round, and with it what is left of the row, of which a thread may have fewer vectors or none:
    // range-checked.  A round of its own for the rest, however short, was waited for like any other: us a pass, 2 903
    // rows x 33 024 bf16 (two rounds and 32 vectors) 37.5 -> 34.5, x 30 000 34.3 -> 32.4, 662 x 32 000 14.8 -> 13.5.
    // Where there is no rest few rows pay for it all the same: 300 x 16 384 fp32 6.1 -> 6.2, 1 000 10.8 -> 11.0, and 11.2
    // if the rest's tests of a lane's vectors are gone through as well.
    {
        const mrl::rsrc_t rest = mrl::make_rsrc(vec + n_full, (uint32_t)(sp.n_vec - n_full) * 16u);
        u32x4 v[kDeep], w[kDeep];
        if (n_full > 0) request(v, n_full - kRound);
#pragma unroll
        for (int q = 0; q < kDeep; ++q) w[q] = mrl::buf_load_nt(rest, (uint32_t)(q * kBlk + tid) * 16u);
        if (n_full > 0) add_round(v);
        if (n_full != sp.n_vec)
#pragma unroll
        for (int q = 0; q < kDeep; ++q) {
            if (n_full + q * kBlk + tid < sp.n_vec) {
                float z[kVec];
                E::unpack(w[q], z);
                float vmax = st.m;
#pragma unroll
                for (int i = 0; i < kVec; ++i) vmax = fmaxf(vmax, z[i]);
                grow_max<kEntropy>(st, vmax, k);
                const float mk = st.m * k;
#pragma unroll
                for (int i = 0; i < kVec; ++i) add_one<kEntropy>(st, z[i], k, mk);
            }
        }
    }
    // head and tail scalars (absent when the row starts on a line and vocab % kVec == 0)
    {
        const int n_edge = sp.head + (vocab - sp.tail_begin);
        if (tid < n_edge) {
            const int j = tid < sp.head ? tid : sp.tail_begin + (tid - sp.head);
            const float z = E::load(row + j);
            grow_max<kEntropy>(st, z, k);
            add_one<kEntropy>(st, z, k, st.m * k);
        }
    }

    const Stats tot = block_reduce<kEntropy, kBlk / 64>(st, k, lds);
    if (tid == 0) {
        // natural-log units of z' = z * inv_t
        const float lse = (tot.m * k + fast_log2(tot.s)) * kLn2;
        const float picked = y_ok ? z_y * inv_t : tot.m * inv_t;
        logp[out] = picked - lse;
        // the cells' entropies are zeros where they are not wanted
        if (kEntropy) entropy[out] = lse - (tot.u / tot.s) * inv_t;
        else if (entropy) entropy[out] = 0.f;
        if (lse_out) lse_out[out] = lse;
    }
}

template <int DT, typename LabelT, bool kEntropy, int kBlk, int kDeep, typename Rows>
__global__ __launch_bounds__(kBlk) void vocab_fwd_kernel(
    const typename Elem<DT>::T* __restrict__ logits, int64_t row_stride, int vocab,
    const LabelT* __restrict__ labels, Rows rows, uint32_t first, float inv_t,
    float* __restrict__ logp, float* __restrict__ entropy, float* __restrict__ lse_out) {
    __shared__ Stats lds[kBlk / 64];
    auto no_row = [&](int64_t out) {
        logp[out] = 0.f;
        if (entropy) entropy[out] = 0.f;
        if (lse_out) lse_out[out] = 0.f;
    };
    auto score = [&](int64_t r, int64_t out, int tid) {
        score_row<DT, LabelT, kEntropy, kBlk, kDeep>(logits, row_stride, vocab, labels, r, out, inv_t, logp, entropy, lse_out, lds,
                                                     tid);
    };
    if constexpr (Rows::kCells == 1) {
        const int64_t out = first + blockIdx.x, r = rows.row(out);
        if (r < 0) {
            if (threadIdx.x == 0) no_row(out);
            return;
        }
        score(r, out, (int)threadIdx.x);
    } else {
        const auto unit = rows.unit(first + blockIdx.x);
        int64_t out, r;
        if (threadIdx.x < Rows::kCells && rows.cell(unit, (int)threadIdx.x, out, r) && r < 0) no_row(out);
        if (unit.n <= (int64_t)unit.j) return;          // then no later one has a row either
#pragma unroll 1
        for (int c = 0; c < Rows::kCells; ++c) {
            if (!rows.cell(unit, c, out, r)) return;
            if (r < 0) continue;
            int tid = (int)threadIdx.x;
            // what follows from it is computed for each cell: kept from cell to cell it would take the registers of a
            // workgroup on every CU (79 instead of 62 with 512 threads and entropies)
            asm volatile("" : "+v"(tid));
            score(r, out, tid);
            __syncthreads();                // the partials have been read
        }
    }
}

// dlogits = e * (c0 + c1 * z) with e = 2^(z*k - lse*log2e), plus g at the label:
//   c0 = inv_t * (-g_lp + g_H * (lse - H)),  c1 = -g_H * inv_t^2
// The row is split by the alignment of the INPUT row; the host only selects this kernel when
// the output row reaches 16-byte alignment at the same element.  Built for DT_OUT == DT_IN and
// for DT_OUT == F32, so one input vector maps to one or two output vectors.
template <int DT_IN, int DT_OUT, typename LabelT, bool kEntropy>
__global__ __launch_bounds__(kBlock) void vocab_bwd_kernel(
    const typename Elem<DT_IN>::T* logits, int64_t row_stride, int vocab,
    const LabelT* __restrict__ labels, float inv_t, const float* __restrict__ lse_in,
    const float* __restrict__ ent_in, const float* __restrict__ g_logp,
    const float* __restrict__ g_entropy, typename Elem<DT_OUT>::T* dlogits, int64_t d_stride) {
    using EI = Elem<DT_IN>;
    using EO = Elem<DT_OUT>;
    using TI = typename EI::T;
    using TO = typename EO::T;
    constexpr int kStep = EI::kVec;
    constexpr int kVecO = EO::kVec;
    static_assert(kStep % kVecO == 0, "an input vector must cover whole output vectors");
    constexpr int kOutPer = kStep / kVecO;

    const int64_t r = blockIdx.x;
    const int tid = threadIdx.x;
    const TI* row = logits + r * row_stride;
    TO* drow = dlogits + r * d_stride;

    const float g_lp = g_logp ? g_logp[r] : 0.f;
    const float g_h = (kEntropy && g_entropy) ? g_entropy[r] : 0.f;
    const bool dead = (g_lp == 0.f) && (g_h == 0.f);

    const float k = inv_t * kLog2e;
    float lse2 = 0.f, c0 = 0.f, c1 = 0.f;
    if (!dead) {
        const float lse = lse_in[r];
        lse2 = lse * kLog2e;
        c0 = -g_lp * inv_t;
        if (kEntropy) {
            c0 = inv_t * (-g_lp + g_h * (lse - ent_in[r]));
            c1 = -g_h * inv_t * inv_t;
        }
    }
    const int64_t y = (int64_t)labels[r];
    const bool y_ok = (y >= 0) && (y < (int64_t)vocab) && !dead;
    const float g_onehot = g_lp * inv_t;

    auto grad_of = [&](float z) -> float {
        const float e = fast_exp2(__builtin_fmaf(z, k, -lse2));
        const float w = kEntropy ? __builtin_fmaf(c1, z, c0) : c0;
        return e * w;
    };

    const RowSplit<TI, kStep> sp(row, vocab);
    const u32x4* ivec = reinterpret_cast<const u32x4*>(row + sp.head);
    u32x4* ovec = reinterpret_cast<u32x4*>(drow + sp.head);
    const bool y_in_body = y_ok && y >= sp.head && y < sp.tail_begin;
    const int y_vec = y_in_body ? (int)((y - sp.head) / kStep) : -1;
    const int y_lane = y_in_body ? (int)((y - sp.head) % kStep) : 0;

    if (dead) {
        const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
        const int n_out = sp.n_vec * kOutPer;
        for (int idx = tid; idx < n_out; idx += kBlock) __builtin_nontemporal_store(zero, ovec + idx);
    } else {
        auto do_vec = [&](int idx, const u32x4& vin) {
            float z[kStep];
            float g[kStep];
            EI::unpack(vin, z);
#pragma unroll
            for (int i = 0; i < kStep; ++i) g[i] = grad_of(z[i]);
            if (idx == y_vec) {
#pragma unroll
                for (int i = 0; i < kStep; ++i)
                    if (i == y_lane) g[i] += g_onehot;
            }
#pragma unroll
            for (int p = 0; p < kOutPer; ++p) {
                float part[kVecO];
#pragma unroll
                for (int i = 0; i < kVecO; ++i) part[i] = g[p * kVecO + i];
                __builtin_nontemporal_store(EO::pack(part), ovec + (int64_t)idx * kOutPer + p);
            }
        };
        const int group = kBlock * kUnroll;
        const int n_full = (sp.n_vec / group) * group;
        for (int base = 0; base < n_full; base += group) {
            u32x4 v[kUnroll];
#pragma unroll
            for (int q = 0; q < kUnroll; ++q) v[q] = __builtin_nontemporal_load(ivec + base + q * kBlock + tid);
#pragma unroll
            for (int q = 0; q < kUnroll; ++q) do_vec(base + q * kBlock + tid, v[q]);
        }
        for (int idx = n_full + tid; idx < sp.n_vec; idx += kBlock) {
            const u32x4 v = __builtin_nontemporal_load(ivec + idx);
            do_vec(idx, v);
        }
    }
    // head and tail scalars
    const int n_edge = sp.head + (vocab - sp.tail_begin);
    if (tid < n_edge) {
        const int j = tid < sp.head ? tid : sp.tail_begin + (tid - sp.head);
        float g = 0.f;
        if (!dead) {
            g = grad_of(EI::load(row + j));
            if (y_ok && (int64_t)j == y) g += g_onehot;
        }
        EO::store(drow + j, g);
    }
}

// Fallback for rows whose input and output are not misaligned alike: scalar accesses.
template <int DT_IN, int DT_OUT, typename LabelT, bool kEntropy>
__global__ __launch_bounds__(kBlock) void vocab_bwd_scalar_kernel(
    const typename Elem<DT_IN>::T* logits, int64_t row_stride, int vocab,
    const LabelT* __restrict__ labels, float inv_t, const float* __restrict__ lse_in,
    const float* __restrict__ ent_in, const float* __restrict__ g_logp,
    const float* __restrict__ g_entropy, typename Elem<DT_OUT>::T* dlogits, int64_t d_stride) {
    using EI = Elem<DT_IN>;
    using EO = Elem<DT_OUT>;
    const int64_t r = blockIdx.x;
    const typename EI::T* row = logits + r * row_stride;
    typename EO::T* drow = dlogits + r * d_stride;
    const float g_lp = g_logp ? g_logp[r] : 0.f;
    const float g_h = (kEntropy && g_entropy) ? g_entropy[r] : 0.f;
    const bool dead = (g_lp == 0.f) && (g_h == 0.f);
    const float k = inv_t * kLog2e;
    float lse2 = 0.f, c0 = 0.f, c1 = 0.f;
    if (!dead) {
        const float lse = lse_in[r];
        lse2 = lse * kLog2e;
        c0 = -g_lp * inv_t;
        if (kEntropy) {
            c0 = inv_t * (-g_lp + g_h * (lse - ent_in[r]));
            c1 = -g_h * inv_t * inv_t;
        }
    }
    const int64_t y = (int64_t)labels[r];
    for (int j = threadIdx.x; j < vocab; j += kBlock) {
        float g = 0.f;
        if (!dead) {
            const float z = EI::load(row + j);
            const float e = fast_exp2(__builtin_fmaf(z, k, -lse2));
            g = e * (kEntropy ? __builtin_fmaf(c1, z, c0) : c0);
            if ((int64_t)j == y) g += g_lp * inv_t;
        }
        EO::store(drow + j, g);
    }
}

// ----------------------------------------------------------------------------- host dispatch
struct FwdArgs {
    const void* logits; int logits_dtype; int64_t vocab, row_stride;
    const void* labels; int labels_dtype;
    float inv_t;
    int64_t n_out;                  // rows or cells
    bool with_entropy;
    float *logp, *entropy, *lse;
    hipStream_t stream;
};

template <int DT, typename LabelT, int kBlk, int kDeep, typename Rows>
int launch_fwd_units(const char* fn, const FwdArgs& a, const Rows& rows, int64_t n_units) {
    using T = typename Elem<DT>::T;
    // a launch has fewer than 2^32 threads: more rows or cells (of a window mostly empty ones) take several
    constexpr int64_t kMost = 0xffffffffLL / kBlk;
    for (int64_t first = 0; first < n_units; first += kMost) {
        const dim3 grid((unsigned)(n_units - first < kMost ? n_units - first : kMost)), block(kBlk);
#define MRL_FWD_LAUNCH(ENT)                                                                                           \
    hipLaunchKernelGGL((vocab_fwd_kernel<DT, LabelT, ENT, kBlk, kDeep, Rows>), grid, block, 0, a.stream,              \
                       (const T*)a.logits, a.row_stride, (int)a.vocab, (const LabelT*)a.labels, rows, (uint32_t)first, \
                       a.inv_t, a.logp, a.entropy, a.lse)
        if (a.with_entropy) MRL_FWD_LAUNCH(true);
        else MRL_FWD_LAUNCH(false);
#undef MRL_FWD_LAUNCH
        const int rc = mrl::check_launch(fn);
        if (rc != MRL_OK) return rc;
    }
    return MRL_OK;
}

template <int DT, typename LabelT, int kBlk, int kDeep>
int launch_fwd_shape(const char* fn, const FwdArgs& a, const FlaggedRows& rows) {
    return launch_fwd_units<DT, LabelT, kBlk, kDeep>(fn, a, rows, a.n_out);
}

// A cell to a workgroup, or several: where most of the cells are known to be empty, or so many, in long windows, that
// their rows keep the chip busy either way.  us a pass over bf16 windows, with 256 threads and a cell each / 512 or 1024
// and a cell each / as it is: 256 x 8 192 cells with 7 rows to a sequence, 152 064 logits 1 123 / 4 263 / 1 162, 32 000
// 1 055 / 2 066 / 998; 16 x 2 048 with 255, 57 344 75 / 76 / 73; with entropies, 20 x 2 048 of which two thirds have rows,
// 152 064 964 / 949 / 938.  Several cells over fewer of them leave CUs idle (2 500 with rows x 152 064 118 / 112 / 124),
// and in short windows the rows of a workgroup are many (384 of up to 78 x 126 784 785 / 760 / 789); where one in ten has
// a row neither shows, 4 x 1 024 x 152 064 32 / 29 / 23.
template <int DT, typename LabelT, int kBlk, int kDeep>
int launch_fwd_shape(const char* fn, const FwdArgs& a, const WindowCells& w) {
    if constexpr (kBlk > 256) {
        constexpr int kCells = kBlk / 256;
        if ((a.n_out >= 16384 && w.width >= 512) || (a.n_out >= 4096 && a.n_out >= 4 * w.n_rows)) {
            const uint32_t step = (w.width + kCells - 1) / kCells;
            const ManyCells<kCells> rows = {w.seqs, w.width, step, w.n_rows};
            return launch_fwd_units<DT, LabelT, kBlk, kDeep>(fn, a, rows, a.n_out / w.width * step);
        }
    }
    return launch_fwd_units<DT, LabelT, kBlk, kDeep>(fn, a, w, a.n_out);
}

// Threads of a row's workgroup and vectors a thread and round, by the row's length alone, so that a row's result
// does not depend on how many rows there are.  Few rows are bound by the rounds that a thread waits for one after the
// other, which more threads make fewer of: 98 x 152 064 bf16 20.2 -> 12.4 us with 1024, 116 x 129 280 18.0 -> 11.9, 49 x
// 152 064 fp32 29.5 -> 15.6.  Many are bound by memory without entropies whatever the shape, and with them by the
// arithmetic as well, which larger workgroups overlap less: fewer of them are on a CU, and more of a row goes with the
// rest.  Windows of which four fifths have rows, sigma 3, us without and with entropies, 256 / 512 / 1024 threads:
//   16 bits  4 000 vectors, 38 069 rows 355 / 350 / 412, 358 / 363 to 375 / 447; 2 022 rows 23 / 22 / 27, 24 / 23 / 28
//            6 500, 23 417 rows 351 / 346 / 365, 354 / 351 / 400; 2 022 36 / 34 / 34, 38 / 35 / 37; 209 9.7 / 7.0 / 6.6
//            8 192, 18 583 rows 357 / 347 / 353, 360 / 348 / 373; 2 022 46 / 42 / 41, 48 / 44 / 44; 209 11 / 8.1 / 7.1
//            11 500, 13 227 rows 352 / 349 / 347, 355 / 349 / 354; 2 022 64 / 58 / 56, 66 / 60 / 58; 209 16 / 10 / 8.6
//            19 008, 8 002 rows 357 / 353 / 346, 360 / 355 / 346; 2 022 104 / 95 / 92; 209 25 / 16 / 12
//   fp32     4 096, 37 185 rows 351 / 357 / 373; 8 000, 19 026 rows 353 / 350 / 348, 2 022 41 / 40 / 39, 209 8.5 / 6.4 / 6.2
// A CU holds two workgroups of 1024 threads: 601 rows of 152 064 bf16, a few more than two to each, take 33 us, and with
// 512 threads 29.  1024 threads with 4 vectors: 7 964 vectors 294 us for 2 GB (286 with 3), 12 500 and more within 0.5 %.
// Rows of 512 vectors and less would gain from a wavefront each (4 000 bf16 458 -> 324), but entropies of merged
// vocabulary shards then differ by up to 2.3e-5 from the whole row's, more than they may.
template <int DT, typename LabelT, typename Rows>
int launch_fwd(const char* fn, const FwdArgs& a, const Rows& rows) {
    const int64_t n_vec = a.vocab / Elem<DT>::kVec;
    if (n_vec <= 4096) return launch_fwd_shape<DT, LabelT, 256, 4>(fn, a, rows);
    if (n_vec <= (DT == MRL_F32 ? 7168 : 11264)) return launch_fwd_shape<DT, LabelT, 512, 4>(fn, a, rows);
    return launch_fwd_shape<DT, LabelT, 1024, 3>(fn, a, rows);
}

template <typename Rows>
int dispatch_fwd(const char* fn, const FwdArgs& a, const Rows& rows) {
#define MRL_FWD(DT) \
    (a.labels_dtype == MRL_I32 ? launch_fwd<DT, int32_t>(fn, a, rows) : launch_fwd<DT, int64_t>(fn, a, rows))
    switch (a.logits_dtype) {
        case MRL_F32: return MRL_FWD(MRL_F32);
        case MRL_BF16: return MRL_FWD(MRL_BF16);
        default: return MRL_FWD(MRL_F16);
    }
#undef MRL_FWD
}

template <int DT_IN, int DT_OUT, typename LabelT>
int launch_bwd(const void* logits, int64_t n_rows, int vocab, int64_t row_stride, const void* labels,
               float inv_t, const float* lse, const float* ent, const float* g_lp, const float* g_h,
               void* dlogits, int64_t d_stride, bool vector_ok, hipStream_t stream) {
    using TI = typename Elem<DT_IN>::T;
    using TO = typename Elem<DT_OUT>::T;
    const dim3 grid((unsigned)n_rows), block(kBlock);
    const bool with_entropy = (g_h != nullptr);
#define MRL_BWD_LAUNCH(KERNEL, ENT)                                                                     \
    hipLaunchKernelGGL((KERNEL<DT_IN, DT_OUT, LabelT, ENT>), grid, block, 0, stream, (const TI*)logits, \
                       row_stride, vocab, (const LabelT*)labels, inv_t, lse, ent, g_lp, g_h,            \
                       (TO*)dlogits, d_stride)
    if (vector_ok) {
        if (with_entropy) MRL_BWD_LAUNCH(vocab_bwd_kernel, true);
        else MRL_BWD_LAUNCH(vocab_bwd_kernel, false);
    } else {
        if (with_entropy) MRL_BWD_LAUNCH(vocab_bwd_scalar_kernel, true);
        else MRL_BWD_LAUNCH(vocab_bwd_scalar_kernel, false);
    }
#undef MRL_BWD_LAUNCH
    return mrl::check_launch("mrl_vocab_logprob_bwd");
}

int check_common(const char* fn, const void* logits, int logits_dtype, int64_t n_rows, int64_t vocab,
                 int64_t row_stride, const void* labels, int labels_dtype, float inv_t) {
    MRL_REQUIRE(n_rows >= 0 && vocab > 0, MRL_ERR_INVALID_ARG, "%s: n_rows=%lld vocab=%lld", fn,
                (long long)n_rows, (long long)vocab);
    MRL_REQUIRE(n_rows <= 0x7fffffffLL, MRL_ERR_UNSUPPORTED, "%s: n_rows=%lld exceeds 2^31 - 1", fn,
                (long long)n_rows);
    MRL_REQUIRE(vocab <= (1LL << 30), MRL_ERR_UNSUPPORTED, "%s: vocab=%lld exceeds 2^30", fn, (long long)vocab);
    const int eb = mrl::float_dtype_bytes(logits_dtype);
    MRL_REQUIRE(eb != 0, MRL_ERR_UNSUPPORTED, "%s: logits dtype %d (want F32, BF16 or F16)", fn, logits_dtype);
    MRL_REQUIRE(mrl::int_dtype_bytes(labels_dtype) != 0, MRL_ERR_UNSUPPORTED,
                "%s: labels dtype %d (want I32 or I64)", fn, labels_dtype);
    MRL_REQUIRE(row_stride >= vocab, MRL_ERR_INVALID_ARG, "%s: row_stride=%lld < vocab=%lld", fn,
                (long long)row_stride, (long long)vocab);
    if (n_rows == 0) return MRL_OK;
    MRL_REQUIRE(logits && labels, MRL_ERR_INVALID_ARG, "%s: NULL logits or labels", fn);
    MRL_REQUIRE(mrl::aligned(logits, eb), MRL_ERR_MISALIGNED, "%s: logits not aligned to %d bytes", fn, eb);
    MRL_REQUIRE(mrl::aligned(labels, mrl::int_dtype_bytes(labels_dtype)), MRL_ERR_MISALIGNED,
                "%s: labels misaligned", fn);
    MRL_REQUIRE(inv_t > 0.f && inv_t < 1.0e6f, MRL_ERR_INVALID_ARG, "%s: inv_temperature=%g must be in (0, 1e6)",
                fn, (double)inv_t);
    return MRL_OK;
}

}  // namespace

extern "C" int mrl_vocab_logprob_fwd(const void* logits, int logits_dtype, int64_t n_rows, int64_t vocab,
                                     int64_t row_stride, const void* labels, int labels_dtype,
                                     const uint8_t* row_active, float inv_temperature, float* logp,
                                     float* entropy, float* lse, void* stream) {
    const char* fn = "mrl_vocab_logprob_fwd";
    int rc = check_common(fn, logits, logits_dtype, n_rows, vocab, row_stride, labels, labels_dtype,
                          inv_temperature);
    if (rc != MRL_OK) return rc;
    if (n_rows == 0) return MRL_OK;
    MRL_REQUIRE(logp != nullptr, MRL_ERR_INVALID_ARG, "%s: logp is NULL", fn);
    MRL_REQUIRE(mrl::aligned(logp, 4) && mrl::aligned(entropy, 4) && mrl::aligned(lse, 4), MRL_ERR_MISALIGNED,
                "%s: fp32 outputs misaligned", fn);
    const FwdArgs a = {logits, logits_dtype, vocab, row_stride, labels, labels_dtype, inv_temperature, n_rows,
                       entropy != nullptr, logp, entropy, lse, mrl::as_stream(stream)};
    return dispatch_fwd(fn, a, FlaggedRows{row_active});
}

extern "C" int mrl_window_logprob(const void* logits, int logits_dtype, int64_t n_rows, int64_t vocab,
                                  int64_t row_stride, const void* labels, int labels_dtype, float inv_temperature,
                                  int layout, int64_t batch, int64_t width, const int32_t* seqlens,
                                  const int32_t* cu_seqlens_padded, int64_t padded_s, const void* prompt_length,
                                  int prompt_dtype, const void* response_length, int response_dtype, int want_entropy,
                                  float* logp, float* entropy, void* stream) {
    const char* fn = "mrl_window_logprob";
    int rc = check_common(fn, logits, logits_dtype, n_rows, vocab, row_stride, labels, labels_dtype, inv_temperature);
    if (rc != MRL_OK) return rc;
    const mrl::SeqWindows q = {layout == 0, seqlens, cu_seqlens_padded, padded_s, prompt_length, prompt_dtype,
                               response_length, response_dtype};
    rc = mrl::check_seq_windows(fn, q, batch, width, n_rows);
    if (rc != MRL_OK || batch == 0 || width == 0) return rc;
    MRL_REQUIRE(width <= 0x7fffffffLL / batch, MRL_ERR_UNSUPPORTED, "%s: batch=%lld x width=%lld exceeds 2^31 - 1", fn,
                (long long)batch, (long long)width);
    MRL_REQUIRE(logp && entropy, MRL_ERR_INVALID_ARG, "%s: NULL output", fn);
    MRL_REQUIRE(mrl::aligned(logp, 4) && mrl::aligned(entropy, 4), MRL_ERR_MISALIGNED, "%s: fp32 outputs misaligned", fn);
    const FwdArgs a = {logits, logits_dtype, vocab, row_stride, labels, labels_dtype, inv_temperature, batch * width,
                       want_entropy != 0, logp, entropy, nullptr, mrl::as_stream(stream)};
    return dispatch_fwd(fn, a, WindowCells{q, (uint32_t)width, n_rows});
}

extern "C" int mrl_vocab_logprob_bwd(const void* logits, int logits_dtype, int64_t n_rows, int64_t vocab,
                                     int64_t row_stride, const void* labels, int labels_dtype,
                                     float inv_temperature, const float* lse, const float* entropy,
                                     const float* g_logp, const float* g_entropy, void* dlogits,
                                     int dlogits_dtype, int64_t dlogits_row_stride, void* stream) {
    const char* fn = "mrl_vocab_logprob_bwd";
    int rc = check_common(fn, logits, logits_dtype, n_rows, vocab, row_stride, labels, labels_dtype,
                          inv_temperature);
    if (rc != MRL_OK) return rc;
    const int ob = mrl::float_dtype_bytes(dlogits_dtype);
    MRL_REQUIRE(ob != 0, MRL_ERR_UNSUPPORTED, "%s: dlogits dtype %d (want F32, BF16 or F16)", fn, dlogits_dtype);
    MRL_REQUIRE(dlogits_row_stride >= vocab, MRL_ERR_INVALID_ARG, "%s: dlogits_row_stride=%lld < vocab", fn,
                (long long)dlogits_row_stride);
    if (n_rows == 0) return MRL_OK;
    MRL_REQUIRE(dlogits != nullptr, MRL_ERR_INVALID_ARG, "%s: dlogits is NULL", fn);
    MRL_REQUIRE(mrl::aligned(dlogits, ob), MRL_ERR_MISALIGNED, "%s: dlogits misaligned", fn);
    MRL_REQUIRE(lse != nullptr, MRL_ERR_INVALID_ARG, "%s: lse is NULL", fn);
    MRL_REQUIRE(g_entropy == nullptr || entropy != nullptr, MRL_ERR_INVALID_ARG,
                "%s: g_entropy given without the forward's entropy", fn);
    // only same-dtype and fp32-output combinations are built
    MRL_REQUIRE(dlogits_dtype == logits_dtype || dlogits_dtype == MRL_F32, MRL_ERR_UNSUPPORTED,
                "%s: dlogits dtype %d must equal the logits dtype %d or be F32", fn, dlogits_dtype, logits_dtype);
    if (dlogits == logits) {
        MRL_REQUIRE(dlogits_dtype == logits_dtype && dlogits_row_stride == row_stride, MRL_ERR_INVALID_ARG,
                    "%s: in-place backward needs identical dtype and stride", fn);
    } else {
        // partial overlap would corrupt rows that other workgroups still read
        const char* a = (const char*)logits;
        const char* b = (const char*)dlogits;
        const int64_t a_bytes = ((n_rows - 1) * row_stride + vocab) * mrl::float_dtype_bytes(logits_dtype);
        const int64_t b_bytes = ((n_rows - 1) * dlogits_row_stride + vocab) * ob;
        MRL_REQUIRE(a + a_bytes <= b || b + b_bytes <= a, MRL_ERR_INVALID_ARG,
                    "%s: dlogits partially overlaps logits", fn);
    }
    // vector path: the kernel splits rows by the input pointer, so every output row must be aligned to 16
    // bytes at the element where its input row reaches a line - which it is if the two start at the same
    // element of an output vector and their strides keep them there, whatever the vocabulary (32 003 bf16
    // logits 2 744 -> 5 290 GB/s; single entries before)
    const int ib = mrl::float_dtype_bytes(logits_dtype);
    bool vector_ok;
    {
        const int64_t vo = 16 / ob;
        const int64_t first_in = (int64_t)((uintptr_t)logits / ib), first_out = (int64_t)((uintptr_t)dlogits / ob);
        vector_ok = (first_in - first_out) % vo == 0 && (n_rows == 1 || (row_stride - dlogits_row_stride) % vo == 0);
    }
    hipStream_t s = mrl::as_stream(stream);
    const int v = (int)vocab;
    // rows from 16 KiB on, same dtype in and out: the streaming kernel (one vector per thread)
    if (dlogits_dtype == logits_dtype &&
        mrl::bwd_chunks_supported(logits_dtype, vocab, logits, row_stride, dlogits, dlogits_row_stride, n_rows)) {
        const mrl::BwdArgs a = {logits, logits_dtype, n_rows, vocab, row_stride, labels, labels_dtype, inv_temperature,
                                lse, entropy, g_logp, g_entropy, dlogits, dlogits_row_stride, s};
        return mrl::launch_bwd_chunks(a);
    }
#define MRL_BWD(DI, DO)                                                                                      \
    (labels_dtype == MRL_I32                                                                                 \
         ? launch_bwd<DI, DO, int32_t>(logits, n_rows, v, row_stride, labels, inv_temperature, lse, entropy, \
                                       g_logp, g_entropy, dlogits, dlogits_row_stride, vector_ok, s)         \
         : launch_bwd<DI, DO, int64_t>(logits, n_rows, v, row_stride, labels, inv_temperature, lse, entropy, \
                                       g_logp, g_entropy, dlogits, dlogits_row_stride, vector_ok, s))
    if (logits_dtype == MRL_F32) return MRL_BWD(MRL_F32, MRL_F32);
    if (logits_dtype == MRL_BF16)
        return dlogits_dtype == MRL_BF16 ? MRL_BWD(MRL_BF16, MRL_BF16) : MRL_BWD(MRL_BF16, MRL_F32);
    return dlogits_dtype == MRL_F16 ? MRL_BWD(MRL_F16, MRL_F16) : MRL_BWD(MRL_F16, MRL_F32);
#undef MRL_BWD
}
