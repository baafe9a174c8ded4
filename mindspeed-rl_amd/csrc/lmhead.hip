// Fused lm_head + log-prob for gfx950: streams W_vocab x hidden^T tiles through bf16 MFMA and
// keeps an online log-sum-exp per token, so the [T, V] logits are never written to memory.
//
//   logits[t, v] = sum_k hidden[t, k] * W[v, k]        (bf16 operands, fp32 accumulate)
//   lse, logp[label], entropy exactly as the vocabulary sweep computes them, on the fp32 logits
//
// Mapping.  The product runs on the shared tile loop of lmhead_tile.h (256 x 256 tiles, one
// wavefront per SIMD with a 128 x 128 sub-tile of v_mfma_f32_16x16x32_bf16 blocks, operands straight
// from global memory into LDS) with the vocabulary as the MFMA's M and the tokens as its
// N: in the 16x16 result layout a lane then owns ONE token column of each block and 4 vocabulary
// rows, so the softmax statistics of a token accumulate inside a lane.  The vocabulary is cut into leaves
// of a few tiles (VocabLeaves) that follow from the vocabulary alone; every leaf leaves its own partial
// statistics per token, and a second kernel merges them in a fixed order, together with the label
// logit (one fp32 dot product per token).  So a token's result does not depend on which other tokens
// share the call, whatever the work distribution is: units of 256 tokens by a group of leaves, as many
// groups as fill the chip (pick_groups), walked by one persistent workgroup per CU.
#include <atomic>
#include <type_traits>

#include "lmhead_tile.h"
#include "mrl_internal.h"
#include "vocab_common.h"

// Partial statistics of mrl_lmhead_logprob_fwd_static: device memory that belongs to the library,
// one copy per GPU that runs it, held until the process ends.  In host code this name is only a
// handle for hipGetSymbolAddress; kernels get the address that call returns.  Its size decides into how many
// slices a call is cut (32 768 tokens x 152 064 x 3 584, ms at 8 / 16 / 32 / 64 MiB: 27.7 / 26.9 / 26.3 / 25.2).
#define MRL_LMHEAD_STATIC_MAX_TOKENS 65536
#define MRL_LMHEAD_STATIC_BYTES (64 << 20)
static __device__ __align__(256) float scratch[MRL_LMHEAD_STATIC_BYTES / sizeof(float)];

namespace {

using namespace mrl_vocab;

// The leaves of a vocabulary: 1 to 3 tiles of 256 rows, more where that would make more than kMaxLeaves of
// them.  A call with few tokens can be spread over no more workgroups than there are leaves (162 tokens x
// 95 920 entries: 187 us with leaves of 2 tiles, 240 us with 3), but a leaf costs its statistics' last
// reduction (19 202 x 148 784 at 1088 hidden: 5.30 ms with 2, 5.20 ms with 3) and 12 bytes per token.
constexpr int kMaxLeaves = 256;
static_assert(kMaxLeaves * 3 * sizeof(float) <= MRL_LMHEAD_GROUPS * 16, "what the header promises to suffice");
struct VocabLeaves {
    int n_tiles, tiles_per_leaf, n;
    __host__ __device__ explicit VocabLeaves(int64_t vocab) {
        n_tiles = (int)((vocab + mrl_tile::BM - 1) / mrl_tile::BM);
        tiles_per_leaf = (n_tiles + kMaxLeaves - 1) / kMaxLeaves;
        const int least = n_tiles <= 128 ? 1 : (n_tiles <= 384 ? 2 : 3);
        if (tiles_per_leaf < least) tiles_per_leaf = least;
        n = (n_tiles + tiles_per_leaf - 1) / tiles_per_leaf;
    }
    __host__ __device__ int begin_tile(int leaf) const {
        const int t = leaf * tiles_per_leaf;
        return t < n_tiles ? t : n_tiles;
    }
};

// Tokens of one launch: bounds the partial statistics (12 bytes per token and leaf) to 192 MiB.
constexpr int64_t kMaxSlice = 65536;
constexpr int kUnitsPerRound = 256;             // one workgroup per CU
constexpr int kMaxRounds = 64;                  // units a workgroup may take

// The tiles of one workgroup: the tiles of its first unit, then of its second, ...  The tile loop runs
// over the flattened (unit, vocabulary tile, k-step) sequence, so the first loads of the next tile are in
// flight during the statistics of the current one, also across units.
//
// Workgroups are dealt round-robin to the 8 XCDs; the 32 of an XCD take consecutive units in each round.
// Units are numbered so that these 32 are 4 token tiles x 8 groups: those that stream the same hidden
// block and those that stream the same weight tiles run side by side and share them in the XCD's L2; and
// so that the 8 XCDs hold 32 token tiles x the SAME 8 groups, so that a weight tile comes from HBM once
// for all of them (numbering all groups of 4 token tiles first: 2 % slower at 8 and more groups).
template <bool kEntropy>
struct UnitTiles : mrl_tile::WholeK {
    // With the entropy's sums the epilogue below needs more registers than there are and puts some aside: their
    // return is waited for before the loop, where the wait would be for the requests in flight (they have landed
    // by then).
    static constexpr bool kSettle = kEntropy;
    int n_tiles;
    // lane r of a wavefront holds the workgroup's unit r: the flattened number of its first tile (beyond every
    // tile where there is no such unit), its first vocabulary tile less that number, its token tile
    int start, tm0, tn0;
    __device__ __forceinline__ void coords(int j, int& tm, int& tn) const {
        const int r = __popcll(__ballot(start <= j)) - 1;
        tm = __builtin_amdgcn_readlane(tm0, r) + j;
        tn = __builtin_amdgcn_readlane(tn0, r);
    }
};

// What bounds it: the matrix cores (1.33 us per k-step of a tile), and between tiles the statistics, 4 us in
// which they idle: per entry a read out of the accumulators, half a max3, an FMA, an exponential and an addition;
// the entropy's sum is one more FMA and taken only where it is asked for.  The lanes' parts of a leaf meet in LDS
// (eight of them merged by a thread per token) and not in two rounds of shuffles, and the statistics' stores are
// not waited for.  us, before -> now: 23 255 x 8 600 x 640 283 -> 249 (256 with entropy), 9 477 x 18 840 x 640
// 246 -> 218 (227), 16 384 x 65 536 x 1 024 1 667 -> 1 594 (1 617), 12 356 x 152 064 x 3 584 9 307 -> 9 284.
//
// partial: [leaf][m, s, u][token of the slice]; without kEntropy u is left out
template <bool kEntropy>
__global__ __launch_bounds__(mrl_tile::kThreads, 1) void lmhead_fwd_kernel(
    const uint16_t* __restrict__ hidden, const uint16_t* __restrict__ weight, int n_tokens, int vocab, int hdim,
    int n_groups, float k_scale, float* __restrict__ partial) {
    using namespace mrl_tile;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    static_assert(kMaxRounds <= 64, "a lane for each unit");

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wv = wave >> 1, wt = wave & 1;
    const VocabLeaves leaves(vocab);
    UnitTiles<kEntropy> seq = {{}, 0, 0x7fffffff, 0, 0};
    {
        const int n_ttiles = (n_tokens + BN - 1) / BN;
        int r = 0;
        for (int u = (int)(blockIdx.x & 7) * 32 + (int)(blockIdx.x >> 3); u < n_ttiles * n_groups; u += kUnitsPerRound, ++r) {
            // 32 token tiles by all groups > 8 groups > 4 token tiles > group > token tile
            const int sp = u / (32 * n_groups), in_sp = u - sp * 32 * n_groups, tt_sp = min(32, n_ttiles - sp * 32);
            const int block = in_sp / (tt_sp * 8), in_block = in_sp - block * tt_sp * 8, gw = min(8, n_groups - block * 8);
            const int panel = in_block / (4 * gw), in_panel = in_block - panel * 4 * gw;
            const int width = min(4, tt_sp - panel * 4), group = block * 8 + in_panel / width;
            const int first = leaves.begin_tile((int)((int64_t)group * leaves.n / n_groups));
            if (lane == r) {
                seq.start = seq.n_tiles;
                seq.tm0 = first - seq.n_tiles;
                seq.tn0 = sp * 32 + panel * 4 + in_panel % width;
            }
            seq.n_tiles += leaves.begin_tile((int)((int64_t)(group + 1) * leaves.n / n_groups)) - first;
        }
    }
    const int tiles_per_leaf = leaves.tiles_per_leaf, n_vtiles = leaves.n_tiles;

    // a lane holds one token of each of its wavefront's 8 token blocks
    Stats st[kBlocks];
#pragma unroll
    for (int tb = 0; tb < kBlocks; ++tb) st[tb] = {kMaxInit, 0.f, 0.f};

    // threadIdx.x, computed where it is needed: kept from one tile to the next, it and what follows from it take
    // registers that the tile loop needs
    auto my_thread = [&]() {
        int t = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(t));
        return t + wave * 64;
    };

    // A leaf is finished: every lane leaves its 8 tokens' statistics in LDS, [part][m, s, u][token] with a part
    // for each quarter of each of the two vocabulary wavefronts, and thread t merges the parts of token t in
    // their order and writes them.
    auto finish_leaf = [&](int leaf, int tn, unsigned char* spare) {
        constexpr int kParts = 8, kValues = kEntropy ? 3 : 2;
        constexpr int kPitch = kValues * kThreads + 16;            // the quarters of a wavefront on different banks
        static_assert(kParts * kPitch * sizeof(float) <= kSpareBytes, "the statistics of a leaf");
        float* const comb = reinterpret_cast<float*>(spare);
        const int tid = my_thread();
        float* const mine = comb + (wv * 4 + ((tid & 63) >> 4)) * kPitch + wt * 128 + (tid & 15);
#pragma unroll
        for (int tb = 0; tb < kBlocks; ++tb) {
            mine[tb * 16] = st[tb].m;
            mine[tb * 16 + kThreads] = st[tb].s;
            if (kEntropy) mine[tb * 16 + 2 * kThreads] = st[tb].u;
            st[tb] = {kMaxInit, 0.f, 0.f};
        }
        // LDS accesses only: a full fence would wait for the requests of the next stages as well
        auto lds_barrier = [&]() {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        };
        lds_barrier();
        const float* const part = comb + tid;
        Stats r = {part[0], 0.f, 0.f};
#pragma unroll
        for (int p = 1; p < kParts; ++p) r.m = fmaxf(r.m, part[p * kPitch]);
#pragma unroll
        for (int p = 0; p < kParts; ++p) {
            const float f = fast_exp2((part[p * kPitch] - r.m) * k_scale);
            r.s = __builtin_fmaf(part[p * kPitch + kThreads], f, r.s);
            if (kEntropy) r.u = __builtin_fmaf(part[p * kPitch + 2 * kThreads], f, r.u);
        }
        lds_barrier();                          // what lies here next is requested by any of the wavefronts
        const int t = tn * BN + tid;
        if (t < n_tokens) {
            float* p = partial + (int64_t)leaf * 3 * n_tokens + t;
            p[0] = r.m;
            p[n_tokens] = r.s;
            if (kEntropy) p[2 * (int64_t)n_tokens] = r.u;
        }
    };

    // online softmax statistics of a tile: per token block a lane holds 8 x 4 vocabulary rows, of which a ragged
    // tile has those 16 vb + r below `valid`
    auto tokens_stats = [&](Accumulators& acc, int valid, bool ragged) {
#pragma unroll
        for (int tb = 0; tb < kBlocks; ++tb) {
            // one block of tokens at a time: without this the compiler copies many blocks out of the
            // accumulator half of the register file at once and parks them in scratch memory
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int vb = 0; vb < kBlocks; ++vb) asm volatile("" : "+a"(acc[vb][tb]));
            float z[4 * kBlocks];
#pragma unroll
            for (int i = 0; i < 4 * kBlocks; ++i) z[i] = acc[i / 4][tb][i % 4];
            if (ragged) {
#pragma unroll
                for (int i = 0; i < 4 * kBlocks; ++i)
                    if (16 * (i / 4) + i % 4 >= valid) z[i] = kMaxInit;
            }
            float vmax = st[tb].m;
#pragma unroll
            for (int i = 0; i < 4 * kBlocks; ++i) vmax = fmaxf(vmax, z[i]);
            grow_max<kEntropy>(st[tb], vmax, k_scale);
            // A lane that has seen no valid vocabulary row yet (the first tile of its leaf is ragged and
            // ends above its rows) still holds the start value as its maximum: z * k - m * k of the masked
            // entries would then be the rounding residual of two numbers of magnitude 1e30 instead of
            // zero.  With an infinite m * k their exponentials are exactly 0.
            const float mk = st[tb].m > kMaxInit ? st[tb].m * k_scale : __builtin_inff();
#pragma unroll
            for (int i = 0; i < 4 * kBlocks; ++i) add_one<kEntropy>(st[tb], z[i], k_scale, mk);
        }
    };
    auto tile_stats = [&](Accumulators& acc, int, int tm, int tn, unsigned char* spare) {
        const int tid = my_thread();
        tokens_stats(acc, vocab - (tm * BM + wv * 128 + 4 * ((tid & 63) >> 4)), tm * BM + BM > vocab);
        const int leaf = tm / tiles_per_leaf;                      // uniform over the workgroup
        if (tm + 1 == n_vtiles || tm + 1 == (leaf + 1) * tiles_per_leaf) finish_leaf(leaf, tn, spare);
    };
    mfma_tile_loop<false, false>(smem, weight, hdim, vocab, hidden, hdim, n_tokens, hdim, seq, tile_stats);
}

// A workgroup finishes 16 tokens.  One wavefront per token computes the label logit as an fp32 dot product of the
// token's hidden row with the label's weight row; 16 threads per token, of the first four wavefronts, merge the leaves
// (thread q takes leaves q, q + 16, ...; the loads of 16 neighbouring tokens are 64 contiguous bytes), then the 16
// partial results are merged in order.  Few tokens are bound by the loads that follow each other, many by the rows'
// bytes: a wavefront to each token up to kFewTokens, 4 tokens to one behind.  us, 4 wavefronts and 512 entries at a time
// -> now, 32 000 logits unless given: 224 tokens x 3 072 14.6 -> 6.3, 589 x 4 224 20.7 -> 8.2, 4 000 x 1 024 10.0 -> 7.2,
// 7 100 x 3 776 26.4 -> 21.6, 12 000 x 2 048 20.0 -> 19.8.  Beyond that the four loads at a time gain nothing and cost up
// to 6 % of a few microseconds in passes of milliseconds: 20 959 x 10 736 x 768 14.8 -> 14.9, 9 000 x 512 10.5 -> 11.2,
// 17 122 x 152 064 x 3 584 49.6 -> 52.1; a wavefront to each there 18.0, 11.9 and 51.6.
constexpr int kFinishTokens = 16;
constexpr int64_t kFewTokens = 4096;
template <typename LabelT, bool kEntropy, int kFinishWaves>
__global__ __launch_bounds__(64 * kFinishWaves) void lmhead_finish_kernel(
    const uint16_t* __restrict__ hidden, const uint16_t* __restrict__ weight, const LabelT* __restrict__ labels,
    const float* __restrict__ partial, int n_tokens, int vocab, int hdim, int n_leaves, float inv_t,
    const int32_t* __restrict__ cells, float* __restrict__ logp, float* __restrict__ entropy,
    float* __restrict__ lse_out) {
    __shared__ Stats part[16][kFinishTokens];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t0 = (int)blockIdx.x * kFinishTokens;
    const float k = inv_t * kLog2e;
    if (wave < 4) {
        const int mine = threadIdx.x & 15, q = threadIdx.x >> 4;
        const int t = min(t0 + mine, n_tokens - 1);
        Stats r = {kMaxInit, 0.f, 0.f};
#pragma unroll 4
        for (int leaf = q; leaf < n_leaves; leaf += 16) {
            const float* p = partial + (int64_t)leaf * 3 * n_tokens + t;
            const Stats o = {p[0], p[n_tokens], kEntropy ? p[2 * (int64_t)n_tokens] : 0.f};
            r = merge<kEntropy>(r, o, k);
        }
        part[q][mine] = r;
    }
    auto label_logit = [&](int t, float& dot, bool& y_ok) {
        dot = 0.f;
        y_ok = false;
        if (t >= n_tokens) return;
        const int64_t y = (int64_t)labels[t];
        y_ok = (y >= 0) && (y < (int64_t)vocab);
        if (!y_ok) return;
        const uint16_t* hrow = hidden + (int64_t)t * hdim;
        const uint16_t* wrow = weight + y * hdim;
        constexpr int kDeep = 4;                    // 2 x 4 loads on their way at a time
        for (int at = 0; at < hdim; at += kDeep * 512) {            // 512 entries a wavefront and load
            const int j = at + lane * 8;
            u32x4 hv[kDeep], wv[kDeep];
#pragma unroll
            for (int d = 0; d < kDeep; ++d) {
                if (at + d * 512 >= hdim) continue;                 // uniform
                const bool in = j + d * 512 < hdim;
                hv[d] = in ? *reinterpret_cast<const u32x4*>(hrow + j + d * 512) : mrl::make_u32x4(0u, 0u, 0u, 0u);
                wv[d] = in ? *reinterpret_cast<const u32x4*>(wrow + j + d * 512) : mrl::make_u32x4(0u, 0u, 0u, 0u);
            }
#pragma unroll
            for (int d = 0; d < kDeep; ++d) {
                if (at + d * 512 >= hdim) continue;
                float a[8], b[8];
                Elem<MRL_BF16>::unpack(hv[d], a);
                Elem<MRL_BF16>::unpack(wv[d], b);
#pragma unroll
                for (int e = 0; e < 8; ++e) dot = __builtin_fmaf(a[e], b[e], dot);
            }
        }
    };
    float dot;
    bool y_ok;
    constexpr bool kOne = kFinishWaves == kFinishTokens;        // the product need not wait for the leaves
    if (kOne) label_logit(t0 + wave, dot, y_ok);
    __syncthreads();
    for (int i = wave; i < kFinishTokens; i += kFinishWaves) {
        const int t = t0 + i;
        if (t >= n_tokens) return;
        if (!kOne) label_logit(t, dot, y_ok);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) dot += __shfl_xor(dot, off, 64);
        Stats r = part[lane & 15][i];
#pragma unroll
        for (int off = 1; off <= 8; off <<= 1) {
            const Stats o = {__shfl_xor(r.m, off, 64), __shfl_xor(r.s, off, 64), kEntropy ? __shfl_xor(r.u, off, 64) : 0.f};
            r = merge<kEntropy>(r, o, k);
        }
        if (lane == 0) {
            const float lse = (r.m * k + fast_log2(r.s)) * kLn2;
            const int64_t at = cells ? (int64_t)cells[t] : (int64_t)t;
            logp[at] = (y_ok ? dot * inv_t : r.m * inv_t) - lse;
            if (kEntropy) entropy[at] = lse - (r.u / r.s) * inv_t;
            if (lse_out) lse_out[at] = lse;
        }
    }
}

// The number of groups that the leaves are dealt into.  A launch takes ceil(token tiles x groups / 256)
// rounds of the chip, each as long as its largest group plus a little (a unit's first tiles come from
// beyond the L2); the cheapest count wins, the smallest among equals.  One and two groups stream more
// different hidden blocks through an L2 than it holds (65 536 tokens: 71.1 ms with 1, 49.7 with 2, 48.9
// with 3, 49.2 with 8).  What this replaces, 8 groups for every size and a launch of as many workgroups
// as that makes, gave 17 122 tokens (67 token tiles) 3 rounds for 2.1 rounds of work, and 1 380 tokens 48
// of the 256 CUs.  Measured with it / now:
//     tokens  vocabulary  hidden     before       now        tokens  vocabulary  hidden    before       now
//        162      95 920    2944   3 184 us    187 us        17 122    152 064    3584  19.77 ms  13.24 ms
//        704      67 512    1344     937 us    153 us        19 202    148 784    1088   6.91 ms   5.14 ms
//      1 380      27 600    2880     803 us    223 us        32 768    152 064    3584  25.69 ms  24.66 ms
int pick_groups(int64_t n_tokens, const VocabLeaves& leaves) {
    const int64_t n_ttiles = (n_tokens + mrl_tile::BN - 1) / mrl_tile::BN;
    int best = 1;
    int64_t best_cost = INT64_MAX;
    for (int g = 1; g <= leaves.n; ++g) {
        const int64_t rounds = (n_ttiles * g + kUnitsPerRound - 1) / kUnitsPerRound;
        if (rounds > kMaxRounds) break;
        int64_t tiles = (int64_t)((leaves.n + g - 1) / g) * leaves.tiles_per_leaf;
        if (tiles > leaves.n_tiles) tiles = leaves.n_tiles;
        const int64_t cost = rounds * (10 * tiles + 3) * (g == 1 ? 140 : (g == 2 ? 102 : 100));
        if (cost < best_cost) {
            best_cost = cost;
            best = g;
        }
    }
    return best;
}

}  // namespace

extern "C" int64_t mrl_lmhead_workspace_bytes(int64_t n_tokens, int64_t vocab) {
    if (n_tokens < 0 || vocab <= 0) return 0;
    return (int64_t)VocabLeaves(vocab).n * (n_tokens < kMaxSlice ? n_tokens : kMaxSlice) * 3 * (int64_t)sizeof(float);
}

// Checks and launches shared by the forward entry points; token t's results go to entry t of the outputs, or with
// `cells` to entry cells[t].  `partial` holds the statistics of `slice`
// tokens (whole tiles); more are taken in equal slices, one after the other on the stream (32 768 tokens x
// 152 064 x 3 584 where 28 160 fit: 26.2 ms as 28 160 + 4 608, 25.2 ms as 2 x 16 384).
static int lmhead_forward(const char* fn, const void* hidden, const void* weight, int64_t n_tokens, int64_t vocab,
                          int64_t hidden_dim, const void* labels, int labels_dtype, float inv_temperature,
                          const int32_t* cells, float* logp, float* entropy, float* lse, float* partial, int64_t slice,
                          hipStream_t s) {
    // 256-token tiles, all of a CU's LDS for the tile loop.  Function
    // attributes belong to a device, so the reservation is made with every launch, on whichever
    // device is current.
    constexpr int kLdsBytes = mrl_tile::kLdsBytes;
    const auto fwd = entropy ? lmhead_fwd_kernel<true> : lmhead_fwd_kernel<false>;
    const bool wide_labels = labels_dtype != MRL_I32;
    const hipError_t attr =
        hipFuncSetAttribute((const void*)fwd, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
    MRL_REQUIRE(attr == hipSuccess, MRL_ERR_LAUNCH, "%s: cannot reserve %d bytes of LDS: %s", fn, kLdsBytes,
                hipGetErrorString(attr));
    MRL_REQUIRE(256 * hidden_dim * 2 < (1LL << 31) && n_tokens <= 0x7fffffffLL, MRL_ERR_UNSUPPORTED,
                "%s: size out of range", fn);
    const VocabLeaves leaves(vocab);
    const int64_t n_slices = (n_tokens + slice - 1) / slice, n_ttiles = (n_tokens + mrl_tile::BN - 1) / mrl_tile::BN;
    slice = (n_ttiles + n_slices - 1) / n_slices * mrl_tile::BN;
    for (int64_t lo = 0; lo < n_tokens; lo += slice) {
        const int n = (int)(n_tokens - lo < slice ? n_tokens - lo : slice);
        const uint16_t* h = (const uint16_t*)hidden + lo * hidden_dim;
        hipLaunchKernelGGL(fwd, dim3(kUnitsPerRound), dim3(mrl_tile::kThreads), kLdsBytes, s, h,
                           (const uint16_t*)weight, n, (int)vocab, (int)hidden_dim, pick_groups(n, leaves),
                           inv_temperature * kLog2e, partial);
        int rc = mrl::check_launch(fn);
        if (rc != MRL_OK) return rc;
        const dim3 fgrid((unsigned)((n + kFinishTokens - 1) / kFinishTokens)), fblock(n <= kFewTokens ? 1024 : 256);
        const int64_t out_lo = cells ? 0 : lo;
        float* ent = entropy ? entropy + out_lo : nullptr;
        float* lse_out = lse ? lse + out_lo : nullptr;
        const int32_t* to = cells ? cells + lo : nullptr;
        auto finish = [&](auto kernel, auto* lab) {
            hipLaunchKernelGGL(kernel, fgrid, fblock, 0, s, h, (const uint16_t*)weight, lab + lo, (const float*)partial, n,
                               (int)vocab, (int)hidden_dim, leaves.n, inv_temperature, to, logp + out_lo, ent, lse_out);
        };
        auto finish_by_count = [&](auto* lab, auto with_entropy) {
            using LabelT = std::remove_cv_t<std::remove_pointer_t<decltype(lab)>>;
            if (n <= kFewTokens) finish(lmhead_finish_kernel<LabelT, decltype(with_entropy)::value, 16>, lab);
            else finish(lmhead_finish_kernel<LabelT, decltype(with_entropy)::value, 4>, lab);
        };
        auto finish_by_label = [&](auto with_entropy) {
            if (wide_labels) finish_by_count((const int64_t*)labels, with_entropy);
            else finish_by_count((const int32_t*)labels, with_entropy);
        };
        if (entropy) finish_by_label(std::true_type());
        else finish_by_label(std::false_type());
        rc = mrl::check_launch(fn);
        if (rc != MRL_OK) return rc;
    }
    return MRL_OK;
}

#define MRL_LMHEAD_CHECK_ARGS(fn)                                                                                      \
    MRL_REQUIRE(n_tokens >= 0 && vocab > 0 && hidden_dim > 0, MRL_ERR_INVALID_ARG,                                     \
                "%s: n_tokens=%lld vocab=%lld hidden_dim=%lld", fn, (long long)n_tokens, (long long)vocab,             \
                (long long)hidden_dim);                                                                                \
    MRL_REQUIRE(hidden_dim % mrl_tile::BK == 0, MRL_ERR_UNSUPPORTED, "%s: hidden_dim=%lld must be a multiple of %d", fn, \
                (long long)hidden_dim, mrl_tile::BK);                                                                          \
    MRL_REQUIRE(vocab <= (1LL << 30) && hidden_dim <= (1LL << 20), MRL_ERR_UNSUPPORTED, "%s: size out of range", fn);  \
    MRL_REQUIRE(mrl::int_dtype_bytes(labels_dtype) != 0, MRL_ERR_UNSUPPORTED, "%s: labels dtype %d (want I32 or I64)", \
                fn, labels_dtype);                                                                                     \
    MRL_REQUIRE(inv_temperature > 0.f && inv_temperature < 1.0e6f, MRL_ERR_INVALID_ARG,                                \
                "%s: inv_temperature=%g must be in (0, 1e6)", fn, (double)inv_temperature)

static int forward_in_workspace(const char* fn, const void* hidden, const void* weight, int64_t n_tokens, int64_t vocab,
                                int64_t hidden_dim, const void* labels, int labels_dtype, float inv_temperature,
                                const int32_t* cells, float* logp, float* entropy, float* lse, void* workspace,
                                int64_t workspace_bytes, void* stream) {
    MRL_LMHEAD_CHECK_ARGS(fn);
    if (n_tokens == 0) return MRL_OK;
    MRL_REQUIRE(hidden && weight && labels && logp && workspace, MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    MRL_REQUIRE(mrl::aligned(hidden, 16) && mrl::aligned(weight, 16) && mrl::aligned(workspace, 16), MRL_ERR_MISALIGNED,
                "%s: hidden, weight and workspace must be 16-byte aligned", fn);
    MRL_REQUIRE(workspace_bytes >= mrl_lmhead_workspace_bytes(n_tokens, vocab), MRL_ERR_INVALID_ARG,
                "%s: workspace of %lld bytes, need %lld", fn, (long long)workspace_bytes,
                (long long)mrl_lmhead_workspace_bytes(n_tokens, vocab));
    return lmhead_forward(fn, hidden, weight, n_tokens, vocab, hidden_dim, labels, labels_dtype, inv_temperature, cells,
                          logp, entropy, lse, (float*)workspace, kMaxSlice, mrl::as_stream(stream));
}

extern "C" int mrl_lmhead_logprob_fwd(const void* hidden, const void* weight, int64_t n_tokens, int64_t vocab,
                                      int64_t hidden_dim, const void* labels, int labels_dtype,
                                      float inv_temperature, float* logp, float* entropy, float* lse,
                                      void* workspace, int64_t workspace_bytes, void* stream) {
    return forward_in_workspace("mrl_lmhead_logprob_fwd", hidden, weight, n_tokens, vocab, hidden_dim, labels, labels_dtype,
                                inv_temperature, nullptr, logp, entropy, lse, workspace, workspace_bytes, stream);
}

extern "C" int mrl_lmhead_logprob_fwd_cells(const void* hidden, const void* weight, int64_t n_tokens, int64_t vocab,
                                            int64_t hidden_dim, const void* labels, int labels_dtype,
                                            float inv_temperature, const int32_t* cells, float* logp, float* entropy,
                                            void* workspace, int64_t workspace_bytes, void* stream) {
    const char* fn = "mrl_lmhead_logprob_fwd_cells";
    MRL_REQUIRE(cells != nullptr || n_tokens == 0, MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    return forward_in_workspace(fn, hidden, weight, n_tokens, vocab, hidden_dim, labels, labels_dtype, inv_temperature, cells,
                                logp, entropy, nullptr, workspace, workspace_bytes, stream);
}

// Address of `scratch` on the current device, looked up once per device (each GPU holds its own
// copy of the array at its own address).  NULL and an error message if the lookup fails.
static float* static_scratch(const char* fn) {
    constexpr int kMaxDevices = 64;
    static std::atomic<float*> known[kMaxDevices];
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        mrl::fail(MRL_ERR_LAUNCH, "%s: no current device (hipGetDevice gave %d)", fn, dev);
        return nullptr;
    }
    float* p = known[dev].load(std::memory_order_acquire);
    if (p) return p;
    void* addr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || addr == nullptr) {
        mrl::fail(MRL_ERR_LAUNCH, "%s: hipGetSymbolAddress(scratch) on device %d: %s", fn, dev, hipGetErrorString(e));
        return nullptr;
    }
    known[dev].store((float*)addr, std::memory_order_release);
    return (float*)addr;
}

extern "C" int64_t mrl_lmhead_static_max_tokens(void) { return MRL_LMHEAD_STATIC_MAX_TOKENS; }

extern "C" int mrl_lmhead_logprob_fwd_static(const void* hidden, const void* weight, int64_t n_tokens, int64_t vocab,
                                             int64_t hidden_dim, const void* labels, int labels_dtype,
                                             float inv_temperature, float* logp, float* entropy, float* lse,
                                             void* stream) {
    const char* fn = "mrl_lmhead_logprob_fwd_static";
    MRL_LMHEAD_CHECK_ARGS(fn);
    MRL_REQUIRE(n_tokens <= MRL_LMHEAD_STATIC_MAX_TOKENS, MRL_ERR_UNSUPPORTED,
                "%s: n_tokens=%lld exceeds the %d tokens the library's own scratch memory holds; call it on slices of "
                "at most that many tokens, or use mrl_lmhead_logprob_fwd with a workspace",
                fn, (long long)n_tokens, MRL_LMHEAD_STATIC_MAX_TOKENS);
    if (n_tokens == 0) return MRL_OK;
    MRL_REQUIRE(hidden && weight && labels && logp, MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    MRL_REQUIRE(mrl::aligned(hidden, 16) && mrl::aligned(weight, 16), MRL_ERR_MISALIGNED,
                "%s: hidden and weight must be 16-byte aligned", fn);
    float* partial = static_scratch(fn);
    if (!partial) return MRL_ERR_LAUNCH;
    // whole token tiles that the scratch memory holds the statistics of (28 160 tokens at 152 064 entries)
    const int64_t slice = MRL_LMHEAD_STATIC_BYTES / (VocabLeaves(vocab).n * 12LL) / 256 * 256;
    return lmhead_forward(fn, hidden, weight, n_tokens, vocab, hidden_dim, labels, labels_dtype, inv_temperature, nullptr,
                          logp, entropy, lse, partial, slice, mrl::as_stream(stream));
}
