// bf16 matrix products of the lm_head training step for gfx950 on the shared tile loop (lmhead_tile.h).
//
// One kernel covers the three products of the step, because each of them can be put in the form
//
//     out[n][m] (+)= sum_k A[m][k] * B[n][k]
//
// (the MFMA's M is the fast dimension of the output: in the 16x16 result layout a lane owns ONE
// column n and 4 consecutive rows m, i.e. 8 contiguous bytes of bf16 or 16 of fp32):
//
//     logits[t][v]  = sum_h W[v][h]      * hidden[t][h]      A = W,           B = hidden chunk
//     dHidden[t][h] = sum_v W[v][h]      * dlogits[t][v]     A = W (k-major), B = dlogits chunk
//     dW[v][h]     += sum_t hidden[t][h] * dlogits[t][v]     A = hidden,      B = dlogits chunk, both k-major
//
// so the backward reads hidden, W and dlogits as they lie: no transposed copies.
//
// Work distribution: one persistent workgroup per CU walks output tiles of 256 x 256.  Tiles are
// numbered so that 32 consecutive numbers are 8 tiles along m by 4 along n, and the 32 workgroups
// that share an XCD (and its L2) take 32 consecutive numbers at a time: the 4 that stream the same A
// tile and the 8 that stream the same B tile run side by side (see tile_coords for the order of the
// groups of 32).
//
// dHidden has few tiles and a long K (the vocabulary): 162 tokens x 2 944 is 12 tiles on 256 CUs, 4 000 x 5 120
// is 1.25 rounds of the chip; dWeight of a small model over many tokens likewise.  Tiles behind the last whole round
// may therefore be cut along K into slices
// (plan_split); a slice leaves its fp32 sums in the caller's workspace and merge_slices_kernel adds them in
// the order of the slices.  Units are numbered slice by slice, so the workgroups of an XCD still share operand
// tiles.  Both backward products, uncut and cut: 300 x 32 000 x 1 024 557 -> 99 us, 1 380 x 152 064 x 3 584
// 4 466 -> 2 404, 4 000 x 129 280 x 5 120 10 030 -> 7 650.
#include <type_traits>

#include "lmhead_tile.h"
#include "mrl_internal.h"
#include "vocab_common.h"

namespace {

using namespace mrl_vocab;
using namespace mrl_tile;

constexpr int kTilesAlongN = 4;                  // tiles along n in a group of consecutive tile numbers

struct TileGrid {
    int tiles_m, tiles_n, panel_m;
    int64_t total;
};

// Tile number -> (tile along m, tile along n).  Tiles are numbered panel by panel, a panel being
// panel_m tiles along m by all tiles along n; inside a panel consecutive numbers walk m first inside
// a group of 4 tiles along n (4 consecutive numbers are one tile of A with 4 tiles of B), and the groups
// walk along n.  With panel_m = 8 the 32 workgroups of an XCD hold 8 (m) x 4 (n) tiles and the 8 XCDs
// 8 x 32; with 32 an XCD still holds 8 x 4 and the chip 32 x 8, which fetches less from beyond the L2
// (B is passed over a quarter as often).
// A workgroup keeps its tile of A from one of its tiles to the next.
__device__ __forceinline__ void tile_coords(const TileGrid& g, int t, int& tm, int& tn) {
    const int per_panel = g.panel_m * g.tiles_n;
    const int p = t / per_panel;
    const int idx = t - p * per_panel;
    const int pm = min(g.panel_m, g.tiles_m - p * g.panel_m);   // rows of tiles in this panel
    const int ng = idx / (pm * kTilesAlongN);
    const int rem = idx - ng * (pm * kTilesAlongN);
    const int width = min(kTilesAlongN, g.tiles_n - ng * kTilesAlongN);
    tm = p * g.panel_m + rem / width;
    tn = ng * kTilesAlongN + rem % width;
}

__host__ __device__ inline TileGrid make_grid(int64_t M, int64_t N) {
    TileGrid g;
    g.tiles_m = (int)((M + BM - 1) / BM);
    g.tiles_n = (int)((N + BN - 1) / BN);
    g.total = (int64_t)g.tiles_m * g.tiles_n;
    // panels of up to 8 rows of tiles (8 x 4 blocks per XCD), tall products up to 32; all panels the same
    // height (14 rows of tiles as 7 + 7 measured 1.7 % faster than as 8 + 6)
    const int panel_cap = g.tiles_m >= 64 ? 32 : 8;
    const int n_panels = (g.tiles_m + panel_cap - 1) / panel_cap;
    g.panel_m = (g.tiles_m + n_panels - 1) / n_panels;
    return g;
}

// Tiles from number `whole` on are cut into n_slices along K (n_slices 1: none is).
struct SplitPlan {
    int64_t whole;
    int rest, n_slices;
};

constexpr int64_t kTileElems = (int64_t)BM * BN;
constexpr int64_t kMaxSlices = 1024;                // of all tiles together: 256 MiB of fp32 sums

// The number of slices with the least expected time, in k-steps (about 1.5 microseconds each): the rounds that
// the units take, and per unit of a round about 10 for turning out the sums and 0.1 for each slice's trip
// through memory to the merge.  dHidden and dWeight together, uncut and in the slices it chooses, ms: 174 of 256
// tiles (12 356 x 152 064 x 3 584) 20.55 and in 4 19.73 (in 3 20.76, in 5 19.98); 104 (9 000 x 152 064 x 2 560)
// 12.33 and in 7 10.27; 144 (2 300 x 32 000 x 4 096) 1.118 and in 3 0.978.
// worth: the share of the whole product that a cut has to save.
inline SplitPlan plan_split(int64_t total, int grid, int64_t n_ksteps, double worth) {
    SplitPlan p = {total / grid * grid, (int)(total % grid), 1};
    if (p.rest == 0) return p;
    double best = (double)n_ksteps * (1.0 - worth * (double)(total / grid + 1));
    for (int64_t s = 2; s * p.rest <= kMaxSlices && s * 4 <= n_ksteps; ++s) {
        const int64_t rounds = (s * p.rest + grid - 1) / grid;
        const double cost = (double)rounds * ((double)((n_ksteps + s - 1) / s) + 10.0) + 0.1 * (double)(s * p.rest) + 10.0;
        if (cost < best) {
            best = cost;
            p.n_slices = (int)s;
        }
    }
    if (p.n_slices == 1) p.whole = total, p.rest = 0;
    return p;
}

// The tiles of one workgroup: number first + j * stride.
struct StridedTiles : WholeK {
    TileGrid grid;
    int first, stride;
    int n_tiles;
    __device__ __forceinline__ void coords(int j, int& tm, int& tn) const { tile_coords(grid, first + j * stride, tm, tn); }
};

// The slices of one workgroup: unit u = first + j * stride is slice u / rest of tile whole + u % rest.
struct SlicedTiles {
    static constexpr bool kSettle = false;
    TileGrid grid;
    int first, stride;
    int n_tiles;
    SplitPlan plan;
    __device__ __forceinline__ void coords(int j, int& tm, int& tn) const {
        tile_coords(grid, (int)plan.whole + (first + j * stride) % plan.rest, tm, tn);
    }
    __device__ __forceinline__ void k_range(int j, int n_ksteps, int& begin, int& end) const {
        const int64_t s = (first + j * stride) / plan.rest;
        begin = (int)(s * n_ksteps / plan.n_slices);
        end = (int)((s + 1) * n_ksteps / plan.n_slices);
    }
};

// What becomes of a finished tile: stored as bf16, stored as fp32, added to the fp32 there, or added to the
// fp32 at `acc` and the sum stored as bf16.
enum Out { kBf16, kF32, kF32Add, kSumToBf16 };

// kATrans / kBTrans: the operand is k-major, [K, M] or [K, N]; else [M, K] or [N, K].  sums: fp32 [N, M] with
// the leading dimension of out (kSumToBf16), or with kSliced (kOut kF32) what the slices' tiles go to; the
// plan says which tiles are whole and how the rest are cut, and a launch does the one or the other (both in
// one kernel need two epilogues and spill).
template <int kOut, bool kATrans, bool kBTrans, bool kSliced>
__global__ __launch_bounds__(kThreads, 1) void gemm_kernel(const uint16_t* __restrict__ A, int64_t lda, int M,
                                                           const uint16_t* __restrict__ B, int64_t ldb, int N, int K,
                                                           void* __restrict__ out, int64_t ldo, float* __restrict__ sums,
                                                           SplitPlan plan) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wv = wave / kWavesN, wt = wave % kWavesN;

    static_assert(!kSliced || kOut == kF32, "a slice leaves fp32 sums");
    std::conditional_t<kSliced, SlicedTiles, StridedTiles> seq;
    seq.grid = make_grid(M, N);
    const int64_t n_units = kSliced ? (int64_t)plan.rest * plan.n_slices : plan.whole;
    if constexpr (kSliced) seq.plan = plan;
    // workgroups are dealt round-robin to the 8 XCDs: the gridDim / 8 workgroups of an XCD take
    // consecutive tile numbers
    const int per_xcd = gridDim.x >> 3;
    seq.first = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    seq.stride = (int)gridDim.x;
    seq.n_tiles = seq.first < n_units ? ((int)n_units - 1 - seq.first) / seq.stride + 1 : 0;

    // The finished tile.  A lane holds column n = lane & 15 of each 16 x 16 block and rows
    // 4 (lane >> 4) .. + 3 of it: stored like that, a store instruction would touch 16 output rows with
    // 8 or 16 bytes each.  Each wavefront therefore turns its blocks through a private 8 KiB of LDS:
    // [64 n][128 bytes of m] at a time (4 blocks along n by 4 along m for bf16, by 2 for fp32), 16-byte
    // chunks XOR-swizzled by the row pair, written in the MFMA layout and read back as 8 lanes x 16 bytes
    // per output row, so that every store covers whole 128-byte lines.
    auto store_tile = [&](mrl_tile::Accumulators& acc, int j, int tm, int tn, unsigned char* spare) {
        unsigned char* const turn = spare + wave * (kSpareBytes / kWaves);
        constexpr bool kWideEntries = kOut != kBf16;              // turned as fp32
        // a slice's tile is a matrix of its own
        const int m_tile = kSliced ? 0 : tm * BM, n_tile = kSliced ? 0 : tn * BN;
        const int m_end = kSliced ? M - tm * BM : M, n_end = kSliced ? N - tn * BN : N;
        const int64_t ld = kSliced ? BM : ldo;
        float* const slice = sums + (kSliced ? (int64_t)(seq.first + j * seq.stride) * kTileElems : 0);
        const int row_w = lane & 15, quarter = lane >> 4;        // writer: its n, its run of 4 m inside the block
        const int row_r = lane >> 3, chunk_r = lane & 7;          // reader: n within a group of 8, 16-byte chunk
        constexpr int kMPerPass = kWideEntries ? 2 : 4;            // 32 fp32 or 64 bf16 entries of m are 128 bytes
#pragma unroll
        for (int tb0 = 0; tb0 < kBlocks; tb0 += 4) {
            const int n0 = n_tile + wt * 128 + tb0 * 16;
#pragma unroll
            for (int vb0 = 0; vb0 < kBlocks; vb0 += kMPerPass) {
                const int m0 = m_tile + wv * 128 + vb0 * 16;
#pragma unroll
                for (int tbi = 0; tbi < 4; ++tbi) {
                    const int row = tbi * 16 + row_w;
                    unsigned char* line = turn + row * 128;
                    const int key = (row >> 1) & 7;
#pragma unroll
                    for (int vbi = 0; vbi < kMPerPass; ++vbi) {
                        const floatx4& c = acc[vb0 + vbi][tb0 + tbi];
                        if (kWideEntries) {
                            *reinterpret_cast<float4*>(line + (((vbi * 4 + quarter) ^ key) * 16)) =
                                make_float4(c[0], c[1], c[2], c[3]);
                        } else {
                            uint2 w;
                            w.x = Elem<MRL_BF16>::pack2(c[0], c[1]);
                            w.y = Elem<MRL_BF16>::pack2(c[2], c[3]);
                            *reinterpret_cast<uint2*>(line + (((vbi * 2 + (quarter >> 1)) ^ key) * 16) + (quarter & 1) * 8) = w;
                        }
                    }
                }
                __builtin_amdgcn_s_waitcnt(0xC07F);            // lgkmcnt(0): the slice is written
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int g = 0; g < 8; ++g) {
                    const int row = g * 8 + row_r;
                    const u32x4 v =
                        *reinterpret_cast<const u32x4*>(turn + row * 128 + ((chunk_r ^ ((row >> 1) & 7)) * 16));
                    const int n = n0 + row;
                    const int m = m0 + chunk_r * (kWideEntries ? 4 : 8);
                    if (n < n_end && m < m_end) {              // M % 8 == 0: a chunk is inside or outside
                        const int64_t at = (int64_t)n * ld + m;
                        if constexpr (kOut == kBf16) {
                            *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(out) + at) = v;
                        } else {
                            float* const dst = kSliced ? slice : reinterpret_cast<float*>(out);
                            float4 c = make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z),
                                                   __uint_as_float(v.w));
                            if constexpr (kOut != kF32) {
                                const float4 o = *reinterpret_cast<const float4*>((kOut == kF32Add ? dst : sums) + at);
                                c = make_float4(o.x + c.x, o.y + c.y, o.z + c.z, o.w + c.w);
                            }
                            if constexpr (kOut == kSumToBf16)
                                *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + at) =
                                    make_uint2(Elem<MRL_BF16>::pack2(c.x, c.y), Elem<MRL_BF16>::pack2(c.z, c.w));
                            else
                                *reinterpret_cast<float4*>(dst + at) = c;
                        }
                    }
                }
                __builtin_amdgcn_s_waitcnt(0xC07F);            // the slice has been read: it may be rewritten
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    mfma_tile_loop<kATrans, kBTrans>(smem, A, lda, M, B, ldb, N, K, seq, store_tile);
}

// out[n][m] = sum over the slices, in their order, of the tiles that SlicedTiles cut.  Grid: (tile, 16 rows of
// it); a wavefront per row of 256 entries, 16 bytes per lane and slice: a read of memory, 4 to 5 TB/s.
__global__ __launch_bounds__(256) void merge_slices_kernel(const float* __restrict__ sums, SplitPlan plan, int M, int N,
                                                           uint16_t* __restrict__ out, int64_t ldo) {
    const TileGrid grid = make_grid(M, N);
    int tm, tn;
    tile_coords(grid, plan.whole + blockIdx.x, tm, tn);
    const int m = (threadIdx.x & 63) * 4;
    if (tm * BM + m >= M) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = (int)blockIdx.y * 16 + i * 4 + (int)(threadIdx.x >> 6);
        if (tn * BN + n >= N) return;
        const float* p = sums + (int64_t)blockIdx.x * kTileElems + n * BM + m;
        float4 c = *reinterpret_cast<const float4*>(p);
        for (int s = 1; s < plan.n_slices; ++s) {
            const float4 o = *reinterpret_cast<const float4*>(p + (int64_t)s * plan.rest * kTileElems);
            c = make_float4(c.x + o.x, c.y + o.y, c.z + o.z, c.w + o.w);
        }
        *reinterpret_cast<uint2*>(out + (int64_t)(tn * BN + n) * ldo + tm * BM + m) =
            make_uint2(Elem<MRL_BF16>::pack2(c.x, c.y), Elem<MRL_BF16>::pack2(c.z, c.w));
    }
}

int persistent_grid() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    return n & ~7;          // a whole number of workgroups per XCD
}

}  // namespace

namespace mrl {

struct Product {
    const void* a; int64_t lda, m;
    const void* b; int64_t ldb, n;
    int64_t k;
    void* out; int64_t ldo;
    float* sums;
    hipStream_t stream;
};

template <int kOut, bool kATrans, bool kBTrans, bool kSliced>
static int launch_gemm(const char* fn, const Product& p, const SplitPlan& plan) {
    // k-contiguous operands are read up to the next multiple of 64 in k
    const int64_t k_steps = (p.k + BK - 1) / BK * BK;
    MRL_REQUIRE(p.m > 0 && p.n > 0 && p.k > 0 && p.m % 8 == 0, MRL_ERR_UNSUPPORTED,
                "%s: product of m=%lld n=%lld k=%lld (m must be a multiple of 8)", fn, (long long)p.m, (long long)p.n,
                (long long)p.k);
    MRL_REQUIRE(p.m <= 0x7fffffffLL && p.n <= 0x7fffffffLL && p.k <= 0x7fffffffLL, MRL_ERR_UNSUPPORTED,
                "%s: size out of range", fn);
    MRL_REQUIRE((kATrans || kBTrans) || p.k % BK == 0, MRL_ERR_UNSUPPORTED,
                "%s: k=%lld must be a multiple of %d when no operand is k-major", fn, (long long)p.k, BK);
    MRL_REQUIRE(!kBTrans || p.n % 8 == 0, MRL_ERR_UNSUPPORTED, "%s: n=%lld must be a multiple of 8 for a k-major b", fn,
                (long long)p.n);
    MRL_REQUIRE(p.lda >= (kATrans ? p.m : k_steps) && p.ldb >= (kBTrans ? p.n : k_steps) && p.ldo >= p.m && p.lda % 8 == 0 &&
                    p.ldb % 8 == 0 && p.ldo % 8 == 0,
                MRL_ERR_INVALID_ARG, "%s: leading dimensions lda=%lld ldb=%lld ldo=%lld", fn, (long long)p.lda,
                (long long)p.ldb, (long long)p.ldo);
    // what one buffer descriptor has to span: a tile of 256 rows, or a slot of 32 k-rows
    MRL_REQUIRE(256 * p.lda * 2 < (1LL << 31) && 256 * p.ldb * 2 < (1LL << 31), MRL_ERR_UNSUPPORTED,
                "%s: 256 rows of an operand must stay below 2 GiB", fn);
    MRL_REQUIRE(aligned(p.a, 16) && aligned(p.b, 16) && aligned(p.out, 16) && aligned(p.sums, 16), MRL_ERR_MISALIGNED,
                "%s: operands must be 16-byte aligned", fn);
    const int grid = persistent_grid();
    MRL_REQUIRE(grid >= 8, MRL_ERR_LAUNCH, "%s: cannot query the device", fn);
    // function attributes belong to a device: reserved with every launch, on whichever device is current
    const hipError_t attr = hipFuncSetAttribute((const void*)gemm_kernel<kOut, kATrans, kBTrans, kSliced>,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
    MRL_REQUIRE(attr == hipSuccess, MRL_ERR_LAUNCH, "%s: cannot reserve %d bytes of LDS", fn, kLdsBytes);
    hipLaunchKernelGGL((gemm_kernel<kOut, kATrans, kBTrans, kSliced>), dim3((unsigned)grid), dim3(kThreads), kLdsBytes,
                       p.stream, (const uint16_t*)p.a, p.lda, (int)p.m, (const uint16_t*)p.b, p.ldb, (int)p.n, (int)p.k,
                       p.out, p.ldo, p.sums, plan);
    return check_launch(fn);
}

static int64_t slice_bytes(const SplitPlan& plan) {
    return plan.n_slices > 1 ? plan.rest * plan.n_slices * kTileElems * (int64_t)sizeof(float) : 0;
}

static SplitPlan whole_tiles(const Product& p) { return SplitPlan{make_grid(p.m, p.n).total, 0, 1}; }

static SplitPlan plan_dhidden(int64_t n_tokens, int64_t vocab, int64_t hidden_dim) {
    const int grid = persistent_grid();
    return plan_split(make_grid(hidden_dim, n_tokens).total, grid < 8 ? 1 : grid, (vocab + BK - 1) / BK, 0.0);
}

// dWeight's last round is cut where that saves a twelfth of the product; else the sums stay those of the fp32
// accumulation over chunks, rounded once.  us, uncut -> cut with its merge: 26 702 x 20 264 x 1 792 (560 tiles) 2 000
// -> 1 559; 23 143 x 9 688 x 768 (114) 507 -> 292; 20 959 x 10 736 x 768 (126) 465 -> 274; 28 849 x 35 104 x 704 (414)
// 1 405 -> 1 218; 13 058 x 8 488 x 512 (68) 291 -> 124; 5 000 x 19 776 x 2 560 (780) 432 -> 403.
static SplitPlan plan_dweight(int64_t n_tokens, int64_t vocab, int64_t hidden_dim) {
    const int grid = persistent_grid();
    return plan_split(make_grid(hidden_dim, vocab).total, grid < 8 ? 1 : grid, (n_tokens + BK - 1) / BK, 1.0 / 12);
}

// The product with a k-major A, cut along k by the plan as far as the workspace reaches.
template <bool kBTrans>
static int cut_product(const char* fn, Product p, const SplitPlan& plan, void* workspace, int64_t workspace_bytes) {
    if (plan.n_slices == 1 || workspace == nullptr || workspace_bytes < slice_bytes(plan))
        return launch_gemm<kBf16, true, kBTrans, false>(fn, p, whole_tiles(p));
    p.sums = reinterpret_cast<float*>(workspace);
    int rc = plan.whole > 0 ? launch_gemm<kBf16, true, kBTrans, false>(fn, p, plan) : MRL_OK;
    if (rc == MRL_OK) rc = launch_gemm<kF32, true, kBTrans, true>(fn, p, plan);
    if (rc != MRL_OK) return rc;
    hipLaunchKernelGGL(merge_slices_kernel, dim3((unsigned)plan.rest, BN / 16), dim3(256), 0, p.stream, p.sums, plan, (int)p.m,
                       (int)p.n, (uint16_t*)p.out, p.ldo);
    return check_launch(fn);
}

// dHidden[t][h] = sum_v W[v][h] * dlogits[t][v]: the weight as it lies is the k-major operand; its rows
// beyond vocab read as zero, dlogits is read up to the next multiple of 64 columns.  Cut along the vocabulary
// as far as the workspace reaches.
static int dhidden(const char* fn, const void* weight, const void* dlogits, int64_t dlogits_row_stride, int64_t n_tokens,
                   int64_t vocab, int64_t hidden_dim, void* d_hidden, void* workspace, int64_t workspace_bytes,
                   hipStream_t s) {
    const Product p = {weight, hidden_dim, hidden_dim, dlogits, dlogits_row_stride, n_tokens, vocab, d_hidden, hidden_dim,
                       nullptr, s};
    return cut_product<false>(fn, p, plan_dhidden(n_tokens, vocab, hidden_dim), workspace, workspace_bytes);
}

// dW[v][h] (+)= sum_t hidden[t][h] * dlogits[t][v]: both operands k-major as they lie, any n_tokens; written as bf16 at
// once, cut along the tokens as far as the workspace reaches
template <int kOut>
static int dweight(const char* fn, const void* hidden, const void* dlogits, int64_t dlogits_row_stride, int64_t n_tokens,
                   int64_t vocab, int64_t hidden_dim, void* out, float* sums, void* workspace, int64_t workspace_bytes,
                   hipStream_t s) {
    const Product p = {hidden, hidden_dim, hidden_dim, dlogits, dlogits_row_stride, vocab, n_tokens, out, hidden_dim, sums, s};
    if constexpr (kOut == kBf16)
        return cut_product<true>(fn, p, plan_dweight(n_tokens, vocab, hidden_dim), workspace, workspace_bytes);
    else
        return launch_gemm<kOut, true, true, false>(fn, p, whole_tiles(p));
}

static int check_bwd(const char* fn, int64_t dlogits_row_stride, int64_t n_tokens, int64_t vocab, int64_t hidden_dim) {
    MRL_REQUIRE(n_tokens >= 0 && vocab > 0 && hidden_dim > 0, MRL_ERR_INVALID_ARG,
                "%s: n_tokens=%lld vocab=%lld hidden_dim=%lld", fn, (long long)n_tokens, (long long)vocab,
                (long long)hidden_dim);
    MRL_REQUIRE(hidden_dim % 8 == 0 && vocab % 8 == 0, MRL_ERR_UNSUPPORTED,
                "%s: hidden_dim=%lld and vocab=%lld must be multiples of 8", fn, (long long)hidden_dim, (long long)vocab);
    MRL_REQUIRE(dlogits_row_stride % BK == 0 && dlogits_row_stride >= vocab, MRL_ERR_INVALID_ARG,
                "%s: dlogits_row_stride=%lld must be a multiple of %d and at least vocab (the padding columns must hold "
                "zeros)", fn, (long long)dlogits_row_stride, BK);
    return MRL_OK;
}

}  // namespace mrl

// ------------------------------------------------------------------------------------------ C ABI
extern "C" int mrl_lmhead_logits(const void* hidden, const void* weight, int64_t n_tokens, int64_t vocab,
                                 int64_t hidden_dim, void* logits, int64_t logits_row_stride, void* stream) {
    const char* fn = "mrl_lmhead_logits";
    MRL_REQUIRE(n_tokens >= 0 && vocab > 0 && hidden_dim > 0, MRL_ERR_INVALID_ARG,
                "%s: n_tokens=%lld vocab=%lld hidden_dim=%lld", fn, (long long)n_tokens, (long long)vocab,
                (long long)hidden_dim);
    MRL_REQUIRE(hidden_dim % BK == 0 && vocab % 8 == 0 && logits_row_stride % 8 == 0, MRL_ERR_UNSUPPORTED,
                "%s: hidden_dim=%lld must be a multiple of %d, vocab=%lld and the row stride of 8", fn, (long long)hidden_dim, BK,
                (long long)vocab);
    MRL_REQUIRE(logits_row_stride >= vocab, MRL_ERR_INVALID_ARG, "%s: logits_row_stride below vocab", fn);
    if (n_tokens == 0) return MRL_OK;
    MRL_REQUIRE(hidden && weight && logits, MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    const mrl::Product p = {weight, hidden_dim, vocab, hidden, hidden_dim, n_tokens, hidden_dim, logits, logits_row_stride,
                            nullptr, mrl::as_stream(stream)};
    return mrl::launch_gemm<kBf16, false, false, false>(fn, p, mrl::whole_tiles(p));
}

extern "C" int mrl_lmhead_logprob_bwd(const void* hidden, const void* weight, const void* dlogits,
                                      int64_t dlogits_row_stride, int64_t n_tokens, int64_t vocab, int64_t hidden_dim,
                                      void* d_hidden, float* d_weight, void* stream) {
    const char* fn = "mrl_lmhead_logprob_bwd";
    int rc = mrl::check_bwd(fn, dlogits_row_stride, n_tokens, vocab, hidden_dim);
    if (rc != MRL_OK || n_tokens == 0) return rc;
    MRL_REQUIRE(hidden && weight && dlogits && d_hidden && d_weight, MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    hipStream_t s = mrl::as_stream(stream);
    rc = mrl::dhidden(fn, weight, dlogits, dlogits_row_stride, n_tokens, vocab, hidden_dim, d_hidden, nullptr, 0, s);
    if (rc != MRL_OK) return rc;
    return mrl::dweight<kF32Add>(fn, hidden, dlogits, dlogits_row_stride, n_tokens, vocab, hidden_dim, d_weight, d_weight, nullptr, 0, s);
}

extern "C" int64_t mrl_lmhead_bwd_workspace_bytes(int64_t n_tokens, int64_t vocab, int64_t hidden_dim) {
    if (n_tokens <= 0 || vocab <= 0 || hidden_dim <= 0) return 0;
    // one after the other
    const int64_t h = mrl::slice_bytes(mrl::plan_dhidden(n_tokens, vocab, hidden_dim));
    const int64_t w = mrl::slice_bytes(mrl::plan_dweight(n_tokens, vocab, hidden_dim));
    return h > w ? h : w;
}

extern "C" int mrl_lmhead_logprob_bwd_chunk(const void* hidden, const void* weight, const void* dlogits,
                                            int64_t dlogits_row_stride, int64_t n_tokens, int64_t vocab, int64_t hidden_dim,
                                            void* d_hidden, void* d_weight, float* d_weight_sums, int first, int last,
                                            void* workspace, int64_t workspace_bytes, void* stream) {
    const char* fn = "mrl_lmhead_logprob_bwd_chunk";
    int rc = mrl::check_bwd(fn, dlogits_row_stride, n_tokens, vocab, hidden_dim);
    if (rc != MRL_OK) return rc;
    MRL_REQUIRE(n_tokens > 0, MRL_ERR_INVALID_ARG, "%s: an empty chunk", fn);
    MRL_REQUIRE(hidden && weight && dlogits && d_hidden && (d_weight || !last) && (d_weight_sums || (first && last)),
                MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    MRL_REQUIRE(mrl::aligned(workspace, 16) && mrl::aligned(d_weight_sums, 16), MRL_ERR_MISALIGNED,
                "%s: the workspace and d_weight_sums must be 16-byte aligned", fn);
    hipStream_t s = mrl::as_stream(stream);
    rc = mrl::dhidden(fn, weight, dlogits, dlogits_row_stride, n_tokens, vocab, hidden_dim, d_hidden, workspace,
                      workspace_bytes, s);
    if (rc != MRL_OK) return rc;
#define MRL_DWEIGHT(OUT, dst) \
    mrl::dweight<OUT>(fn, hidden, dlogits, dlogits_row_stride, n_tokens, vocab, hidden_dim, dst, d_weight_sums, workspace, workspace_bytes, s)
    if (first) return last ? MRL_DWEIGHT(kBf16, d_weight) : MRL_DWEIGHT(kF32, d_weight_sums);
    return last ? MRL_DWEIGHT(kSumToBf16, d_weight) : MRL_DWEIGHT(kF32Add, d_weight_sums);
#undef MRL_DWEIGHT
}
