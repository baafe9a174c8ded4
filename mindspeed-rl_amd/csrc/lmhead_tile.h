// The tile loop of the lm_head matrix products on the bf16 matrix cores of gfx950, shared by the plain
// products (lmhead_gemm.hip) and by the fused lm_head + log-prob forward (lmhead.hip), which differ in
// what they do with a finished 256 x 256 tile of fp32 results.
//
//     tile[n][m] = sum_k A[m][k] * B[n][k]
//
// A workgroup of 256 threads (2 x 2 wavefronts, one per SIMD, wavefront tile 128 x 128 = 8 x 8 blocks of
// v_mfma_f32_16x16x32_bf16 in 256 accumulator registers) walks a sequence of tiles; operands go from
// global memory straight into LDS (buffer_load ... lds), XOR-swizzled 16-byte chunks, 64 k to a k-step, and
// the loop runs over the flattened (tile, k-step) sequence, so the first loads of the next tile are in flight
// while the current one is finished.  At the board's power limit the 16x16x32 MFMA runs the same flops about
// 18 % faster than 32x32x16.
//
// An operand is k-contiguous ([rows, K]) or "k-major" ([K, rows] with the rows contiguous, kATrans /
// kBTrans): its fragments (8 consecutive k per lane) then come out of ds_read_b64_tr_b16, the LDS read
// of gfx950 that transposes 4 x 4 blocks of 16-bit entries across lanes, and rows of k beyond K read as
// zero through the range check of the buffer descriptor, so K needs no padding there.
//
// What bounds it: the matrix cores at the board's power limit, and before that the time from a request to its
// bytes in LDS, since a wavefront that is alone on its SIMD idles whenever it waits.  So requests go out evenly,
// 8 a sub-step, and as early as the 160 KiB of LDS allow: two buffers of a k-step for an operand are the least;
// a k-contiguous A has a third one (its bytes lie a whole k-step ahead), and a k-major operand is requested by
// halves of a k-step (32 k-rows, still whole 128-byte lines; halves of a k-contiguous operand would be half
// lines, which measured 10 % slower).  With two buffers and all 16 requests in every other sub-step, before ->
// now, ms (12 356 x 152 064 x 3 584; 4 000 x 129 280 x 5 120; medians of 12 steps in turn on one board): logits 9.58 ->
// 9.33, 3.86 -> 3.72; dWeight 10.41 -> 9.92, 4.05 -> 3.97; dHidden 10.76 -> 9.70, 4.41 -> 3.73, of which its whole tiles at
// the second size 3.32 -> 2.93 (the rest are cut, see plan_split); fused forward 9.37 -> 9.31, 3.87 -> 3.75.
#pragma once

#include "mrl_internal.h"

namespace mrl_tile {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// Wavefront layout of the 256 x 256 tile: 2 wavefronts along m (128 rows of A each) by 2 along n
// (128 rows of B each); a wavefront owns 8 x 8 MFMA blocks of 16 x 16.
constexpr int kWavesN = 2;
constexpr int kWaves = 2 * kWavesN;
constexpr int kThreads = 64 * kWaves;
constexpr int kBlocks = 8;                       // 16-row blocks of A, and of B, per wavefront
constexpr int kLoadsPerWave = 32 / kWaves;       // requests of a wavefront for a k-step of an operand
constexpr int kSlotK = 32;                       // k-rows of a slot of a k-major operand: half a k-step
constexpr int kSlotLoads = kLoadsPerWave / 2;    // requests of a wavefront for a slot
constexpr int BM = 256;                          // rows of A per tile
constexpr int BN = 256;                          // rows of B per tile
constexpr int BK = 64;                           // k elements per k-step
constexpr int kOperandBytes = 256 * BK * 2;      // one operand of one k-step: 256 rows x 128 bytes
constexpr int kSlotBytes = kOperandBytes / 2;
constexpr int kSpareBytes = kOperandBytes;       // what the epilogue may use
constexpr int kLdsBytes = 4 * kOperandBytes + kSpareBytes;      // two buffers each, and A's third or the spare one

// Element offset (row * ld + column, without the k-step) of the chunk that lane `lane` of wavefront `wave`
// brings in with its load j (0..3) of an operand tile; load j + 4 lies 32 rows further on.  Physical slot of a
// 16-byte chunk inside its 256-byte pair of rows: logical slot ^ (pair & 15), logical = (row & 1) * 8 + chunk.
__device__ __forceinline__ int64_t kstep_src_offset(int wave, int lane, int j, int64_t ld) {
    const int phys_row = (wave * kLoadsPerWave + j) * 8 + (lane >> 3);
    const int pair = phys_row >> 1;
    const int slot = ((phys_row & 1) << 3) | (lane & 7);
    const int logical = slot ^ (pair & 15);
    return (int64_t)(2 * pair + (logical >> 3)) * ld + (logical & 7) * 8;
}

// The same for a k-major operand [K, rows], j 0..1; load j + 2 lies 16 k-rows further on.  Its slot is cut into 4
// column blocks of 64 rows of the operand; a column block holds its 32 k-rows at a pitch of 128 bytes (4 KiB),
// one for each wavefront to bring in: a load fills 1 KiB with 8 k-rows, 8 lanes per 128-byte line as for the
// k-contiguous operand.  Inside a k-row the four 32-byte segments (16 rows of the operand, what one
// fragment read takes from it) are permuted: byte offset ^ (f(k) << 5), f(k) = (k >> 1 & 1) |
// ((k >> 3 & 1) << 1); with the bank half that k & 1 selects, the 8 k-rows that half a wavefront
// reads at a time fall on different banks.
__device__ __forceinline__ int tr_swizzle(int k) { return (((k >> 1) & 1) | (((k >> 3) & 1) << 1)) << 5; }
__device__ __forceinline__ int64_t slot_src_offset_kmajor(int wave, int lane, int j, int64_t ld) {
    const int k = 8 * j + (lane >> 3);
    const int byte = ((lane & 7) * 16) ^ tr_swizzle(k);
    return (int64_t)k * ld + wave * 64 + (byte >> 1);
}

typedef floatx4 Accumulators[kBlocks][kBlocks];

// The k_range of a sequence whose tiles all run over the whole of K.
struct WholeK {
    static constexpr bool kSettle = false;
    __device__ __forceinline__ void k_range(int, int n_ksteps, int& begin, int& end) const {
        begin = 0;
        end = n_ksteps;
    }
};

// Runs the workgroup's tiles.  `smem`: kLdsBytes of LDS, 16-byte aligned.
// `seq`: n_tiles; coords(j, tm, tn), the tile coordinates (in units of 256 rows of A and of B) of the j-th
// tile of this workgroup, and k_range(j, n_ksteps, begin, end), the k-steps of 64 that go into it (at least
// one), all uniform over the workgroup; kSettle: loads that the epilogue leaves behind are waited for ahead of the
// k loop.  `epilogue(acc, j, tm, tn, spare)` is called with the
// finished tile: wavefront (wv, wt) = (wave / 2, wave % 2) holds rows wv * 128 .. + 127 of A (m) and
// wt * 128 .. + 127 of B (n); acc[vb][tb] is the 16 x 16 block at m = 16 vb, n = 16 tb of it, of which a
// lane holds column n = lane & 15 and rows m = 4 (lane >> 4) .. + 3.  Rows of a ragged last tile beyond
// M or N hold products of whatever is read there (zeros mostly): the epilogue must skip them.  spare: kSpareBytes
// of LDS until it returns, wavefront w's requests going to its w-th quarter from then on: what one wavefront
// reads of another's quarter is read before a barrier.  K % 64 == 0 unless an operand is k-major.  Every thread of
// the workgroup must call this (it contains barriers).
template <bool kATrans, bool kBTrans, typename Seq, typename Epilogue>
__device__ __forceinline__ void mfma_tile_loop(unsigned char* smem, const uint16_t* __restrict__ A, int64_t lda, int M,
                                               const uint16_t* __restrict__ B, int64_t ldb, int N, int K, const Seq& seq,
                                               Epilogue&& epilogue) {
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wv = wave / kWavesN, wt = wave % kWavesN;
    const int n_tiles = seq.n_tiles;
    if (n_tiles <= 0) return;
    const int n_ksteps = (K + BK - 1) / BK;           // a last partial step only with k-major operands

    // ---- loader state, one for each operand: the tile whose k-steps (k-contiguous) or slots (k-major) are
    // being requested, and which of them
    struct Loader {
        int j, at, begin, end;                        // index into the workgroup's tiles; k-step or slot, the tile's range
        int off[kLoadsPerWave / 2];                   // per lane, the same for every tile
        int half;                                     // from the first half of a wavefront's requests to the second
        mrl::rsrc_t rsrc;
        const uint16_t* base;                         // k-major: where the slot's rows begin
        uint32_t bytes, last_bytes;                   // k-major: range of a whole slot, and of one that K ends in
    };
    Loader la, lb;
    // What lies outside of an operand is cut off by the range of its descriptor and reads as zero: rows beyond
    // the last of a ragged tile (of a k-major operand in its last k-row; in the others such columns hold what
    // the next k-row begins with - no product of them is stored either), and k-rows beyond K.  A k-major
    // operand takes a descriptor per slot: its base moves by 32 k-rows, which may be more than the 4 GiB
    // that an offset can span.  The range is checked against the lane's offset alone: rows have to be in that,
    // the uniform offset (the k-step of a k-contiguous operand) stays inside a row.
    auto describe_slot = [&](Loader& l) {
        const int rest = K - l.at * kSlotK;
        l.rsrc = mrl::make_rsrc(l.base, rest >= kSlotK ? l.bytes : (rest > 0 ? l.last_bytes : 0u));
    };
    auto set_tile = [&](Loader& l, bool is_a, int j) {
        const uint16_t* P = is_a ? A : B;
        const int64_t ld = is_a ? lda : ldb;
        int tm, tn, begin, end;
        seq.coords(j, tm, tn);
        seq.k_range(j, n_ksteps, begin, end);
        // uniform, but the compiler cannot tell from what a division leaves
        const int t = __builtin_amdgcn_readfirstlane(is_a ? tm : tn);
        l.begin = __builtin_amdgcn_readfirstlane(begin);
        l.end = __builtin_amdgcn_readfirstlane(end);
        l.j = j;
        const int rows = (is_a ? M : N) - t * BM;
        static_assert(BM == BN, "one tile size");
        if (is_a ? kATrans : kBTrans) {
            l.begin *= 2;
            l.end *= 2;
            l.base = P + (int64_t)l.begin * kSlotK * ld + (int64_t)t * BM;
            l.bytes = (uint32_t)(((kSlotK - 1) * ld + rows) * 2);
            l.last_bytes = (uint32_t)((((K & (kSlotK - 1)) - 1) * ld + rows) * 2);
            l.at = l.begin;
            describe_slot(l);
        } else {
            l.rsrc = mrl::make_rsrc(P + (int64_t)t * BM * ld, (uint32_t)(min(BM, rows) * ld * 2));
            l.at = l.begin;
        }
    };
    // the wavefront's request i of a k-step or slot of an operand, into the 32 or 16 KiB at `dst`
    auto request = [&](const Loader& l, bool trans, unsigned char* dst, int i) {
        const int per = trans ? kSlotLoads : kLoadsPerWave;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(l.rsrc, (void __attribute__((address_space(3)))*)(dst + (wave * per + i) * 1024),
                                                 16, l.off[i % (per / 2)] + (i < per / 2 ? 0 : l.half),
                                                 trans ? 0u : (uint32_t)(l.at * BK * 2), 0, 0);
    };
    auto set_offsets = [&](Loader& l, bool trans, int64_t ld) {
#pragma unroll
        for (int i = 0; i < (trans ? kSlotLoads : kLoadsPerWave) / 2; ++i)
            l.off[i] = (int)((trans ? slot_src_offset_kmajor(wave, lane, i, ld) : kstep_src_offset(wave, lane, i, ld)) * 2);
        l.half = (int)((trans ? 16 : 32) * ld * 2);
    };
    // with describe_slot: the next slot of the same tile
    auto next_slot_base = [&](Loader& l, int64_t ld) {
        l.base += kSlotK * ld;
        ++l.at;
    };
    // After the last k-step of the last tile the requests go on (the schedule below has no branches):
    // they fetch valid bytes of the last tile into a buffer that nobody reads any more.
    auto next_tile_if_done = [&](Loader& l, bool is_a) {
        if (l.at == l.end) set_tile(l, is_a, l.j + 1 < n_tiles ? l.j + 1 : l.j);
    };

    // Fragment addresses.  A lane reads row (lane & 15) of a 16-row block (8 row pairs, 2 KiB), chunk
    // 4 ks + (lane >> 4) of its 8: inside the block its pair is (lane >> 1) & 7, the pair's low bits
    // are ((block & 1) << 3) | that, and the physical slot is the logical one XOR those bits.
    int frag_off[2][2];                                   // [block parity][k sub-step of 32]
#pragma unroll
    for (int par = 0; par < 2; ++par)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int pair_in_block = (lane >> 1) & 7;
            const int slot = ((((lane & 1) ^ par) << 3) | ((4 * ks + (lane >> 4)) ^ pair_in_block));
            frag_off[par][ks] = pair_in_block * 256 + slot * 16;
        }
    // The same for a k-major operand: k-row 8 (lane >> 4) + 4 r + ((lane >> 2) & 3) of a slot for the two
    // reads r = 0, 1 of a fragment, 8 bytes at row 16 block + 4 (lane & 3) of it (column block
    // block >> 2, segment block & 3 of the k-row); after the transposing read, lane i of each 16 holds
    // row 16 block + i for 4 consecutive k.
    int tr_off[4];                                        // [block & 3]
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int g = lane >> 4, kk = (lane >> 2) & 3;
        tr_off[j] = (8 * g + kk) * 128 + ((j * 32) ^ tr_swizzle(8 * g + kk)) + (lane & 3) * 8;
    }
    // A k-contiguous operand's fragments are ordinary 16-byte loads (the compiler waits for them); a k-major
    // operand's arrive as the two 8-byte halves that the asm reads below deliver, and stay two values until
    // `landed` has passed them through the loop's own wait (members that a product does not use fold away).
    typedef long long2v __attribute__((ext_vector_type(2)));
    struct Frags {
        bf16x8 a[kBlocks], b[kBlocks];
        long a_lo[kBlocks], a_hi[kBlocks], b_lo[kBlocks], b_hi[kBlocks];
    };
    // fragment of 16-row block `blk` (0..15 inside the tile) of an operand whose k-step starts at `op`
    auto read_kcontig = [&](const unsigned char* op, int blk, int ks) {
        return *reinterpret_cast<const bf16x8*>(op + blk * 2048 + frag_off[blk & 1][ks]);
    };
    // The transposing read goes out as inline assembly: through the builtin the compiler cannot tell it
    // from an access to the bytes that the requests in flight are writing and waits for all of them
    // (vmcnt(0)) before every read.  The price: it does not wait for the result either - the loop
    // below does (lgkmcnt(0) before a sub-step consumes fragments read during the one before), and
    // `landed` makes that wait the point where the halves become usable values: whatever the compiler does
    // with them (join them in place, or copy them) it can only do behind the wait.
    const unsigned smem_lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    auto read_kmajor = [&](unsigned addr, int at, long& lo, long& hi) {
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(addr), "i"(at) : "memory");
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(addr), "i"(at + 512) : "memory");
    };
    auto join = [](long lo, long hi) {
        long2v both;
        both[0] = lo;
        both[1] = hi;
        return __builtin_bit_cast(bf16x8, both);
    };
    // placed right behind the wait for a fragment set: every half of the set is an input and an output of an
    // empty statement there, so no use of it (and no copy of it) can be scheduled ahead of the wait
    auto landed = [&](Frags& f) {
        static_assert(kBlocks == 8, "the operand lists below name 8 fragments");
        if (kATrans)
            asm volatile("" : "+v"(f.a_lo[0]), "+v"(f.a_hi[0]), "+v"(f.a_lo[1]), "+v"(f.a_hi[1]), "+v"(f.a_lo[2]),
                              "+v"(f.a_hi[2]), "+v"(f.a_lo[3]), "+v"(f.a_hi[3]), "+v"(f.a_lo[4]), "+v"(f.a_hi[4]),
                              "+v"(f.a_lo[5]), "+v"(f.a_hi[5]), "+v"(f.a_lo[6]), "+v"(f.a_hi[6]), "+v"(f.a_lo[7]),
                              "+v"(f.a_hi[7]));
        if (kBTrans)
            asm volatile("" : "+v"(f.b_lo[0]), "+v"(f.b_hi[0]), "+v"(f.b_lo[1]), "+v"(f.b_hi[1]), "+v"(f.b_lo[2]),
                              "+v"(f.b_hi[2]), "+v"(f.b_lo[3]), "+v"(f.b_hi[3]), "+v"(f.b_lo[4]), "+v"(f.b_hi[4]),
                              "+v"(f.b_lo[5]), "+v"(f.b_hi[5]), "+v"(f.b_lo[6]), "+v"(f.b_hi[6]), "+v"(f.b_lo[7]),
                              "+v"(f.b_hi[7]));
    };
    // Where a k-step lies: byte offsets of its parts of A and B.  A k-contiguous A has three buffers, everything
    // else two; a k-major operand's buffer is two slots.
    struct Place {
        int a, b;
    };
    constexpr int kOperandBytesA = (kATrans ? 2 : 3) * kOperandBytes;
    // LDS addresses of this wavefront's k-major fragments, by block & 3, in a k-step at 0
    unsigned tr_a[4], tr_b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        tr_a[j] = smem_lds + (unsigned)(wv * (kBlocks / 4) * 4096 + tr_off[j]);
        tr_b[j] = smem_lds + (unsigned)(wt * (kBlocks / 4) * 4096 + tr_off[j]);
    }
    // read r (0..15) of a fragment set, in the order the MFMAs need them: a0, all of b, a1..a7.  at: the
    // k-step, ks: its half
    auto read1 = [&](Frags& f, const Place& at, int ks, int r) {
        const bool is_a = r == 0 || r > kBlocks;
        const int blk = r == 0 ? 0 : (r <= kBlocks ? r - 1 : r - kBlocks);
        if (is_a) {
            if (kATrans) read_kmajor(tr_a[blk & 3] + at.a, (blk >> 2) * 4096 + ks * kSlotBytes, f.a_lo[blk], f.a_hi[blk]);
            else f.a[blk] = read_kcontig(smem + at.a, wv * kBlocks + blk, ks);
        } else {
            if (kBTrans) read_kmajor(tr_b[blk & 3] + at.b, (blk >> 2) * 4096 + ks * kSlotBytes, f.b_lo[blk], f.b_hi[blk]);
            else f.b[blk] = read_kcontig(smem + at.b, wt * kBlocks + blk, ks);
        }
    };
    floatx4 acc[kBlocks][kBlocks];
    auto zero_acc = [&]() {
#pragma unroll
        for (int vb = 0; vb < kBlocks; ++vb)
#pragma unroll
            for (int tb = 0; tb < kBlocks; ++tb)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[vb][tb][i] = 0.f;
    };
    // Empty statements that demand every accumulator in the accumulator half of the register file:
    // placed after the zeroing and before the store, they keep the allocator from spreading the 64
    // four-register values over both halves (and copying them around inside the k loop).
    auto pin_acc = [&]() {
#pragma unroll
        for (int vb = 0; vb < kBlocks; ++vb)
#pragma unroll
            for (int tb = 0; tb < kBlocks; ++tb) asm volatile("" : "+a"(acc[vb][tb]));
    };
    auto mfma1 = [&](const Frags& f, int i) {
        const int vb = i / kBlocks, tb = i % kBlocks;
        const bf16x8 a = kATrans ? join(f.a_lo[vb], f.a_hi[vb]) : f.a[vb];
        const bf16x8 b = kBTrans ? join(f.b_lo[tb], f.b_hi[tb]) : f.b[tb];
        acc[vb][tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[vb][tb], 0, 0, 0);
    };

    // One wavefront per SIMD: memory instructions are placed between the MFMAs of the same instruction
    // stream (an MFMA holds the matrix pipe for 16 cycles, other instructions issue meanwhile).  A k-step p is an
    // even and an odd sub-step of 64 MFMAs, each on a fragment set that was read during the one before:
    //   even: MFMAs on G0 | reads G1 (p, k 32..63)  | requests: k-major slot 2p+4, or k-step p+2 of a k-contiguous A
    //   odd:  MFMAs on G1 | reads G0 (p+1, k 0..31) | requests: k-major slot 2p+5, k-step p+2 of a k-contiguous B
    // A wait and a barrier stand before the odd sub-step: k-step p+1 (its first slot) has landed, the buffers of
    // k-step p are free; with a k-major operand also before the even one: slot 2p+1 has landed, slot 2p is free.
    // Requests land in order, so a wait is for all but the youngest: those that follow what the next reads need
    // (stores of an epilogue in between only make it wait for more).
    // Sweeping a product's requests over one in 3 .. 8 MFMAs changes it by less than 1 %, the fused forward by 2 %
    // (densest best); the mixed product's 12 of the odd sub-step one in 3 MFMAs: 3 % slower than one in 5.
#define MRL_SB __builtin_amdgcn_sched_barrier(0)
    constexpr int kMfmas = kBlocks * kBlocks, kReads = 2 * kBlocks;
    static_assert(kMfmas == 64 && kReads == 16 && kLoadsPerWave == 8, "the schedule below is written for these counts");
    constexpr bool kSlots = kATrans || kBTrans, kMixed = kSlots && !(kATrans && kBTrans);
    constexpr int kOddRequests = kMixed ? 12 : 8, kEvenRequests = kMixed ? 4 : 8;
    constexpr int kOddEvery = kMixed ? 5 : (kSlots ? 6 : 3), kEvenEvery = kMixed ? 12 : (kSlots ? 6 : 3);
    // request i of the odd sub-step of the k-step at `at`, and of its even one (free_a: A's third buffer)
    auto odd_request = [&](const Place& at, int i) {
        if (kATrans && i < kSlotLoads) request(la, true, smem + at.a + kSlotBytes, i);
        else if (kBTrans) request(lb, true, smem + at.b + kSlotBytes, i - (kATrans ? kSlotLoads : 0));
        else request(lb, false, smem + at.b, i - (kATrans ? kSlotLoads : 0));
    };
    auto even_request = [&](const Place& at, int free_a, int i) {
        if (kATrans && i < kSlotLoads) request(la, true, smem + at.a, i);
        else if (kBTrans) request(lb, true, smem + at.b, i - (kATrans ? kSlotLoads : 0));
        else request(la, false, smem + free_a, i);
    };
    auto sub_step = [&](Frags& now, Frags& next, const Place& at, const Place& read_at, int free_a, bool odd) {
        MRL_SB;
        if (kSlots || odd) {
            if (!kSlots) __builtin_amdgcn_s_waitcnt(0x0078);                  // vmcnt(8) lgkmcnt(0)
            else if (odd && kMixed) __builtin_amdgcn_s_waitcnt(0x0074);       // vmcnt(4) lgkmcnt(0)
            else __builtin_amdgcn_s_waitcnt(0x4070);                          // vmcnt(16) lgkmcnt(0)
            landed(now);
            asm volatile("s_barrier" ::: "memory");
        }
        MRL_SB;
#pragma unroll
        for (int i = 0; i < kMfmas; ++i) {
            mfma1(now, i);
            MRL_SB;
            if (i % 3 == 0 && i / 3 < kReads) {
                read1(next, read_at, odd ? 0 : 1, i / 3);
                MRL_SB;
            }
            if (odd ? (i % kOddEvery == 1 && i / kOddEvery < kOddRequests)
                    : (i % kEvenEvery == 1 && i / kEvenEvery < kEvenRequests)) {
                if (odd) odd_request(at, i / kOddEvery);
                else even_request(at, free_a, i / kEvenEvery);
                MRL_SB;
            }
            // behind the last request; scalar work left to the end of the sub-step would leave the matrix pipe idle
            if (kATrans && i == 57) {
                next_slot_base(la, lda);
                MRL_SB;
                describe_slot(la);
                MRL_SB;
            }
            if (kBTrans && i == 60) {
                next_slot_base(lb, ldb);
                MRL_SB;
                describe_slot(lb);
                MRL_SB;
            }
        }
        if (!kATrans && !odd) ++la.at;
        if (!kBTrans && odd) ++lb.at;
        if (odd == kATrans) next_tile_if_done(la, true);
        if (odd) next_tile_if_done(lb, false);
    };
    static_assert(kATrans || !kBTrans, "only a k-contiguous A has a third buffer");
    Frags G0, G1;
    set_offsets(la, kATrans, lda);
    set_offsets(lb, kBTrans, ldb);
    set_tile(la, true, 0);
    set_tile(lb, false, 0);
    Place at = {0, kOperandBytesA};
    Place next = {kOperandBytes, kOperandBytesA + kOperandBytes};
    int free_a = kATrans ? 0 : 2 * kOperandBytes;
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        const Place& p = which ? next : at;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
#pragma unroll
            for (int i = 0; i < kSlotLoads; ++i)
                request(la, kATrans, smem + p.a + (kATrans ? half * kSlotBytes : 0), kATrans ? i : half * kSlotLoads + i);
#pragma unroll
            for (int i = 0; i < kSlotLoads; ++i)
                request(lb, kBTrans, smem + p.b + (kBTrans ? half * kSlotBytes : 0), kBTrans ? i : half * kSlotLoads + i);
            if (kATrans) {
                next_slot_base(la, lda);
                describe_slot(la);
            }
            if (kBTrans) {
                next_slot_base(lb, ldb);
                describe_slot(lb);
            }
        }
        if (!kATrans) ++la.at;
        if (!kBTrans) ++lb.at;
        next_tile_if_done(la, true);
        next_tile_if_done(lb, false);
    }
    __builtin_amdgcn_s_waitcnt(0x4F70);                // vmcnt(16): the first k-step has landed
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int r = 0; r < kReads; ++r) read1(G0, at, 0, r);
    for (int mine = 0; mine < n_tiles; ++mine) {
        zero_acc();
        pin_acc();
        int k_begin, k_end;
        seq.k_range(mine, n_ksteps, k_begin, k_end);
        if (Seq::kSettle) __builtin_amdgcn_s_waitcnt(0x0F70);
        for (int kstep = k_begin; kstep < k_end; ++kstep) {
            sub_step(G0, G1, at, at, free_a, false);
            sub_step(G1, G0, at, next, free_a, true);
            const Place done = at;
            at = next;
            next.b = done.b;
            next.a = kATrans ? done.a : free_a;
            if (!kATrans) free_a = done.a;
        }
        pin_acc();
        int tm, tn;
        seq.coords(mine, tm, tn);
        epilogue(acc, mine, tm, tn, kATrans ? smem + 4 * kOperandBytes : smem + free_a);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                // nothing is in flight into LDS when the workgroup ends
#undef MRL_SB
}

}  // namespace mrl_tile
