// Response windows in rows of the logits: what sequence i's tokens occupy of a packed or padded batch.
#pragma once

#include "mrl_internal.h"

namespace mrl {

__device__ __forceinline__ int64_t load_index(const void* p, int dtype, int64_t i) {
    return dtype == MRL_I32 ? (int64_t) reinterpret_cast<const int32_t*>(p)[i]
                            : reinterpret_cast<const int64_t*>(p)[i];
}

// (start, n) of the window that postprocess_packed_seqs copies for sequence i
__device__ __forceinline__ void unpad_window(const int32_t* __restrict__ seqlens, const int32_t* __restrict__ cu,
                                             const void* __restrict__ prompt, int prompt_dtype, int i,
                                             int64_t& start, int64_t& n) {
    start = (int64_t)cu[i];
    n = (int64_t)seqlens[i];
    if (prompt != nullptr) {
        const int64_t skip = load_index(prompt, prompt_dtype, i) - 1;
        if (skip < n) {
            n -= skip + 1;
            start += skip;
        }
    }
}

// What a sequence's response window is in rows of the logits, for both layouts: `n` rows from row `start` on.
struct SeqWindows {
    int packed;
    const int32_t* seqlens;         // packed
    const int32_t* cu;
    int64_t padded_s;               // padded: rows per sequence
    const void* prompt;
    int prompt_dtype;
    const void* resp;               // padded
    int resp_dtype;
    __device__ __forceinline__ void window(int64_t i, int64_t& start, int64_t& n) const {
        if (packed) {
            unpad_window(seqlens, cu, prompt, prompt_dtype, (int)i, start, n);
        } else {
            const int64_t p = load_index(prompt, prompt_dtype, i);
            int64_t lo = p - 1, hi = p + load_index(resp, resp_dtype, i) - 1;
            lo = lo < 0 ? 0 : (lo > padded_s ? padded_s : lo);
            hi = hi < 0 ? 0 : (hi > padded_s ? padded_s : hi);
            start = i * padded_s + lo;
            n = hi - lo;
        }
    }
};

inline int check_seq_windows(const char* fn, const SeqWindows& q, int64_t batch, int64_t width, int64_t n_rows) {
    MRL_REQUIRE(batch >= 0 && batch <= (1LL << 20) && width >= 0 && n_rows >= 0, MRL_ERR_INVALID_ARG,
                "%s: batch=%lld width=%lld n_rows=%lld", fn, (long long)batch, (long long)width, (long long)n_rows);
    // callers multiply the two
    MRL_REQUIRE(batch == 0 || width <= 0x7fffffffffffffffLL / batch, MRL_ERR_UNSUPPORTED, "%s: batch=%lld x width=%lld out of range",
                fn, (long long)batch, (long long)width);
    MRL_REQUIRE(int_dtype_bytes(q.prompt_dtype) != 0 && (q.packed || int_dtype_bytes(q.resp_dtype) != 0),
                MRL_ERR_UNSUPPORTED, "%s: length dtypes %d and %d (want I32 or I64)", fn, q.prompt_dtype, q.resp_dtype);
    MRL_REQUIRE(batch == 0 || (q.prompt && (q.packed ? q.seqlens && q.cu : q.resp && q.padded_s >= 0)), MRL_ERR_INVALID_ARG,
                "%s: NULL pointer", fn);
    return MRL_OK;
}

}  // namespace mrl
