// PPO's value side of the path: token-level rewards with the KL penalty, the GAE reverse scan, masked
// whitening, and the clipped value loss of the critic (forward and backward).  All operands are
// [batch, width] fp32 tensors of a few hundred thousand entries, so every kernel here is
// launch-bound; the layouts are chosen for determinism (fixed summation order, fp64 accumulators,
// no float atomics) and, for the scan, for the reference's exact operation order.
#include "mrl_internal.h"
#include "policy_terms.h"

namespace {

using namespace mrl_loss;

constexpr int kScanBlock = 512;
constexpr int kScanChunk = 4096;     // entries of a row staged in LDS per step of the scan
constexpr int kReplay = 16;          // steps of the scan between two results that the chain keeps
constexpr int kReduceBlock = 1024;

// Sum of one double per thread over a workgroup of kReduceBlock threads, fixed order; every thread
// gets the total.  `lds` holds kReduceBlock / 64 + 1 doubles.
__device__ __forceinline__ double block_sum(double x, double* lds) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    constexpr int kWaves = kReduceBlock / 64;
    __syncthreads();                     // the previous call's total has been read by everyone
    if (lane == 0) lds[wave] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < kWaves; ++w) t += lds[w];
        lds[kWaves] = t;
    }
    __syncthreads();
    return lds[kWaves];
}

// Three of them at once: the same sums in the same order, one pair of barriers (value_loss_finish_kernel 3.7 -> 3.1 us,
// whiten_moments_kernel 4.6 -> 4.2 with three calls before).
__device__ __forceinline__ void block_sum3(double (&x)[3], double (*lds)[kReduceBlock / 64 + 1]) {
    constexpr int kWaves = kReduceBlock / 64;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) x[q] += __shfl_xor(x[q], off, 64);
        if ((threadIdx.x & 63) == 0) lds[q][threadIdx.x >> 6] = x[q];
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) t += lds[threadIdx.x][w];
        lds[threadIdx.x][kWaves] = t;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 3; ++q) x[q] = lds[q][kWaves];
}

// ---------------------------------------------------------------------------- KL-penalised rewards
// One workgroup per sample: kld = penalty(old, ref) * mask, rewards = onehot(last response token) *
// score - beta * kld, row_kl = sum(kld * mask) / (sum(mask) + 1e-8).  A thread has four columns on their way at a time:
// bound by loads that follow each other, 122 x 4 096 8.4 -> 6.6 us, 128 x 2 048 5.5 -> 4.9.
constexpr int kColumns = 4;
__global__ __launch_bounds__(256) void kl_rewards_kernel(const float* __restrict__ old_lp,
                                                         const float* __restrict__ ref_lp,
                                                         const void* __restrict__ lens, int ldtype,
                                                         const float* __restrict__ scores, int64_t width, int penalty,
                                                         float beta, float* __restrict__ rewards,
                                                         float* __restrict__ row_kl) {
    __shared__ double part[256 / 64];
    const int64_t i = blockIdx.x;
    const int64_t n = ldtype == MRL_I32 ? (int64_t) reinterpret_cast<const int32_t*>(lens)[i]
                                        : reinterpret_cast<const int64_t*>(lens)[i];
    // python indexing of reward_tensor[i, n - 1]: a zero length lands on the last column
    int64_t hot = n - 1;
    if (hot < 0) hot += width;
    const float score = scores[i];
    Params p = {0.f, 0.f, 0.f, 0.f, 1.f, penalty, 0};
    double acc = 0.0;
    for (int64_t j0 = threadIdx.x; j0 < width; j0 += kColumns * 256) {
        float old_mine[kColumns], ref_mine[kColumns];
#pragma unroll
        for (int q = 0; q < kColumns; ++q) {
            const int64_t e = i * width + (j0 + q * 256 < width ? j0 + q * 256 : j0);
            old_mine[q] = old_lp[e];
            ref_mine[q] = ref_lp[e];
        }
#pragma unroll
        for (int q = 0; q < kColumns; ++q) {
            const int64_t j = j0 + q * 256;
            if (j >= width) break;
            const float m = j < n ? 1.f : 0.f;
            const Token t = token_terms<false>(old_mine[q], 0.f, false, ref_mine[q], 0.f, p);
            const float kld = t.kl * m;
            const float r = j == hot ? score : 0.f;
            rewards[i * width + j] = r - beta * kld;
            if (m != 0.f) acc += (double)(kld * m);
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double s = part[0] + part[1] + part[2] + part[3];
        const float cnt = (float)(n < 0 ? 0 : (n > width ? width : n));
        row_kl[i] = (float)s / (cnt + 1e-8f);
    }
}

// ---------------------------------------------------------------------------- GAE reverse scan
// One workgroup per sample.  The recurrence lastgaelam = delta_t + (gamma*lam) * lastgaelam is
// evaluated in the reference's order and with its roundings (separate multiply and
// add, no contraction), so advantages and returns are bit-identical to the torch loop.  gl is gamma*lam
// as the host formed it: python multiplies the two in double and torch rounds the product to fp32 once.
//
// Bound by that chain: two dependent operations per token, 13.3 cycles measured without anything else.  So
// nothing else is left on it.  All threads form the deltas; one wavefront runs through them, 64 at a time in
// the lanes of one register and read from there (v_readlane fits into the chain's own gaps, where a lane's own
// LDS reads and writes of four entries took another 12 cycles a token), and keeps every 16th result only.  From
// those all threads then take the 16 steps in between once more, side by side: the same operations on the same
// operands, so the same bits.
// Batch 128 x width 2048: 14.9 us, 14.4 cycles a token (24.4 with the chain in one lane, its entries by LDS);
// x 4096 46.3 -> 27.1; 16 x 512 7.8 -> 5.5.  16 steps apart: each kept result costs the chain an LDS write.
//
// kMoments: leaves the masked moments (sum m, sum m x, sum m x^2) of the sample's advantages, in fp64, for
// the whitening that follows.
struct Moments {
    double w, x, xx;
};

template <bool kMoments>
__global__ __launch_bounds__(kScanBlock) void gae_scan_kernel(const float* __restrict__ rewards,
                                                              const float* __restrict__ values, int64_t width,
                                                              float gamma, float gl, float* __restrict__ adv,
                                                              float* __restrict__ ret, const void* __restrict__ mask,
                                                              int mdtype, Moments* __restrict__ moments,
                                                              double* __restrict__ host_sums) {
    // in the order of the chain: slot e is the chunk's e-th token from its end
    __shared__ __attribute__((aligned(16))) float slot[kScanChunk + 64];
    __shared__ float kept[kScanChunk / kReplay];           // results of steps kReplay - 1, 2 kReplay - 1, ...
    const int64_t base = (int64_t)blockIdx.x * width;
    const int tid = (int)threadIdx.x;
    __shared__ double wave_masked[kScanBlock / 64];
    double masked = 0.0;
    Moments mom = {0.0, 0.0, 0.0};
    constexpr int kPer = kScanChunk / kScanBlock;
    float last = 0.f;                                      // result behind the chunk
    for (int64_t hi = width; hi > 0; hi -= kScanChunk) {
        const int64_t lo = hi > kScanChunk ? hi - kScanChunk : 0;
        const int n = (int)(hi - lo);
        const float* r = rewards + base + lo;
        const float* v = values + base + lo;
        // everything the chunk needs of memory is requested here, in one go; values and mask stay in registers
        float v_mine[kPer], m_mine[kPer], r_mine[kPer], v_next[kPer];
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const int t = min(q * kScanBlock + tid, n - 1);
            r_mine[q] = r[t];
            v_mine[q] = v[t];
            v_next[q] = v[lo + t + 1 < width ? t + 1 : t];
        }
        if (kMoments) {
#pragma unroll
            for (int q = 0; q < kPer; ++q)
                m_mine[q] = q * kScanBlock < n ? mask_at(mask, mdtype, nullptr, 0, 0, base + lo + min(q * kScanBlock + tid, n - 1), 0)
                                               : 0.f;
        }
        __syncthreads();                                   // the previous chunk has been written out
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const int t = q * kScanBlock + tid;
            const float next = lo + t + 1 < width ? v_next[q] : 0.f;
            if (t < n) slot[n - 1 - t] = mrl::sub_rn(mrl::add_rn(r_mine[q], mrl::mul_rn(gamma, next)), v_mine[q]);
        }
        if (kMoments && host_sums) {
            // the row's mask sum, for a caller that waits for nothing else; on its way before the chain starts
#pragma unroll
            for (int q = 0; q < kPer; ++q) masked += q * kScanBlock + tid < n ? (double)m_mine[q] : 0.0;
            double s = masked;
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
            if ((tid & 63) == 0) wave_masked[tid >> 6] = s;
        }
        __syncthreads();
        if (kMoments && host_sums && lo == 0 && tid == kScanBlock - 1) {
            double s = wave_masked[0];
            for (int w = 1; w < kScanBlock / 64; ++w) s += wave_masked[w];
            // past the caches, which would keep it until the kernel ends
            __hip_atomic_store(host_sums + blockIdx.x, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        const float behind = last;
        if (tid < 64) {
            // steps past the n-th take what lies in their slots; nobody looks at them
            const int blocks = (n + 63) >> 6;
            float d = slot[tid], x = behind;
            for (int g = 0; g < blocks; ++g) {
                const float d_next = slot[(g + 1) * 64 + tid];
#pragma unroll
                for (int e = 0; e < 64; ++e) {
                    const float delta = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(d), e));
                    x = mrl::add_rn(delta, mrl::mul_rn(gl, x));
                    if (e % kReplay == kReplay - 1) kept[(g * 64 + e) / kReplay] = x;      // the same from every lane
                }
                d = d_next;
            }
        }
        __syncthreads();
        if (tid * kReplay < n) {
            float x = tid == 0 ? behind : kept[tid - 1];
            float4* mine = reinterpret_cast<float4*>(slot + tid * kReplay);
#pragma unroll
            for (int g = 0; g < kReplay / 4; ++g) {
                float4 d = mine[g];
                d.x = x = mrl::add_rn(d.x, mrl::mul_rn(gl, x));
                d.y = x = mrl::add_rn(d.y, mrl::mul_rn(gl, x));
                d.z = x = mrl::add_rn(d.z, mrl::mul_rn(gl, x));
                d.w = x = mrl::add_rn(d.w, mrl::mul_rn(gl, x));
                mine[g] = d;
            }
        }
        last = kept[kScanChunk / kReplay - 1];             // of a whole chunk; behind another there is none
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const int t = q * kScanBlock + tid;
            if (t >= n) break;
            const float a = slot[n - 1 - t];
            adv[base + lo + t] = a;
            ret[base + lo + t] = mrl::add_rn(a, v_mine[q]);
            if (kMoments && m_mine[q] != 0.f) {
                const double m = (double)m_mine[q];
                mom.w += m;
                mom.x += m * (double)a;
                mom.xx += m * ((double)a * (double)a);
            }
        }
    }
    if (kMoments) {
        __shared__ double lds[3][kScanBlock / 64];
        const double part[3] = {mom.w, mom.x, mom.xx};
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            double s = part[q];
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
            if ((threadIdx.x & 63) == 0) lds[q][threadIdx.x >> 6] = s;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double s[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                s[q] = lds[q][0];
                for (int w = 1; w < kScanBlock / 64; ++w) s[q] += lds[q][w];
            }
            moments[blockIdx.x] = {s[0], s[1], s[2]};
        }
    }
}

// ---------------------------------------------------------------------------- masked whitening
// One workgroup: mean and (Bessel-corrected) variance over the masked entries, then
// out = (x - mean) * rsqrt(var + 1e-8) (+ mean).  Sums in fp64, the scalar arithmetic in fp32 as in
// torch.  info[0] = number of masked entries (sum of the mask).
__global__ __launch_bounds__(kReduceBlock) void masked_whiten_kernel(const float* __restrict__ x,
                                                                    const void* __restrict__ mask, int mdtype,
                                                                    int64_t n, int shift_mean,
                                                                    float* __restrict__ out,
                                                                    double* __restrict__ info) {
    __shared__ double lds[kReduceBlock / 64 + 1];
    double s = 0.0, cnt = 0.0;
    for (int64_t e = threadIdx.x; e < n; e += kReduceBlock) {
        const float m = mask_at(mask, mdtype, nullptr, 0, 0, e, 0);
        cnt += (double)m;
        if (m != 0.f) s += (double)(x[e] * m);
    }
    const double total = block_sum(s, lds);
    const double count = block_sum(cnt, lds);
    const float denom = (float)count + 1e-8f;
    const float mean = (float)total / denom;
    double q = 0.0;
    for (int64_t e = threadIdx.x; e < n; e += kReduceBlock) {
        const float m = mask_at(mask, mdtype, nullptr, 0, 0, e, 0);
        if (m != 0.f) {
            const float c = x[e] - mean;
            q += (double)((c * c) * m);
        }
    }
    const double qsum = block_sum(q, lds);
    float var = (float)qsum / denom;
    const float fc = (float)count;
    if (fc != 1.f) var = var * (fc / (fc - 1.f));
    const float scale = 1.f / sqrtf(var + 1e-8f);
    for (int64_t e = threadIdx.x; e < n; e += kReduceBlock) {
        float w = (x[e] - mean) * scale;
        if (!shift_mean) w += mean;
        out[e] = w;
    }
    if (threadIdx.x == 0) {
        info[0] = count;
        info[1] = (double)mean;
        info[2] = (double)var;
    }
}

// The same from the moments that gae_scan_kernel left, in place: every workgroup adds the rows' moments
// up in the same fixed order and whitens its share.  sum m (x - mean)^2 is expanded about the fp32 mean, in
// fp64: its cancellation error, (mean / std)^2 * 2^-52, stays below what the rounding of the mean to fp32
// already costs the two-pass form, (mean / std)^2 * 2^-50.  One launch over the chip in place of three
// passes by one workgroup (128 x 2048: 5.5 us, was 314 us).
__global__ __launch_bounds__(kReduceBlock) void whiten_moments_kernel(float* __restrict__ x,
                                                                     const Moments* __restrict__ moments,
                                                                     int64_t n_moments, int64_t n,
                                                                     double* __restrict__ info) {
    __shared__ double lds[3][kReduceBlock / 64 + 1];
    Moments mom = {0.0, 0.0, 0.0};
    for (int64_t i = threadIdx.x; i < n_moments; i += kReduceBlock) {
        const Moments o = moments[i];
        mom.w += o.w;
        mom.x += o.x;
        mom.xx += o.xx;
    }
    double sums[3] = {mom.w, mom.x, mom.xx};
    block_sum3(sums, lds);
    const double count = sums[0], total = sums[1], squares = sums[2];
    const float fc = (float)count, denom = fc + 1e-8f;
    const float mean = (float)total / denom;
    const double md = (double)mean;
    const double about = squares - md * (2.0 * total - md * count);
    float var = (float)(about < 0.0 ? 0.0 : about) / denom;           // a NaN stays one
    if (fc != 1.f) var = var * (fc / (fc - 1.f));
    const float scale = 1.f / sqrtf(var + 1e-8f);
    for (int64_t e = (int64_t)blockIdx.x * kReduceBlock + threadIdx.x; e < n; e += (int64_t)gridDim.x * kReduceBlock)
        x[e] = (x[e] - mean) * scale;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        info[0] = count;
        info[1] = md;
        info[2] = (double)var;
    }
}

// ---------------------------------------------------------------------------- clipped value loss
struct ValueTerm {
    float loss;      // max((vp - ret)^2, (clamp(vp, v - c, v + c) - ret)^2)
    float clipped;   // second operand strictly larger
    float d;         // d loss / d vp
};

__device__ __forceinline__ ValueTerm value_term(float vp, float ret, float v, float c) {
    ValueTerm t;
    const float lo = v - c, hi = v + c;
    const float vc = clampf(vp, lo, hi);
    const float e1 = vp - ret, e2 = vc - ret;
    const float l1 = e1 * e1, l2 = e2 * e2;
    t.loss = torch_max(l1, l2);
    t.clipped = l2 > l1 ? 1.f : 0.f;
    const float d1 = 2.f * e1;
    const float d2 = (vp >= lo && vp <= hi) ? 2.f * e2 : 0.f;
    if (l1 > l2) t.d = d1;
    else if (l2 > l1) t.d = d2;
    else if (l1 == l2) t.d = 0.5f * d1 + 0.5f * d2;
    else t.d = l1 + l2;      // NaN operands propagate
    return t;
}

// out[0] = loss_scale * vf_loss, out[1] = vf_loss = 0.5 * masked_mean(max(l1, l2)), out[2] =
// masked_mean(l2 > l1), out[3] = sum(mask)
// (loss_out, if given: out[0] once more, a 0-dim tensor of its own for autograd)
__device__ __forceinline__ void write_value_loss(double ssum, double csum, double count, float loss_scale,
                                                 float* __restrict__ out, float* __restrict__ loss_out,
                                                 float* __restrict__ host_out = nullptr) {
    const float denom = (float)count + 1e-8f;
    const float vf = 0.5f * ((float)ssum / denom);
    out[0] = loss_scale * vf;
    out[1] = vf;
    out[2] = (float)csum / denom;
    out[3] = (float)count;
    if (loss_out) *loss_out = loss_scale * vf;
    if (host_out) {
#pragma unroll
        for (int q = 0; q < 4; ++q) host_out[q] = out[q];
    }
}

__global__ __launch_bounds__(kReduceBlock) void value_loss_fwd_kernel(
    const float* __restrict__ vpreds, const float* __restrict__ returns, const float* __restrict__ values,
    const void* __restrict__ mask, int mdtype, const void* __restrict__ lens, int ldtype, int64_t batch,
    int64_t width, float clip, float loss_scale, float* __restrict__ out) {
    __shared__ double lds[kReduceBlock / 64 + 1];
    double s = 0.0, cf = 0.0, cnt = 0.0;
    const int64_t n = batch * width;
    for (int64_t e = threadIdx.x; e < n; e += kReduceBlock) {
        const int64_t i = e / width, j = e - i * width;
        const float m = mask_at(mask, mdtype, lens, ldtype, i, j, width);
        cnt += (double)m;
        if (m != 0.f) {
            const ValueTerm t = value_term(vpreds[e], returns[e], values[e], clip);
            s += (double)(t.loss * m);
            cf += (double)(t.clipped * m);
        }
    }
    const double ssum = block_sum(s, lds);
    const double csum = block_sum(cf, lds);
    const double count = block_sum(cnt, lds);
    if (threadIdx.x == 0) write_value_loss(ssum, csum, count, loss_scale, out, nullptr);
}

// The critic's loss reads the value head's output where it lies: with the windows cut out first and scattered
// back by the backward, five more launches and an autograd node went into 2 MB (128 x (256 + 2048) tokens: PPO
// value side 278 us a pass, now 217).  The forward leaves each token's slope, d loss / d vp, for the backward,
// which so depends neither on the head's output nor on the operands (the caller may overwrite them).
//
// Where the predicted value of token j of sample i lies: element i * width + j of [batch, width], or (kHead)
// in the value head's output [batch, padded_s] at the response window [P - 1, P + R - 1) of the sample,
// clamped to its row; tokens behind the window have the value 0 and no gradient.
struct ValuePlace {
    int64_t width, padded_s;
    const void* prompt;
    int prompt_dtype;
    const void* resp;
    int resp_dtype;
    __device__ __forceinline__ int64_t at(const void* p, int dtype, int64_t i) const {
        return dtype == MRL_I32 ? (int64_t) reinterpret_cast<const int32_t*>(p)[i]
                                : reinterpret_cast<const int64_t*>(p)[i];
    }
    __device__ __forceinline__ void window(int64_t i, int64_t& lo, int64_t& hi) const {
        const int64_t p = at(prompt, prompt_dtype, i), e = p + at(resp, resp_dtype, i) - 1;
        lo = p - 1 < 0 ? 0 : (p - 1 > padded_s ? padded_s : p - 1);
        hi = e < 0 ? 0 : (e > padded_s ? padded_s : e);
    }
};

// The same spread over the chip: one workgroup per row (rows strided beyond kLossRows of them), or per part of a
// row where few wide rows would leave the chip idle, leaves its three sums in fp64, a second launch adds them
// up in a fixed order.  128 x 2048: 11 us for both, was 167 us by one workgroup, which pays off only where no
// scratch memory is at hand.  Rows are cut into parts of up to kLossPart entries as far as there are workgroups
// (1 x 32 768, a call: 44.5 us whole, 22.9 us in 16 parts; one workgroup of 1024 threads 25.1 us).
constexpr int64_t kLossRows = 1024;             // workgroups, and partial sums
constexpr int64_t kLossPart = 2048;
struct LossSums {
    double loss, clipped, count;
};

template <bool kHead>
__global__ __launch_bounds__(256) void value_loss_rows_kernel(
    const float* __restrict__ vpreds, ValuePlace place, const float* __restrict__ returns,
    const float* __restrict__ values, const void* __restrict__ mask, int mdtype, const void* __restrict__ lens, int ldtype,
    int64_t batch, float clip, LossSums* __restrict__ sums, float* __restrict__ slope) {
    const int64_t width = place.width;
    __shared__ double part[3][256 / 64];
    double acc[3] = {0.0, 0.0, 0.0};
    const int64_t begin = width * blockIdx.y / gridDim.y, end = width * (blockIdx.y + 1) / gridDim.y;
    for (int64_t i = blockIdx.x; i < batch; i += gridDim.x) {
        int64_t lo = 0, hi = width;
        if (kHead) place.window(i, lo, hi);
        const float* row = vpreds + (kHead ? i * place.padded_s + lo : i * width);
        for (int64_t j = begin + threadIdx.x; j < end; j += 256) {
            const float m = mask_at(mask, mdtype, lens, ldtype, i, j, width);
            acc[2] += (double)m;
            if (m != 0.f) {
                const int64_t e = i * width + j;
                const ValueTerm t = value_term(j < hi - lo ? row[j] : 0.f, returns[e], values[e], clip);
                acc[0] += (double)(t.loss * m);
                acc[1] += (double)(t.clipped * m);
                if (kHead) slope[e] = t.d;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) acc[q] += __shfl_xor(acc[q], off, 64);
        if ((threadIdx.x & 63) == 0) part[q][threadIdx.x >> 6] = acc[q];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double s[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) s[q] = (part[q][0] + part[q][1]) + (part[q][2] + part[q][3]);
        sums[blockIdx.y * gridDim.x + blockIdx.x] = {s[0], s[1], s[2]};
    }
}

__global__ __launch_bounds__(kReduceBlock) void value_loss_finish_kernel(const LossSums* __restrict__ sums, int n,
                                                                        float loss_scale, float* __restrict__ out,
                                                                        float* __restrict__ loss_out,
                                                                        float* __restrict__ host_out) {
    __shared__ double lds[3][kReduceBlock / 64 + 1];
    LossSums s = {0.0, 0.0, 0.0};
    if ((int)threadIdx.x < n) s = sums[threadIdx.x];       // n <= kLossRows = kReduceBlock
    double all[3] = {s.loss, s.clipped, s.count};
    block_sum3(all, lds);
    if (threadIdx.x == 0) write_value_loss(all[0], all[1], all[2], loss_scale, out, loss_out, host_out);
}
static_assert(kLossRows == kReduceBlock, "the finishing workgroup takes one partial sum per thread");

__global__ __launch_bounds__(256) void value_loss_bwd_kernel(
    const float* __restrict__ vpreds, const float* __restrict__ returns, const float* __restrict__ values,
    const void* __restrict__ mask, int mdtype, const void* __restrict__ lens, int ldtype, int64_t batch,
    int64_t width, float clip, float loss_scale, const float* __restrict__ out, const float* __restrict__ upstream,
    float* __restrict__ g_vpreds) {
    const int64_t n = batch * width;
    const float coef = (*upstream) * loss_scale * 0.5f / (out[3] + 1e-8f);
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        const int64_t i = e / width, j = e - i * width;
        const float m = mask_at(mask, mdtype, lens, ldtype, i, j, width);
        float g = 0.f;
        if (m != 0.f) g = coef * m * value_term(vpreds[e], returns[e], values[e], clip).d;
        g_vpreds[e] = g;
    }
}

// The gradient of the whole value head output: every entry finds its token, entries outside the windows get 0.
__global__ __launch_bounds__(256) void critic_loss_bwd_kernel(
    const float* __restrict__ slope, ValuePlace place, int64_t batch, float loss_scale, const float* __restrict__ out,
    const float* __restrict__ upstream, float* __restrict__ g_head) {
    const float coef = (*upstream) * loss_scale * 0.5f / (out[3] + 1e-8f);
    const int64_t n = batch * place.padded_s;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        const int64_t i = e / place.padded_s, s = e - i * place.padded_s;
        int64_t lo, hi;
        place.window(i, lo, hi);
        const int64_t j = s - lo;
        float g = 0.f;
        if (j >= 0 && s < hi && j < place.width) {
            const float m = mask_at(nullptr, 0, place.resp, place.resp_dtype, i, j, place.width);
            if (m != 0.f) g = coef * m * slope[i * place.width + j];
        }
        g_head[e] = g;
    }
}

// Workgroups of value_loss_rows_kernel: rows by parts, at most kLossRows.
dim3 loss_grid(int64_t batch, int64_t width) {
    const int64_t rows = batch < kLossRows ? batch : kLossRows, most = rows > 0 ? kLossRows / rows : 1;
    const int64_t parts = (width + kLossPart - 1) / kLossPart;
    return dim3((unsigned)rows, (unsigned)(parts < most ? parts : most));
}

int check_mask(const char* fn, const void* mask, int mask_dtype, const void* lens, int lens_dtype) {
    MRL_REQUIRE(mask != nullptr || lens != nullptr, MRL_ERR_INVALID_ARG, "%s: neither mask nor response_length given", fn);
    if (mask != nullptr)
        MRL_REQUIRE(mrl::mask_dtype_bytes(mask_dtype) != 0, MRL_ERR_UNSUPPORTED, "%s: mask dtype %d", fn, mask_dtype);
    else
        MRL_REQUIRE(mrl::int_dtype_bytes(lens_dtype) != 0, MRL_ERR_UNSUPPORTED, "%s: response_length dtype %d", fn,
                    lens_dtype);
    return MRL_OK;
}

}  // namespace

extern "C" int mrl_kl_token_rewards(const float* old_log_prob, const float* ref_log_prob,
                                    const void* response_length, int length_dtype, const float* scores,
                                    int64_t batch, int64_t width, int kl_penalty, float beta, float* rewards,
                                    float* row_kl, void* stream) {
    const char* fn = "mrl_kl_token_rewards";
    MRL_REQUIRE(batch >= 0 && width > 0 && batch <= 0x7fffffffLL, MRL_ERR_INVALID_ARG, "%s: batch=%lld width=%lld", fn,
                (long long)batch, (long long)width);
    MRL_REQUIRE(kl_penalty >= MRL_KL_KL && kl_penalty <= MRL_KL_LOW_VAR, MRL_ERR_INVALID_ARG, "%s: kl_penalty=%d", fn,
                kl_penalty);
    MRL_REQUIRE(mrl::int_dtype_bytes(length_dtype) != 0, MRL_ERR_UNSUPPORTED, "%s: response_length dtype %d", fn,
                length_dtype);
    if (batch == 0) return MRL_OK;
    MRL_REQUIRE(old_log_prob && ref_log_prob && response_length && scores && rewards && row_kl, MRL_ERR_INVALID_ARG,
                "%s: NULL pointer", fn);
    hipLaunchKernelGGL(kl_rewards_kernel, dim3((unsigned)batch), dim3(256), 0, mrl::as_stream(stream), old_log_prob,
                       ref_log_prob, response_length, length_dtype, scores, width, kl_penalty, beta, rewards, row_kl);
    return mrl::check_launch(fn);
}

extern "C" int mrl_gae_scan(const float* rewards, const float* values, int64_t batch, int64_t width, float gamma,
                            float gamma_lam, float* advantages, float* returns, void* stream) {
    const char* fn = "mrl_gae_scan";
    MRL_REQUIRE(batch >= 0 && width > 0 && batch <= 0x7fffffffLL, MRL_ERR_INVALID_ARG, "%s: batch=%lld width=%lld", fn,
                (long long)batch, (long long)width);
    if (batch == 0) return MRL_OK;
    MRL_REQUIRE(rewards && values && advantages && returns, MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    MRL_REQUIRE(advantages != rewards && advantages != values && returns != rewards && returns != values &&
                    advantages != returns,
                MRL_ERR_INVALID_ARG, "%s: outputs must not alias the inputs or each other", fn);
    hipLaunchKernelGGL(gae_scan_kernel<false>, dim3((unsigned)batch), dim3(kScanBlock), 0, mrl::as_stream(stream),
                       rewards, values, width, gamma, gamma_lam, advantages, returns, (const void*)nullptr, 0,
                       (Moments*)nullptr, (double*)nullptr);
    return mrl::check_launch(fn);
}

extern "C" int64_t mrl_gae_whiten_workspace_bytes(int64_t batch) {
    return batch < 0 ? 0 : batch * (int64_t)sizeof(Moments);
}

extern "C" int mrl_gae_whiten(const float* rewards, const float* values, const void* mask, int mask_dtype, int64_t batch,
                              int64_t width, float gamma, float gamma_lam, float* advantages, float* returns,
                              double* info, void* workspace, int64_t workspace_bytes, void* stream) {
    return mrl_gae_whiten_host(rewards, values, mask, mask_dtype, batch, width, gamma, gamma_lam, advantages, returns, info,
                               nullptr, workspace, workspace_bytes, stream);
}

extern "C" int mrl_gae_whiten_host(const float* rewards, const float* values, const void* mask, int mask_dtype,
                                   int64_t batch, int64_t width, float gamma, float gamma_lam, float* advantages,
                                   float* returns, double* info, double* host_sums, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
    const char* fn = "mrl_gae_whiten";
    MRL_REQUIRE(batch >= 0 && width > 0 && batch <= 0x7fffffffLL, MRL_ERR_INVALID_ARG, "%s: batch=%lld width=%lld", fn,
                (long long)batch, (long long)width);
    MRL_REQUIRE(mrl::mask_dtype_bytes(mask_dtype) != 0, MRL_ERR_UNSUPPORTED, "%s: mask dtype %d", fn, mask_dtype);
    MRL_REQUIRE(info != nullptr, MRL_ERR_INVALID_ARG, "%s: info is NULL", fn);
    MRL_REQUIRE(batch == 0 || (rewards && values && mask && advantages && returns && workspace), MRL_ERR_INVALID_ARG,
                "%s: NULL pointer", fn);
    MRL_REQUIRE(mrl::aligned(workspace, 8) && mrl::aligned(info, 8) && mrl::aligned(host_sums, 8), MRL_ERR_MISALIGNED,
                "%s: workspace, info and host_sums must be 8-byte aligned", fn);
    MRL_REQUIRE(workspace_bytes >= mrl_gae_whiten_workspace_bytes(batch), MRL_ERR_INVALID_ARG,
                "%s: workspace of %lld bytes, need %lld", fn, (long long)workspace_bytes,
                (long long)mrl_gae_whiten_workspace_bytes(batch));
    MRL_REQUIRE(batch == 0 || (advantages != rewards && advantages != values && returns != rewards && returns != values &&
                               advantages != returns),
                MRL_ERR_INVALID_ARG, "%s: outputs must not alias the inputs or each other", fn);
    hipStream_t s = mrl::as_stream(stream);
    Moments* moments = reinterpret_cast<Moments*>(workspace);
    if (batch > 0) {
        hipLaunchKernelGGL(gae_scan_kernel<true>, dim3((unsigned)batch), dim3(kScanBlock), 0, s, rewards, values, width,
                           gamma, gamma_lam, advantages, returns, mask, mask_dtype, moments, host_sums);
        const int rc = mrl::check_launch(fn);
        if (rc != MRL_OK) return rc;
    }
    // one entry per thread up to a workgroup per CU; every workgroup reads all moments
    const int64_t n = batch * width, want = (n + kReduceBlock - 1) / kReduceBlock;
    hipLaunchKernelGGL(whiten_moments_kernel, dim3((unsigned)(want < 1 ? 1 : (want < 256 ? want : 256))),
                       dim3(kReduceBlock), 0, s, advantages, (const Moments*)moments, batch, n, info);
    return mrl::check_launch(fn);
}

extern "C" int mrl_masked_whiten(const float* x, const void* mask, int mask_dtype, int64_t n, int shift_mean,
                                 float* out, double* info, void* stream) {
    const char* fn = "mrl_masked_whiten";
    MRL_REQUIRE(n >= 0, MRL_ERR_INVALID_ARG, "%s: n=%lld", fn, (long long)n);
    MRL_REQUIRE(mrl::mask_dtype_bytes(mask_dtype) != 0, MRL_ERR_UNSUPPORTED, "%s: mask dtype %d", fn, mask_dtype);
    MRL_REQUIRE(info != nullptr, MRL_ERR_INVALID_ARG, "%s: info is NULL", fn);
    MRL_REQUIRE(n == 0 || (x && mask && out), MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    hipLaunchKernelGGL(masked_whiten_kernel, dim3(1), dim3(kReduceBlock), 0, mrl::as_stream(stream), x, mask, mask_dtype,
                       n, shift_mean, out, info);
    return mrl::check_launch(fn);
}

extern "C" int mrl_value_loss_fwd(const float* vpreds, const float* returns, const float* values, const void* mask,
                                  int mask_dtype, const void* response_length, int length_dtype, int64_t batch,
                                  int64_t width, float cliprange_value, float loss_scale, float* out, void* stream) {
    const char* fn = "mrl_value_loss_fwd";
    MRL_REQUIRE(batch >= 0 && width > 0, MRL_ERR_INVALID_ARG, "%s: batch=%lld width=%lld", fn, (long long)batch,
                (long long)width);
    int rc = check_mask(fn, mask, mask_dtype, response_length, length_dtype);
    if (rc != MRL_OK) return rc;
    MRL_REQUIRE(out != nullptr && (batch == 0 || (vpreds && returns && values)), MRL_ERR_INVALID_ARG, "%s: NULL pointer",
                fn);
    hipLaunchKernelGGL(value_loss_fwd_kernel, dim3(1), dim3(kReduceBlock), 0, mrl::as_stream(stream), vpreds, returns,
                       values, mask, mask_dtype, response_length, length_dtype, batch, width, cliprange_value, loss_scale,
                       out);
    return mrl::check_launch(fn);
}

extern "C" int64_t mrl_value_loss_workspace_bytes(int64_t batch) {
    return batch <= 0 ? 0 : kLossRows * (int64_t)sizeof(LossSums);
}

extern "C" int mrl_value_loss_fwd_split(const float* vpreds, const float* returns, const float* values, const void* mask,
                                        int mask_dtype, const void* response_length, int length_dtype, int64_t batch,
                                        int64_t width, float cliprange_value, float loss_scale, float* out,
                                        float* loss_out, void* workspace, int64_t workspace_bytes, void* stream) {
    const char* fn = "mrl_value_loss_fwd_split";
    MRL_REQUIRE(batch >= 0 && width > 0, MRL_ERR_INVALID_ARG, "%s: batch=%lld width=%lld", fn, (long long)batch,
                (long long)width);
    int rc = check_mask(fn, mask, mask_dtype, response_length, length_dtype);
    if (rc != MRL_OK) return rc;
    MRL_REQUIRE(out != nullptr && (batch == 0 || (vpreds && returns && values && workspace)), MRL_ERR_INVALID_ARG,
                "%s: NULL pointer", fn);
    MRL_REQUIRE(mrl::aligned(workspace, 8), MRL_ERR_MISALIGNED, "%s: workspace must be 8-byte aligned", fn);
    MRL_REQUIRE(workspace_bytes >= mrl_value_loss_workspace_bytes(batch), MRL_ERR_INVALID_ARG,
                "%s: workspace of %lld bytes, need %lld", fn, (long long)workspace_bytes,
                (long long)mrl_value_loss_workspace_bytes(batch));
    hipStream_t s = mrl::as_stream(stream);
    LossSums* sums = reinterpret_cast<LossSums*>(workspace);
    const dim3 grid = loss_grid(batch, width);
    if (grid.x > 0) {
        const ValuePlace place = {width, 0, nullptr, 0, nullptr, 0};
        hipLaunchKernelGGL(value_loss_rows_kernel<false>, grid, dim3(256), 0, s, vpreds, place, returns,
                           values, mask, mask_dtype, response_length, length_dtype, batch, cliprange_value, sums,
                           (float*)nullptr);
        rc = mrl::check_launch(fn);
        if (rc != MRL_OK) return rc;
    }
    hipLaunchKernelGGL(value_loss_finish_kernel, dim3(1), dim3(kReduceBlock), 0, s, (const LossSums*)sums,
                       (int)(grid.x * grid.y), loss_scale, out, loss_out, (float*)nullptr);
    return mrl::check_launch(fn);
}

static int check_critic(const char* fn, int64_t batch, int64_t padded_s, int64_t width, int prompt_dtype, int response_dtype) {
    MRL_REQUIRE(batch >= 0 && padded_s >= 0 && width > 0, MRL_ERR_INVALID_ARG, "%s: batch=%lld padded_s=%lld width=%lld", fn,
                (long long)batch, (long long)padded_s, (long long)width);
    MRL_REQUIRE(mrl::int_dtype_bytes(prompt_dtype) != 0 && mrl::int_dtype_bytes(response_dtype) != 0, MRL_ERR_UNSUPPORTED,
                "%s: length dtypes %d and %d (want I32 or I64)", fn, prompt_dtype, response_dtype);
    return MRL_OK;
}

extern "C" int mrl_critic_loss_fwd_slope(const float* head, int64_t batch, int64_t padded_s, const void* prompt_length,
                                         int prompt_dtype, const void* response_length, int response_dtype,
                                         const float* returns, const float* values, int64_t width,
                                         float cliprange_value, float loss_scale, float* slope, float* out,
                                         float* loss_out, void* workspace, int64_t workspace_bytes, void* stream) {
    return mrl_critic_loss_fwd_slope_host(head, batch, padded_s, prompt_length, prompt_dtype, response_length, response_dtype,
                                          returns, values, width, cliprange_value, loss_scale, slope, out, loss_out,
                                          nullptr, workspace, workspace_bytes, stream);
}

extern "C" int mrl_critic_loss_fwd_slope_host(const float* head, int64_t batch, int64_t padded_s, const void* prompt_length,
                                              int prompt_dtype, const void* response_length, int response_dtype,
                                              const float* returns, const float* values, int64_t width,
                                              float cliprange_value, float loss_scale, float* slope, float* out,
                                              float* loss_out, float* host_out, void* workspace,
                                              int64_t workspace_bytes, void* stream) {
    const char* fn = "mrl_critic_loss_fwd_slope";
    int rc = check_critic(fn, batch, padded_s, width, prompt_dtype, response_dtype);
    if (rc != MRL_OK) return rc;
    MRL_REQUIRE(out != nullptr && (batch == 0 || ((head || padded_s == 0) && prompt_length && response_length && returns &&
                                                  values && slope && workspace)),
                MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    MRL_REQUIRE(mrl::aligned(workspace, 8) && mrl::aligned(host_out, 4), MRL_ERR_MISALIGNED,
                "%s: workspace must be 8-byte and host_out 4-byte aligned", fn);
    MRL_REQUIRE(workspace_bytes >= mrl_value_loss_workspace_bytes(batch), MRL_ERR_INVALID_ARG,
                "%s: workspace of %lld bytes, need %lld", fn, (long long)workspace_bytes,
                (long long)mrl_value_loss_workspace_bytes(batch));
    hipStream_t s = mrl::as_stream(stream);
    LossSums* sums = reinterpret_cast<LossSums*>(workspace);
    const dim3 grid = loss_grid(batch, width);
    if (grid.x > 0) {
        const ValuePlace place = {width, padded_s, prompt_length, prompt_dtype, response_length, response_dtype};
        hipLaunchKernelGGL(value_loss_rows_kernel<true>, grid, dim3(256), 0, s, head, place, returns, values,
                           (const void*)nullptr, 0, response_length, response_dtype, batch, cliprange_value, sums, slope);
        rc = mrl::check_launch(fn);
        if (rc != MRL_OK) return rc;
    }
    hipLaunchKernelGGL(value_loss_finish_kernel, dim3(1), dim3(kReduceBlock), 0, s, (const LossSums*)sums,
                       (int)(grid.x * grid.y), loss_scale, out, loss_out, host_out);
    return mrl::check_launch(fn);
}

extern "C" int mrl_critic_loss_bwd_slope(const float* slope, int64_t batch, int64_t padded_s,
                                         const void* prompt_length, int prompt_dtype, const void* response_length,
                                         int response_dtype, int64_t width, float loss_scale, const float* out,
                                         const float* upstream, float* g_head, void* stream) {
    const char* fn = "mrl_critic_loss_bwd_slope";
    int rc = check_critic(fn, batch, padded_s, width, prompt_dtype, response_dtype);
    if (rc != MRL_OK || batch * padded_s == 0) return rc;
    MRL_REQUIRE(slope && prompt_length && response_length && out && upstream && g_head, MRL_ERR_INVALID_ARG,
                "%s: NULL pointer", fn);
    const ValuePlace place = {width, padded_s, prompt_length, prompt_dtype, response_length, response_dtype};
    const int64_t n = batch * padded_s;
    const unsigned grid = (unsigned)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096);
    hipLaunchKernelGGL(critic_loss_bwd_kernel, dim3(grid), dim3(256), 0, mrl::as_stream(stream), slope, place, batch, loss_scale,
                       out, upstream, g_head);
    return mrl::check_launch(fn);
}

extern "C" int mrl_value_loss_bwd(const float* vpreds, const float* returns, const float* values, const void* mask,
                                  int mask_dtype, const void* response_length, int length_dtype, int64_t batch,
                                  int64_t width, float cliprange_value, float loss_scale, const float* out,
                                  const float* upstream, float* g_vpreds, void* stream) {
    const char* fn = "mrl_value_loss_bwd";
    MRL_REQUIRE(batch >= 0 && width > 0, MRL_ERR_INVALID_ARG, "%s: batch=%lld width=%lld", fn, (long long)batch,
                (long long)width);
    int rc = check_mask(fn, mask, mask_dtype, response_length, length_dtype);
    if (rc != MRL_OK) return rc;
    if (batch == 0) return MRL_OK;
    MRL_REQUIRE(vpreds && returns && values && out && upstream && g_vpreds, MRL_ERR_INVALID_ARG, "%s: NULL pointer", fn);
    const int64_t n = batch * width;
    const unsigned grid = (unsigned)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096);
    hipLaunchKernelGGL(value_loss_bwd_kernel, dim3(grid), dim3(256), 0, mrl::as_stream(stream), vpreds, returns, values,
                       mask, mask_dtype, response_length, length_dtype, batch, width, cliprange_value, loss_scale, out,
                       upstream, g_vpreds);
    return mrl::check_launch(fn);
}
