// Row-wise selection on a score matrix [B, I] -> union-over-rows byte mask.
//
//   top-k        per row the k largest scores are active (equal scores: lower index first)
//                SkipDecoderLayer._compute_binary_mask, src/modeling_skip.py:208-211
//   statistical  per row: score > mean + std_pop * z, population std, strict >
//                _gaussian_topk, src/modeling_skip.py:197-202
//   union        any(dim=0), src/modeling_skip.py:214
//   sketch       approx_topk_threshold, sparse_transformers/csrc/approx_topk.h:10-88
//
// One block per row.  The row is read from HBM once; every thread keeps its scores in registers (rows of up
// to 16384 scores) as order-preserving 32-bit keys.  The k-th largest key is found exactly, with nothing sorted, by a radix
// select (10-bit digits, longer rows 8-bit ones, most significant first, one LDS histogram per digit; once at most 64 keys
// share the prefix they are ranked directly).  With several
// rows every block leaves its row mask in the workspace and the block that finishes last ORs them together; which block that
// is does not change the result.  A caller with a mask of zeros has the blocks set their rows' bytes in it instead.
#include "st_common.h"

namespace st {

constexpr int kSelThreads = 1024;
constexpr int kSelWaves = kSelThreads / kWave;
constexpr int kSelMaxLdsKeys = 36 * 1024;  // 144 KB of keys next to the small shared struct

// float -> unsigned key with the same order (-0 and +0 share one key, as they compare equal)
__device__ __forceinline__ uint32_t order_key(float v)
{
    uint32_t u = __float_as_uint(v);
    if (u == 0x80000000u) u = 0u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k)
{
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

constexpr int kHistCopies = 8;  // a digit's counter exists once per lane % 8: equal digits in a wave spread over banks

// of key_select_desc: digits, counters of each, and counters from one digit's first to its second (equal digits on other banks)
constexpr int kKeyDigits = 1024, kKeyCopies = 8, kKeyPitch = kKeyDigits + kWave / kKeyCopies;
constexpr size_t kKeyHistBytes = (size_t)kKeyPitch * kKeyCopies * 4;

struct SelShared {
    uint32_t hist[256 * kHistCopies];
    uint32_t hsum[256];
    uint32_t cand[kWave];
    uint32_t digit, rem, cnt, ncand;
    int wave_tot[kSelWaves];
    double wave_sum[2][kSelWaves];
    int last;
};

// k-th largest (1 <= k <= number of keys) of the block's keys.  `sweep(fn)` calls fn(key) for every key
// this thread owns.  Returns the key; `rem` = how many of the keys equal to it belong to the k largest
// (1..cnt), `cnt` = how many keys equal it.  Every thread of the block calls.
template <typename Sweep>
__device__ __forceinline__ uint32_t radix_select_desc(Sweep sweep, uint32_t k, SelShared &sh, int tid,
                                                      uint32_t &rem_out, uint32_t &cnt_out)
{
    const int copy = tid & (kHistCopies - 1);
    uint32_t prefix = 0u, pmask = 0u, rem = k, cnt = 0u;
    for (int shift = 24; shift >= 0; shift -= 8) {
        sh.hist[tid] = 0u;
        sh.hist[tid + kSelThreads] = 0u;
        static_assert(256 * kHistCopies == 2 * kSelThreads, "two counters per thread");
        __syncthreads();
        sweep([&](uint32_t kv) {
            if ((kv & pmask) == prefix) atomicAdd(&sh.hist[((kv >> shift) & 255u) * kHistCopies + copy], 1u);
        });
        __syncthreads();
        if (tid < 256) {
            uint32_t t = 0u;
#pragma unroll
            for (int c = 0; c < kHistCopies; ++c) t += sh.hist[tid * kHistCopies + c];
            sh.hsum[tid] = t;
        }
        __syncthreads();
        if (tid < kWave) {  // lane l owns digits 4l .. 4l+3; find the digit that holds the rem-th largest
            uint32_t h[4], local = 0u;
#pragma unroll
            for (int j = 0; j < 4; ++j) { h[j] = sh.hsum[4 * tid + j]; local += h[j]; }
            uint32_t incl = local;  // sum over lanes >= this one
#pragma unroll
            for (int off = 1; off < kWave; off <<= 1) {
                const uint32_t t = __shfl_down(incl, off, kWave);
                if (tid + off < kWave) incl += t;
            }
            uint32_t above = incl - local;  // keys whose digit is larger than 4l+3
#pragma unroll
            for (int j = 3; j >= 0; --j) {
                if (above < rem && rem <= above + h[j]) {
                    sh.digit = (uint32_t)(4 * tid + j);
                    sh.rem = rem - above;
                    sh.cnt = h[j];
                }
                above += h[j];
            }
        }
        __syncthreads();
        prefix |= sh.digit << shift;
        pmask |= 255u << shift;
        rem = sh.rem;
        cnt = sh.cnt;
        if (shift > 0 && cnt <= (uint32_t)kWave) {
            // Few keys are left under this prefix: list them and let one wave rank them directly instead
            // of spending a full pass on each remaining digit.  (cnt is uniform over the block.)
            if (tid == 0) sh.ncand = 0u;
            __syncthreads();
            sweep([&](uint32_t kv) {
                if ((kv & pmask) == prefix) sh.cand[atomicAdd(&sh.ncand, 1u)] = kv;
            });
            __syncthreads();
            if (tid < kWave) {
                const uint32_t mine = (uint32_t)tid < cnt ? sh.cand[tid] : 0u;
                uint32_t greater = 0u, equal = 0u;
                for (uint32_t j = 0; j < cnt; ++j) {
                    const uint32_t c = sh.cand[j];
                    greater += c > mine;
                    equal += c == mine;
                }
                if ((uint32_t)tid < cnt && greater < rem && rem <= greater + equal) {  // lanes that agree write the same
                    sh.digit = mine;
                    sh.rem = rem - greater;
                    sh.cnt = equal;
                }
            }
            __syncthreads();
            rem_out = sh.rem;
            cnt_out = sh.cnt;
            return sh.digit;
        }
    }
    rem_out = rem;
    cnt_out = cnt;
    return prefix;
}

template <int CTRL> __device__ __forceinline__ uint32_t dpp_u32(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}
// sum over the lanes below and this one (DPP row shifts, the row totals through scalar registers)
__device__ __forceinline__ int wave_incl_sum(int v, int lane)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1, zeros from outside the row
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    const int t0 = __builtin_amdgcn_readlane(v, 15), t1 = __builtin_amdgcn_readlane(v, 31), t2 = __builtin_amdgcn_readlane(v, 47);
    const int row = lane >> 4;
    return v + (row >= 1 ? t0 : 0) + (row >= 2 ? t1 : 0) + (row >= 3 ? t2 : 0);
}

// The same for a row that every thread holds KPT keys of (index tid + 1024 u < I), by digits of 10 bits: the first is sign,
// exponent and one bit of the mantissa, and a second one mostly leaves few enough to rank, which every wave does for itself.
// What bounds it is the chain of barriers (eight; eleven with 8-bit digits, a sum of the counters by some waves and a ranking
// by one) and, where many keys share a digit, the counters' addresses: lanes that share one take turns.  Top-k, 30 % of a row,
// replayed, us, 8-bit digits / so: normal scores, 8192 6.80 / 6.40, 14336 9.28 / 8.24, four rows of 8192 8.80 / 8.41; of 14336, log-normal
// 9.13 / 8.16, one score of 1e4 among normal ones 9.27 / 8.20, half of them zero 9.33 / 8.96, 60 % filled with -1e4 9.21 / 9.14.
// Built and taken back: 2048 equal intervals of value between the row's ends, one histogram, the digits where more than 64
// scores share the interval: normal 8192 5.50, 14336 8.64, but 14336 log-normal 18.6, one score of 1e4 20.2, of 30 12.2.  11-bit
// digits of four counters each: normal 6.02 / 8.07, 60 % filled 10.1.
template <int KPT>
__device__ __forceinline__ uint32_t key_select_desc(const uint32_t (&key)[KPT], int I, uint32_t k, uint32_t *hist, SelShared &sh,
                                                    int tid, uint32_t &rem_out, uint32_t &cnt_out)
{
    static_assert(kKeyDigits == kSelThreads, "one digit per thread");
    const int lane = tid & (kWave - 1), wave = tid >> 6, mine_at = (tid & (kKeyCopies - 1)) * kKeyPitch;
    auto own = [&](int c) __attribute__((always_inline)) -> uint32_t & { return hist[c * kKeyPitch + tid]; };
#pragma unroll
    for (int c = 0; c < kKeyCopies; ++c) own(c) = 0u;
    if (tid == 0) sh.ncand = 0u;
    __syncthreads();
    uint32_t prefix = 0u, pmask = 0u, rem = k, cnt = (uint32_t)I;
#pragma unroll 1
    for (int shift = 22;; shift = shift > 10 ? shift - 10 : 0) {
        const uint32_t digits = shift ? kKeyDigits - 1 : 3u;
#pragma unroll
        for (int u = 0; u < KPT; ++u)
            if (tid + u * kSelThreads < I && (key[u] & pmask) == prefix) atomicAdd(&hist[((key[u] >> shift) & digits) + mine_at], 1u);
        __syncthreads();
        uint32_t mine = 0u;
#pragma unroll
        for (int c = 0; c < kKeyCopies; ++c) mine += own(c);
#pragma unroll
        for (int c = 0; c < kKeyCopies; ++c) own(c) = 0u;
        const int incl = wave_incl_sum((int)mine, lane);
        if (lane == kWave - 1) sh.wave_tot[wave] = incl;
        __syncthreads();
        int upto = incl;   // keys with this thread's digit and the lower ones
#pragma unroll
        for (int w = 0; w < kSelWaves; ++w) upto += w < wave ? sh.wave_tot[w] : 0;
        const uint32_t above = cnt - (uint32_t)upto;
        if (above < rem && rem <= above + mine) { sh.digit = (uint32_t)tid; sh.rem = rem - above; sh.cnt = mine; }
        __syncthreads();
        prefix |= sh.digit << shift;
        pmask |= digits << shift;
        rem = sh.rem;
        cnt = (uint32_t)__builtin_amdgcn_readfirstlane((int)sh.cnt);
        if (shift == 0) {
            rem_out = rem;
            cnt_out = cnt;
            return prefix;
        }
        if (cnt <= (uint32_t)kWave) break;
    }
#pragma unroll
    for (int u = 0; u < KPT; ++u)
        if (tid + u * kSelThreads < I && (key[u] & pmask) == prefix) sh.cand[atomicAdd(&sh.ncand, 1u)] = key[u];
    __syncthreads();
    const uint32_t mine = (uint32_t)lane < cnt ? sh.cand[lane] : 0u;
    uint32_t greater = 0u, equal = 0u;
    for (uint32_t j = 0; j < cnt; ++j) {
        const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)j);
        greater += c > mine;
        equal += c == mine;
    }
    const uint64_t is = __builtin_amdgcn_ballot_w64((uint32_t)lane < cnt && greater < rem && rem <= greater + equal);
    const int l = __builtin_ctzll(is);   // (lanes that agree hold the same)
    rem_out = rem - (uint32_t)__builtin_amdgcn_readlane((int)greater, l);
    cnt_out = (uint32_t)__builtin_amdgcn_readlane((int)equal, l);
    return (uint32_t)__builtin_amdgcn_readlane((int)mine, l);
}

template <int CTRL> __device__ __forceinline__ double dpp_add_f64(double v)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint64_t o = (uint64_t)dpp_u32<CTRL>((uint32_t)b) | (uint64_t)dpp_u32<CTRL>((uint32_t)(b >> 32)) << 32;
    return v + __builtin_bit_cast(double, o);
}
__device__ __forceinline__ double wave_sum_f64(double v)
{
    v = dpp_add_f64<0xB1>(v);
    v = dpp_add_f64<0x4E>(v);
    v = dpp_add_f64<0x141>(v);
    v = dpp_add_f64<0x140>(v);
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    auto row = [&](int l) __attribute__((always_inline)) {
        const uint64_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l), h = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
        return __builtin_bit_cast(double, lo | h << 32);
    };
    return (row(0) + row(16)) + (row(32) + row(48));
}

__device__ __forceinline__ double block_sum(double v, SelShared &sh, int tid)
{
    v = wave_sum_f64(v);
    __syncthreads();  // the previous reader of wave_sum is done
    if ((tid & (kWave - 1)) == 0) sh.wave_sum[0][tid >> 6] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kSelWaves; ++w) s += sh.wave_sum[0][w];
    return s;
}

// Both sums over the block, in every thread (once per kernel).
__device__ __forceinline__ void block_sums(double &s, double &q, SelShared &sh, int tid)
{
    s = wave_sum_f64(s);
    q = wave_sum_f64(q);
    if ((tid & (kWave - 1)) == 0) { sh.wave_sum[0][tid >> 6] = s; sh.wave_sum[1][tid >> 6] = q; }
    __syncthreads();
    s = q = 0.0;
#pragma unroll
    for (int w = 0; w < kSelWaves; ++w) { s += sh.wave_sum[0][w]; q += sh.wave_sum[1][w]; }
}

// Exclusive prefix of one int per thread, threads in order.
__device__ __forceinline__ int block_excl_count(int v, SelShared &sh, int tid)
{
    const int lane = tid & (kWave - 1), wave = tid >> 6;
    int incl = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int t = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += t;
    }
    if (lane == kWave - 1) sh.wave_tot[wave] = incl;
    __syncthreads();
    int base = 0;
    for (int w = 0; w < wave; ++w) base += sh.wave_tot[w];
    return base + incl - v;
}

// KPT > 0: the row has at most KPT * 1024 scores and every thread keeps its KPT of them (index
// tid + u * 1024) in registers for all passes; a copy of the keys in LDS serves the one step that walks the
// row in index order.  KPT == 0: rows of any length, every pass reads the keys from LDS (`in_lds`) or the
// scores again from memory.
// `into`: the mask holds zeros and the rows' blocks only set what they select, so that nothing is left to unite.  Predictor and
// selection, replayed, the blocks' row masks united by the last one (and by 8-bit digits) / so: top-k, four rows of 8192 15.1 / 12.8
// us, sixteen of 14336 24.2 / 19.4; statistical 12.5 / 10.4 and 19.9 / 16.0.
template <int KPT, int METHOD>
__global__ __launch_bounds__(kSelThreads) void mask_select_kernel(const float *__restrict__ scores,
                                                                  uint8_t *__restrict__ mask,
                                                                  uint8_t *__restrict__ rowmask,
                                                                  float *__restrict__ cutoff,
                                                                  unsigned int *__restrict__ ticket, int B, int I,
                                                                  int ldm, int flags, long k_in, float z)
{
    // (pointers and sizes first: the first 14 dwords of the arguments are in scalar registers when the wave starts)
    const bool in_lds = (flags & 1) != 0, into = (flags & 2) != 0;
    constexpr int NR = KPT > 0 ? KPT : 1;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ SelShared sh;
    uint32_t *keys = reinterpret_cast<uint32_t *>(smem);
    const int tid = threadIdx.x, b = blockIdx.x;
    const float *row = scores + (size_t)b * I;
    uint8_t *dst = B == 1 || into ? mask : rowmask + (size_t)b * ldm;
    auto put = [&](int i, bool on) __attribute__((always_inline)) {
        if (!into) dst[i] = on ? 1 : 0;
        else if (on) dst[i] = 1;
    };

    float v[NR];
    if constexpr (KPT > 0) {  // all loads of the row are in flight together
#pragma unroll
        for (int u = 0; u < KPT; ++u) {
            const int i = tid + u * kSelThreads;
            v[u] = row[i < I ? i : I - 1];
        }
    }
    // fn(index, score) for every score of this thread
    auto each = [&](auto &&fn) __attribute__((always_inline)) {
        if constexpr (KPT > 0) {
#pragma unroll
            for (int u = 0; u < KPT; ++u)
                if (tid + u * kSelThreads < I) fn(tid + u * kSelThreads, v[u]);
        } else {
            for (int i = tid; i < I; i += kSelThreads)
                fn(i, in_lds && METHOD == ST_MASK_TOPK ? key_value(keys[i]) : row[i]);
        }
    };

    if constexpr (METHOD == ST_MASK_TOPK) {
        const uint32_t k = k_in < 0 ? 0u : (k_in > I ? (uint32_t)I : (uint32_t)k_in);
        if (k == 0u || k == (uint32_t)I) {  // nothing / everything (uniform over the block)
            each([&](int i, float) { put(i, k != 0u); });
        } else {
            if (KPT == 0 && in_lds)
                for (int i = tid; i < I; i += kSelThreads) keys[i] = order_key(row[i]);
            auto sweep = [&](auto &&fn) __attribute__((always_inline)) {
                each([&](int, float f) { fn(order_key(f)); });
            };
            uint32_t rem = 0u, cnt = 0u, kth = 0u;
            if constexpr (KPT > 0) {
                uint32_t key[KPT];
#pragma unroll
                for (int u = 0; u < KPT; ++u) key[u] = order_key(v[u]);
                kth = key_select_desc<KPT>(key, I, k, keys, sh, tid, rem, cnt);
            } else {
                kth = radix_select_desc(sweep, k, sh, tid, rem, cnt);
            }
            if (cutoff && tid == 0) cutoff[b] = key_value(kth);
            if (rem == cnt) {  // every score equal to the k-th belongs to the k largest
                each([&](int i, float f) { put(i, order_key(f) >= kth); });
            } else {
                // only the first `rem` of the equal scores, by index: threads take contiguous index ranges
                if constexpr (KPT > 0) {
                    each([&](int i, float f) { keys[i] = order_key(f); });
                    __syncthreads();
                }
                auto key = [&](int i) { return (KPT > 0 || in_lds) ? keys[i] : order_key(row[i]); };
                const int per = (I + kSelThreads - 1) / kSelThreads;
                const int i0 = tid * per < I ? tid * per : I, i1 = i0 + per < I ? i0 + per : I;
                int eq = 0;
                for (int i = i0; i < i1; ++i) eq += key(i) == kth;
                int seen = block_excl_count(eq, sh, tid);
                for (int i = i0; i < i1; ++i) {
                    const uint32_t kv = key(i);
                    bool on = kv > kth;
                    if (kv == kth) { on = (uint32_t)seen < rem; ++seen; }
                    put(i, on);
                }
            }
        }
    } else {
        // sums of the scores' distances from the row's first one, and of their squares, in one sweep.  Where that score lies more
        // than eight deviations out the differences below cancel (by up to I); such rows are summed again, plainly
        const double first = (double)row[0];
        double s = 0.0, q = 0.0;
        each([&](int, float f) { const double d = (double)f - first; s += d; q += d * d; });
        block_sums(s, q, sh, tid);
        const double off = s / (double)I;
        double mean = first + off, var = q / (double)I - off * off;
        if (off * off > 64.0 * var) {   // (uniform: every thread has the same sums)
            s = q = 0.0;
            for (int i = tid; i < I; i += kSelThreads) s += (double)row[i];
            mean = block_sum(s, sh, tid) / (double)I;
            for (int i = tid; i < I; i += kSelThreads) { const double d = (double)row[i] - mean; q += d * d; }
            var = block_sum(q, sh, tid) / (double)I;
        }
        const float cut = (float)mean + (float)sqrt(var) * z;
        if (cutoff && tid == 0) cutoff[b] = cut;
        each([&](int i, float f) { put(i, f > cut); });
    }
    if (B == 1 || into) return;

    // ---- union over rows by the block that finishes last
    for (int i = I + tid; i < ldm; i += kSelThreads) dst[i] = 0;  // padding of the row
    __syncthreads();
    if (tid == 0) {  // one release / acquire per block: the barriers on either side extend it to every thread
        __threadfence();
        sh.last = atomicAdd(ticket, 1u) == (unsigned int)(B - 1);
        __threadfence();
    }
    __syncthreads();
    if (!sh.last) return;
    const bool aligned = (reinterpret_cast<uintptr_t>(mask) & 15) == 0;
    for (int c = tid; c * 16 < I; c += kSelThreads) {
        uint4 acc = make_uint4(0u, 0u, 0u, 0u);
        for (int r0 = 0; r0 < B; r0 += 8) {
            uint4 w[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) w[u] = ld16(rowmask + (size_t)(r0 + u < B ? r0 + u : B - 1) * ldm + c * 16);
#pragma unroll
            for (int u = 0; u < 8; ++u) { acc.x |= w[u].x; acc.y |= w[u].y; acc.z |= w[u].z; acc.w |= w[u].w; }
        }
        if (aligned && c * 16 + 16 <= I) {
            st16(mask + c * 16, acc);
        } else {
            const uint32_t w[4] = {acc.x, acc.y, acc.z, acc.w};
            for (int e = 0; e < 16 && c * 16 + e < I; ++e) mask[c * 16 + e] = (uint8_t)((w[e >> 2] >> (8 * (e & 3))) & 0xffu);
        }
    }
    if (tid == 0) *ticket = 0u;  // ready for the next call
}

// approx_topk_threshold: four max-sketches of width W per row; cell (s, p) holds the largest score of the
// features f with (s*F + f) % W == p (the reference hashes with std::hash<int64_t>, the identity).  The
// threshold is the sketch_k-th largest cell times 0.9, sketch_k = max(1, k * cells / F).
__global__ __launch_bounds__(kSelThreads) void approx_topk_kernel(const float *__restrict__ scores, int F, long k,
                                                                 int W, float *__restrict__ threshold)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ SelShared sh;
    uint32_t *cell = reinterpret_cast<uint32_t *>(smem);  // [4][W], W <= 1024
    const int tid = threadIdx.x, b = blockIdx.x;
    const float *row = scores + (size_t)b * F;
    const uint32_t kNegInf = order_key(-__builtin_inff());
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (tid + u * kSelThreads < 4 * W) cell[tid + u * kSelThreads] = kNegInf;
    __syncthreads();
    // position of feature f in sketch s: (s*F + f) % W = (off[s] + f % W) % W, with f % W advanced by
    // 1024 % W per iteration instead of a division per feature
    int off[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) off[s] = (int)(((long)s * F) % W);
    const int step = kSelThreads % W;
    int p = tid % W;
    for (int f0 = tid; f0 < F; f0 += 8 * kSelThreads) {
        float fv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int f = f0 + u * kSelThreads;
            fv[u] = row[f < F ? f : F - 1];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (f0 + u * kSelThreads < F) {
                const uint32_t kv = order_key(fv[u]);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    int q = p + off[s];
                    if (q >= W) q -= W;
                    atomicMax(&cell[s * W + q], kv);
                }
            }
            p += step;
            if (p >= W) p -= W;
        }
    }
    __syncthreads();
    uint32_t kr[4];
    int filled = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = tid + u * kSelThreads;
        kr[u] = i < 4 * W ? cell[i] : kNegInf;
        filled += kr[u] != kNegInf;
    }
    const long cells = (long)(block_sum((double)filled, sh, tid) + 0.5);
    if (cells == 0) {
        if (tid == 0) threshold[b] = 0.f;
        return;
    }
    long sk = k * cells / F;
    if (sk < 1) sk = 1;
    if (sk > cells) sk = cells;
    uint32_t rem, cnt;
    auto sweep = [&](auto &&fn) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (tid + u * kSelThreads < 4 * W) fn(kr[u]);
    };
    const uint32_t kth = radix_select_desc(sweep, (uint32_t)sk, sh, tid, rem, cnt);
    if (tid == 0) threshold[b] = key_value(kth) * 0.9f;
}

// The same for double scores (the reference dispatches on every floating type, approx_topk.h:33).  Cells are 64-bit
// order-preserving keys; the k-th largest is found by the 32-bit radix select twice: on the upper halves, then --
// among the keys that share the winning upper half -- on the lower halves.
__device__ __forceinline__ unsigned long long order_key64(double v)
{
    unsigned long long u = (unsigned long long)__double_as_longlong(v);
    if (u == 0x8000000000000000ull) u = 0ull;
    return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
__device__ __forceinline__ double key_value64(unsigned long long k)
{
    return __longlong_as_double((long long)((k >> 63) ? (k & 0x7fffffffffffffffull) : ~k));
}

__global__ __launch_bounds__(kSelThreads) void approx_topk_f64_kernel(const double *__restrict__ scores, int F, long k,
                                                                     int W, double *__restrict__ threshold)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ SelShared sh;
    unsigned long long *cell = reinterpret_cast<unsigned long long *>(smem);  // [4][W], W <= 1024
    const int tid = threadIdx.x, b = blockIdx.x;
    const double *row = scores + (size_t)b * F;
    const unsigned long long kNegInf = order_key64(-__builtin_inf());
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (tid + u * kSelThreads < 4 * W) cell[tid + u * kSelThreads] = kNegInf;
    __syncthreads();
    for (int f = tid; f < F; f += kSelThreads) {
        const unsigned long long kv = order_key64(row[f]);
#pragma unroll
        for (int s = 0; s < 4; ++s) atomicMax(&cell[s * W + (int)(((long)s * F + f) % W)], kv);
    }
    __syncthreads();
    unsigned long long kr[4];
    int filled = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = tid + u * kSelThreads;
        kr[u] = i < 4 * W ? cell[i] : kNegInf;
        filled += kr[u] != kNegInf;
    }
    const long cells = (long)(block_sum((double)filled, sh, tid) + 0.5);
    if (cells == 0) {
        if (tid == 0) threshold[b] = 0.0;
        return;
    }
    long sk = k * cells / F;
    if (sk < 1) sk = 1;
    if (sk > cells) sk = cells;
    // (empty cells hold the key of -inf, the smallest there is: they never reach the sk <= cells largest)
    uint32_t rem, cnt;
    auto sweep_hi = [&](auto &&fn) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (tid + u * kSelThreads < 4 * W) fn((uint32_t)(kr[u] >> 32));
    };
    const uint32_t hi = radix_select_desc(sweep_hi, (uint32_t)sk, sh, tid, rem, cnt);
    const uint32_t want = rem;   // the rem-th largest lower half among the keys whose upper half is `hi`
    __syncthreads();
    auto sweep_lo = [&](auto &&fn) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (tid + u * kSelThreads < 4 * W && (uint32_t)(kr[u] >> 32) == hi) fn((uint32_t)kr[u]);
    };
    const uint32_t lo = radix_select_desc(sweep_lo, want, sh, tid, rem, cnt);
    if (tid == 0) threshold[b] = key_value64(((unsigned long long)hi << 32) | lo) * 0.9;
}

}  // namespace st

extern "C" int64_t st_mask_select_workspace_bytes(int64_t B, int64_t I)
{
    if (B < 1 || I < 1) return 0;
    return 16 + B * ((I + 15) / 16 * 16);
}

extern "C" int st_mask_select(const float *scores, int64_t B, int64_t I, int method, int64_t k, float z,
                              uint8_t *mask, float *cutoff, void *workspace, int64_t workspace_bytes, void *stream)
{
    using namespace st;
    ST_REQUIRE(scores && mask, "st_mask_select: null pointer");
    const int into = method >= 0 && (method & ST_MASK_INTO_ZEROS) ? 1 : 0;
    method &= ~ST_MASK_INTO_ZEROS;
    ST_REQUIRE(method == ST_MASK_TOPK || method == ST_MASK_STATISTICAL, "st_mask_select: unknown method %d", method);
    ST_REQUIRE(B >= 1 && B <= 4096, "st_mask_select: B=%lld out of range [1,4096]", (long long)B);
    ST_REQUIRE(I >= 1 && I <= (1 << 24), "st_mask_select: I=%lld out of range", (long long)I);
    const int ldm = (int)((I + 15) / 16 * 16);
    unsigned int *ticket = nullptr;
    uint8_t *rowmask = nullptr;
    if (B > 1 && !into) {
        ST_REQUIRE(workspace && workspace_bytes >= st_mask_select_workspace_bytes(B, I),
                   "st_mask_select: workspace of %lld bytes needed for B=%lld, I=%lld",
                   (long long)st_mask_select_workspace_bytes(B, I), (long long)B, (long long)I);
        ST_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0, "st_mask_select: workspace must be 16-byte aligned");
        ticket = static_cast<unsigned int *>(workspace);
        rowmask = static_cast<uint8_t *>(workspace) + 16;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    ProfScope ps(ST_K_MASK_SELECT, s);
    auto go = [&](auto kern, size_t lds) {
        ST_LAUNCH(ps, kern, dim3((unsigned)B), dim3(kSelThreads), lds, s, scores, mask, rowmask, cutoff, ticket, (int)B, (int)I, ldm,
                  (lds > 0 ? 1 : 0) | (into ? 2 : 0), (long)k, z);
    };
    const size_t keys = (size_t)I * 4, lds = keys > kKeyHistBytes ? keys : kKeyHistBytes;   // keys, or the histogram before them
    if (method == ST_MASK_TOPK) {
        const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(mask_select_kernel<0, ST_MASK_TOPK>), kSelMaxLdsKeys * 4);
        if (rc != ST_OK) return rc;
        if (I <= 8 * kSelThreads) go(mask_select_kernel<8, ST_MASK_TOPK>, lds);
        else if (I <= 16 * kSelThreads) go(mask_select_kernel<16, ST_MASK_TOPK>, lds);
        else go(mask_select_kernel<0, ST_MASK_TOPK>, I <= kSelMaxLdsKeys ? keys : 0);
    } else {
        if (I <= 8 * kSelThreads) go(mask_select_kernel<8, ST_MASK_STATISTICAL>, 0);
        else if (I <= 16 * kSelThreads) go(mask_select_kernel<16, ST_MASK_STATISTICAL>, 0);
        else go(mask_select_kernel<0, ST_MASK_STATISTICAL>, 0);
    }
    ST_HIP(hipGetLastError());
    return ST_OK;
}

extern "C" int st_approx_topk_threshold(const float *scores, int64_t B, int64_t F, int64_t k, float *threshold,
                                        void *stream)
{
    using namespace st;
    ST_REQUIRE(scores && threshold, "st_approx_topk_threshold: null pointer");
    ST_REQUIRE(B >= 1 && B <= 65535, "st_approx_topk_threshold: B=%lld out of range", (long long)B);
    ST_REQUIRE(F >= 4 && F <= (1 << 24), "st_approx_topk_threshold: feature size %lld out of range [4, 2^24]",
               (long long)F);
    ST_REQUIRE(k > 0, "st_approx_topk_threshold: k must be positive");
    ST_REQUIRE(k <= F, "st_approx_topk_threshold: k cannot be larger than feature size");
    const int W = (int)(F / 4 < 1024 ? F / 4 : 1024);
    hipStream_t s = static_cast<hipStream_t>(stream);
    ProfScope ps(ST_K_MASK_SELECT, s);
    ST_LAUNCH(ps, approx_topk_kernel, dim3((unsigned)B), dim3(kSelThreads), (size_t)4 * W * 4, s, scores, (int)F, (long)k,
              W, threshold);
    ST_HIP(hipGetLastError());
    return ST_OK;
}

extern "C" int st_approx_topk_threshold_f64(const double *scores, int64_t B, int64_t F, int64_t k, double *threshold,
                                            void *stream)
{
    using namespace st;
    ST_REQUIRE(scores && threshold, "st_approx_topk_threshold_f64: null pointer");
    ST_REQUIRE(B >= 1 && B <= 65535, "st_approx_topk_threshold_f64: B=%lld out of range", (long long)B);
    ST_REQUIRE(F >= 4 && F <= (1 << 24), "st_approx_topk_threshold_f64: feature size %lld out of range [4, 2^24]",
               (long long)F);
    ST_REQUIRE(k > 0, "st_approx_topk_threshold_f64: k must be positive");
    ST_REQUIRE(k <= F, "st_approx_topk_threshold_f64: k cannot be larger than feature size");
    const int W = (int)(F / 4 < 1024 ? F / 4 : 1024);
    hipStream_t s = static_cast<hipStream_t>(stream);
    ProfScope ps(ST_K_MASK_SELECT, s);
    ST_LAUNCH(ps, approx_topk_f64_kernel, dim3((unsigned)B), dim3(kSelThreads), (size_t)4 * W * 8, s, scores, (int)F,
              (long)k, W, threshold);
    ST_HIP(hipGetLastError());
    return ST_OK;
}
