// LoRA importance predictor for several rows of x (fp16 / bf16): both maps on the matrix cores.
//
//   kernel 1  t[b,k] = <x[b,:], A[k,:]>     tiles of (16 MI) x (16 NI), the block's waves split the hidden dimension;
//                                           also clears the mask
//   kernel 2  s[b,i] = <t[b,:], Bm[i,:]>    a wave keeps its rows of t in registers and walks over rows of Bm;
//             mask[i] = 1 where any s[b,i] passes the cut (only ones are stored)
//
// The rank-r intermediate is fp32, and the matrix cores multiply 16-bit operands: kernel 2 splits t into three parts of the
// storage type that sum to it, each made of what the parts before it left over.  Three parts hold all 24 bits (two of fp16
// hold 23, which a quarter of all values exceed).  Rows of fp16 parts are scaled by a power of two that puts their largest
// element near 2^14; only of elements below 2^-15 of that one something may be lost to the subnormals, less than 2^-38 of
// the largest.  In kernel 2 every product is exact and the sums are fp32: the scores keep fp32 accuracy.
//
// Same contract as predictor.hip (src/modeling_skip.py:52-53,204-207,214).
#include "st_mfma.h"

#include <type_traits>

namespace st {

constexpr int kSplitParts = 3;

// ---------------------------------------------------------------------------
// kernel 1
// ---------------------------------------------------------------------------
// A tile of 16 MI rows of x by 16 NI rank rows per block.  Its W waves deal out pieces of 8 PC of the hidden dimension among
// themselves; a wave loads the 16 PC bytes of every row of its next pieces straight into a ring of NB buffers of its own in
// LDS while it multiplies the present one, so nothing waits for another wave until the sums meet at the end.  (Fragments
// loaded from memory into registers, 16 rows x 64 bytes per instruction, went through a CU at 15 bytes per clock.)
// Bound by what a CU pulls through its L2, so by the rows of a tile per result and by the bytes in flight: 2048 rows, H 4096,
// rank 256, bf16: 32 x 32 tiles with rank tiles fastest (every XCD read all of x) 25.2 us, 64 x 32 by XCD 12.1.
// LDS rows are PC chunks of 16 bytes; chunk c of row k at c ^ (k % 16), or c ^ (k / 2 % 8) for rows of 128 bytes: the 16 rows
// of a fragment read meet every bank alike.
template <typename T, int MI, int NI, int W, int PC, int NB, typename Tab>
__global__ __launch_bounds__(W * kWave) void predictor_down_mfma_kernel(const T *__restrict__ x, const T *__restrict__ A,
                                                                        int B, int H, int r,
                                                                        float *__restrict__ t, uint8_t *__restrict__ mask,
                                                                        int I, int launch_word, int blocks, Tab tab)
{
    if constexpr (Tab::kLayers) {   // several layers of equal shape at once: x [layers,B,H], t [layers,B,r]
        A = static_cast<const T *>(tab.l[blockIdx.z].A);
        mask = tab.l[blockIdx.z].mask;
        x += (size_t)blockIdx.z * B * H;
        t += (size_t)blockIdx.z * B * r;
    }
    // (14 dwords of arguments, all in scalar registers when the wave starts; the grid's size would arrive by a load)
    const int gx = launch_word >> 2, rank_first = launch_word & 2, round_storage = launch_word & 1;
    constexpr int kThreads = W * kWave, kPiece = 8 * PC;
    constexpr int kRows = 16 * (MI + NI), kBuf = kRows * PC, kDma = kBuf / 64;   // a wave's buffer in chunks, its 1 KB loads
    static_assert((PC == 16 || PC == 8) && (NB - 1) * kDma < 64, "swizzle; waits count to 63");
    extern __shared__ __align__(16) uint4 lds[];   // [W][NB][kRows][PC]
    auto swz = [](int row) __attribute__((always_inline)) { return PC == 16 ? row & 15 : (row >> 1) & 7; };
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    // (tiles of x fastest, their number padded to a multiple of the XCDs: a tile's rows come through one L2 only.  Or tiles of
    // the rank, launch_t.  No division, which takes a launch of this size 0.3 us)
    const int m0 = (rank_first ? blockIdx.y : blockIdx.x) * 16 * MI, k0 = (rank_first ? blockIdx.x : blockIdx.y) * 16 * NI;
    const bool live = m0 < B;
    const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
    const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) uint4 *)lds;

    // load j fills 64 / PC LDS rows, lane i position i % PC of row i / PC.  Rows are clamped into range (what they
    // feed is not stored), and so are columns past the end of a row (replaced by zeros below).  Offsets of 32 bits only
    // reach over the tile's own rows: x may be larger than 4 GiB.
    constexpr int kLoadRows = 64 / PC;
    const char *const x_tile = reinterpret_cast<const char *>(x + (size_t)m0 * H);
    const char *const a_tile = reinterpret_cast<const char *>(A + (size_t)k0 * H);
    unsigned doff[kDma];
#pragma unroll
    for (int j = 0; j < kDma; ++j) {
        const int row = kLoadRows * j + lane / PC;
        int g = row < 16 * MI ? row : row - 16 * MI;
        const int last = row < 16 * MI ? B - 1 - m0 : r - 1 - k0;
        g = g < last ? g : last;
        doff[j] = (unsigned)g * (unsigned)H * (unsigned)sizeof(T);
    }
    const int pieces = (H + kPiece - 1) / kPiece;
    auto dma = [&](int piece, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kDma; ++j) {
            const int row = kLoadRows * j + lane / PC, c = (lane % PC) ^ swz(row);
            const int h = piece * kPiece + 8 * c;
            load_to_lds(lds_base + (unsigned)((wave * NB + b) * kBuf + j * 64) * 16u, doff[j] + (unsigned)(h < H ? h : 0) * (unsigned)sizeof(T),
                        kLoadRows * j < 16 * MI ? x_tile : a_tile);
        }
    };
    f32x4_t acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < NB - 1; ++p)
        if (live && wave + p * W < pieces) dma(wave + p * W, p);
    // the mask is cleared here, a kernel ahead of the one that switches bytes on (the stores are newer than the loads that are
    // counted below: the first wait lets that many fewer of the second piece's loads be outstanding)
    for (int i = (blockIdx.y * gx + blockIdx.x) * kThreads + tid; i < I; i += blocks * kThreads) mask[i] = 0;
    if (!live) return;
    int b = 0;
    for (int piece = wave; piece < pieces; piece += W) {
        // this piece has arrived once all but the newer ones' loads have; the next loads go out once the reads of the last
        // use of their buffer are done
        if (NB > 2 && piece + W < pieces) ST_WAIT_VM_LGKM0((NB - 2) * kDma); else ST_WAIT_VM_LGKM0(0);
        asm volatile("" ::: "memory");
        const int before = b == 0 ? NB - 1 : b - 1;
        if (piece + (NB - 1) * W < pieces) dma(piece + (NB - 1) * W, before);
        const uint4 *buf = lds + (wave * NB + b) * kBuf;
#pragma unroll
        for (int ks = 0; ks < kPiece / 32; ++ks) {
            uint4 fa[MI], fb[NI];
            const int c = (4 * ks + q) ^ swz(l16);
#pragma unroll
            for (int i = 0; i < MI; ++i) fa[i] = buf[(16 * i + l16) * PC + c];
#pragma unroll
            for (int j = 0; j < NI; ++j) fb[j] = buf[(16 * (MI + j) + l16) * PC + c];
            if (piece * kPiece + 32 * ks + 8 * q >= H) {   // (both operands: a product with zero must not meet an infinity)
#pragma unroll
                for (int i = 0; i < MI; ++i) fa[i] = zero4;
#pragma unroll
                for (int j = 0; j < NI; ++j) fb[j] = zero4;
            }
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j) acc[i][j] = Mfma<T>::run(fa[i], fb[j], acc[i][j]);
        }
        b = b == NB - 1 ? 0 : b + 1;
    }
    // (the sums lie over the front of the buffers, the first waves': behind the barrier nobody reads those any more)
    typedef float Red[MI * NI][256];
    Red *red = reinterpret_cast<Red *>(lds);
    static_assert(sizeof(Red) <= NB * kBuf * 16, "a wave's sums exceed its buffers");
    __syncthreads();

    // D[m][n]: a lane holds rows 4 q + e of column l16
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[wave][i * NI + j][(4 * q + e) * 16 + l16] = acc[i][j][e];
    __syncthreads();
    for (int o = tid; o < MI * NI * 256; o += kThreads) {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) s += red[w][o >> 8][o & 255];
        const int tile = o >> 8, m = m0 + 16 * (tile / NI) + ((o >> 4) & 15), k = k0 + 16 * (tile % NI) + (o & 15);
        if (m < B && k < r) t[(size_t)m * r + k] = round_storage ? to_float<T>(from_float<T>(s)) : s;
    }
}

// ---------------------------------------------------------------------------
// kernel 2
// ---------------------------------------------------------------------------
constexpr float kMaxF32 = 3.402823466e+38f;

// Eight floats of t -> the parts of one A operand register quad each.  TINY (fp16): some are too small for a first part.
template <typename T, bool TINY> __device__ __forceinline__ void split_parts(const float *v, uint4 *parts)
{
    if constexpr (std::is_same<T, bf16_t>::value) {
        // The first part is the upper half of the float: no finite value becomes an infinity (rounding it did, above
        // 3.396e38), and what it leaves over has 16 bits, which two rounded parts hold.
        uint32_t hi[4];
        bf16x8_t w[kSplitParts - 1];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            float rest = v[k] - __uint_as_float(__float_as_uint(v[k]) & 0xffff0000u);
            rest = rest == rest ? rest : 0.f;           // an infinity or NaN has nothing left over
#pragma unroll
            for (int p = 0; p < kSplitParts - 1; ++p) {
                const __bf16 b = (__bf16)rest;          // (the hardware's conversion: round to nearest even)
                w[p][k] = b;
                rest -= (float)b;
            }
            if (k & 1) hi[k >> 1] = __builtin_amdgcn_perm(__float_as_uint(v[k]), __float_as_uint(v[k - 1]), 0x07060302u);
        }
        parts[0] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
#pragma unroll
        for (int p = 1; p < kSplitParts; ++p) parts[p] = __builtin_bit_cast(uint4, w[p - 1]);
    } else {
        uint32_t w[kSplitParts][8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            float rest = v[k];
#pragma unroll
            for (int p = 0; p < kSplitParts; ++p) {
                f16_t h = from_float<f16_t>(rest);
                // (the first part keeps the sign of what is too small for it: it decides what an infinite weight gives)
                if (TINY && p == 0 && (h.bits & 0x7fffu) == 0u && rest != 0.f) h.bits |= 1u;
                w[p][k] = h.bits;
                rest -= to_float<f16_t>(h);
                if (p == 0) rest = rest == rest ? rest : 0.f;   // an infinity or NaN has nothing left over
            }
        }
#pragma unroll
        for (int p = 0; p < kSplitParts; ++p)
            parts[p] = make_uint4(w[p][0] | (w[p][1] << 16), w[p][2] | (w[p][3] << 16), w[p][4] | (w[p][5] << 16),
                                  w[p][6] | (w[p][7] << 16));
    }
}

// A wave owns 16 rows of t (KS k steps of 32 of the rank, in registers as parts) and walks over rows of Bm, which the
// block loads 64 rows (a stage) at a time straight into LDS, one stage ahead: its W waves share them (fragments loaded by
// every wave on its own: 97 us for 2048 rows at rank 256, I 14336).  W / IG of the waves own different rows of t, the IG
// groups take different 16-row tiles of a stage; a block takes `per` stages.
// MFMA bound: a tile of 16 indices is 3 KS of them, and while they run each fragment they have consumed is replaced by the
// next tile's, so that no read is waited for.  What is left of a tile's work is the decision.  Unless scores are written or
// rounded, rows of t past B are copies of the last one and columns past I are dropped at the end, so that a
// lane's four scores become one comparison of their maximum.  Rows 2048, rank 256, I 14336, bf16 (45 GFLOP with the parts, 23
// us of MFMAs): 58.8 us with reads just ahead of their use and a decision per score, now 39.5.
// LDS rows are 4 KS chunks of 16 bytes (the rank rounded up; the surplus chunks repeat others and are not used), chunk c of
// row k sits at c ^ (k % 16): the 16 rows of a fragment read meet different banks.  Which indices a row switched on is
// collected in LDS too: a store to memory inside the loop would have to be waited for together with the next stage.
constexpr int kPmStage = 64;

template <typename T, int KS, int W, int IG, typename Tab>
__global__ __launch_bounds__(W * kWave) void predictor_up_mfma_kernel(const float *__restrict__ t,
                                                                      const T *__restrict__ Bm, int B, int r, int I,
                                                                      int per, float thr, int flags,
                                                                      float *__restrict__ scores,
                                                                      uint8_t *__restrict__ mask, Tab tab)
{
    if constexpr (Tab::kLayers) {
        const st_predictor_layer &ly = tab.l[blockIdx.z];
        Bm = static_cast<const T *>(ly.Bm);
        mask = ly.mask;
        thr = ly.thr;
        flags = (flags & ~1) | (ly.cmp_ge ? 1 : 0);
        t += (size_t)blockIdx.z * B * r;
    }
    constexpr int P = kSplitParts;
    constexpr bool kScaled = std::is_same<T, f16_t>::value;
    constexpr int kRow = 4 * KS, kBuf = kPmStage * kRow;      // 16-byte chunks
    constexpr int kDma = kBuf / 64 / W;                       // 1 KB loads per wave and stage
    extern __shared__ __align__(16) uint4 lds[];              // two buffers, then a byte per index of the block
    uint8_t *hits = reinterpret_cast<uint8_t *>(lds + 2 * kBuf);
    const int cmp_ge = flags & 1, round_storage = (flags >> 1) & 1;
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    constexpr int WB = W / IG, NT = kPmStage / 16 / IG;       // waves with rows of t of their own, tiles of a wave per stage
    const int j0 = wave / WB;                                 // first of them: j0, j0 + IG, ...
    // blocks of one XCD (ids equal modulo 8; the grid's x is a multiple of 8 where it can be) work on the same rows of Bm
    const int m0 = (blockIdx.y * WB + wave % WB) * 16;
    const int stages = (I + kPmStage - 1) / kPmStage;
    const int s0 = blockIdx.x * per, s1 = s0 + per < stages ? s0 + per : stages;
    const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);

    const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) uint4 *)lds;
    unsigned doff[kDma];
    auto lane_off = [&](int j, int last) __attribute__((always_inline)) {
        const int at = (wave * kDma + j) * 64 + lane, row = at / kRow, c = (at % kRow) ^ (row & 15);
        return ((unsigned)(row < last ? row : last) * (unsigned)r + (unsigned)(8 * c < r ? 8 * c : 0)) * (unsigned)sizeof(T);
    };
#pragma unroll
    for (int j = 0; j < kDma; ++j) doff[j] = lane_off(j, kPmStage);
    auto dma = [&](int stage, int b) __attribute__((always_inline)) {
        const T *const rows = Bm + (size_t)stage * kPmStage * r;   // (offsets within the stage: Bm may be larger than 4 GiB)
        const int last = I - 1 - stage * kPmStage;
        const bool clip = last < kPmStage - 1;                      // uniform: the last row is repeated
#pragma unroll
        for (int j = 0; j < kDma; ++j)
            load_to_lds(lds_base + (unsigned)(b * kBuf + (wave * kDma + j) * 64) * 16u, clip ? lane_off(j, last) : doff[j],
                        reinterpret_cast<const char *>(rows));
    };
    if (s0 >= s1) return;
    dma(s0, 0);
    for (int i = threadIdx.x; i < per * (kPmStage / 4); i += W * kWave) reinterpret_cast<uint32_t *>(hits)[i] = 0u;

    uint4 tf[P][KS];
    float unscale[4];        // of the rows this lane's results belong to
    {
        const int m = m0 + l16;
        const float *row = t + (size_t)(m < B ? m : B - 1) * r;
        float v[KS][8];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int k = 32 * ks + 8 * q;
            const float4 lo = *reinterpret_cast<const float4 *>(row + (k < r ? k : 0));
            const float4 hi = *reinterpret_cast<const float4 *>(row + (k < r ? k + 4 : 0));
            const float w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) v[ks][e] = k < r ? w[e] : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) unscale[e] = 1.f;
        if constexpr (kScaled) {
            // a power of two per row that puts its largest finite element near 2^14
            float big = 0.f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float a = fabsf(v[ks][e]);
                    big = a < 3.0e38f ? fmaxf(big, a) : big;
                }
            big = fmaxf(big, __shfl_xor(big, 16, kWave));
            big = fmaxf(big, __shfl_xor(big, 32, kWave));
            int ex = (int)(__float_as_uint(big) >> 23) - 127;
            ex = ex < -96 ? -96 : ex;                              // (also for a row of zeros)
            const float scale = __uint_as_float((uint32_t)(127 + 13 - ex) << 23);
            const float back = __uint_as_float((uint32_t)(127 - 13 + ex) << 23);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int e = 0; e < 8; ++e) v[ks][e] *= scale;
#pragma unroll
            for (int e = 0; e < 4; ++e) unscale[e] = __shfl(back, 4 * q + e, kWave);
        }
        auto split = [&](auto tiny) __attribute__((always_inline)) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                uint4 parts[P];
                split_parts<T, decltype(tiny)::value>(v[ks], parts);
#pragma unroll
                for (int p = 0; p < P; ++p) tf[p][ks] = parts[p];
            }
        };
        if constexpr (kScaled) {
            // elements of up to 2^-25 that are not zero have no first part (the smallest of them all, zeros last)
            uint32_t least = ~0u;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint32_t m = (__float_as_uint(v[ks][e]) << 1) - 1u;
                    least = m < least ? m : least;
                }
            if (__builtin_amdgcn_ballot_w64(least < (uint32_t)(127 - 25) << 24) != 0) split(std::true_type{});
            else split(std::false_type{});
        } else {
            split(std::false_type{});
        }
    }
    const bool gen = scores != nullptr || round_storage;
    // v > thr as v >= the next number up (none above infinity: nothing passes)
    float least_in = thr;
    if (!cmp_ge) {
        const uint32_t u = __float_as_uint(thr);
        const uint32_t up = (u << 1) == 0u ? 1u : (u >> 31) ? u - 1u : u + 1u;
        least_in = thr < __builtin_inff() ? __uint_as_float(up) : __uint_as_float(0x7fc00000u);
    }
    // A lane's score: the parts' sums, smallest first.  An infinite element of Bm decides the score by the sign of t, which
    // its first part has; the others are zero or of either sign and would make a NaN of it: they are kept finite (the median
    // with a NaN among them is the least of the others).
    auto score = [&](const f32x4_t (&acc)[P], int e) __attribute__((always_inline)) {
        float rest = acc[P - 1][e];
#pragma unroll
        for (int p = P - 2; p >= 1; --p) rest += acc[p][e];
        float v = __builtin_amdgcn_fmed3f(rest, -kMaxF32, kMaxF32) + acc[0][e];
        if constexpr (kScaled) v *= unscale[e];
        return v;
    };
    auto decide = [&](const f32x4_t (&acc)[P], int col) __attribute__((always_inline)) -> bool {
        if (__builtin_expect(!gen, 1)) {
            const float v = fmaxf(fmaxf(score(acc, 0), score(acc, 1)), fmaxf(score(acc, 2), score(acc, 3)));
            return v >= least_in;   // (a NaN never passes, and the maximum is one only if all four are)
        }
        bool any = false;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float v = score(acc, e);
            if (round_storage) v = to_float<T>(from_float<T>(v));
            const bool in = m0 + 4 * q + e < B;
            any = any || (in && v >= least_in);
            if (scores && in && col < I) scores[(size_t)(m0 + 4 * q + e) * I + col] = v;
        }
        return any;
    };

    const bool ragged = r < 32 * KS;   // (r > 32 (KS - 4): the launch picks KS; past the rank t is zero, and so must be what it meets)
    uint4 bf[KS];
    // (a lane's fragments of the wave's first tile in the stage that is read: everything else is a constant offset)
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    const __attribute__((address_space(3))) u32x4_t *at[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
        at[ks] = (const __attribute__((address_space(3))) u32x4_t *)lds + (16 * j0 + l16) * kRow + ((4 * ks + q) ^ l16);
    ST_WAIT_VM_LGKM0(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s0 + 1 < s1) dma(s0 + 1, 1);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) bf[ks] = __builtin_bit_cast(uint4, *at[ks]);
    for (int s = s0; s < s1; ++s) {
        const int b = (s - s0) & 1;
        uint64_t stage_hits = 0;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            if (i == NT - 1 && s + 1 < s1) {
                // the wave's last tile of the stage is in registers: behind the barrier the next stage is in LDS, and the
                // buffer of this one is free for the one after it
                ST_WAIT_VM_LGKM0(0);
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                if (s + 2 < s1) dma(s + 2, b);
            }
            if (ragged) {
#pragma unroll
                for (int ks = KS - 4; ks < KS; ++ks)
                    if (32 * ks + 8 * q >= r) bf[ks] = zero4;
            }
            f32x4_t acc[P];
#pragma unroll
            for (int p = 0; p < P; ++p) acc[p] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
                for (int p = 0; p < P; ++p) acc[p] = Mfma<T>::run(tf[p][ks], bf[ks], acc[p]);
                __builtin_amdgcn_sched_barrier(0);
                // (past the last stage: a stale buffer, not used)
                if (i == NT - 1) at[ks] += b ? -kBuf : kBuf;
                bf[ks] = __builtin_bit_cast(uint4, at[ks][i == NT - 1 ? 0 : 16 * IG * (i + 1) * kRow]);
                __builtin_amdgcn_sched_barrier(0);
            }
            const int j = j0 + IG * i;
            uint64_t hit = __builtin_amdgcn_ballot_w64(decide(acc, s * kPmStage + 16 * j + l16));
            hit |= hit >> 32;
            hit |= hit >> 16;
            stage_hits |= (hit & 0xffffull) << (16 * j);
        }
        if ((stage_hits >> lane) & 1ull) hits[(s - s0) * kPmStage + lane] = 1;
    }
    __syncthreads();
    const int first = s0 * kPmStage, count = (I < s1 * kPmStage ? I : s1 * kPmStage) - first;
    for (int i = threadIdx.x; i < count; i += W * kWave)
        if (hits[i]) mask[first + i] = 1;
}

// From nine rows of x on.  The kernels of predictor.hip read every element of t from LDS for every row of x (about 1 us a
// row at rank 256) and take x in passes of eight, sixteen and at last 64 rows; these take 7-14 us for any number up to 64.
// Both kernels, replayed from a graph, there / here, at H 3072, rank 128, I 8192 (bf16): 7.5 / 8.4 us for 8 rows, 9.9 / 8.7
// for 12, 17.0 / 9.6 for 32, 29.5 / 10.6 for 64, 233 / 15.6 for 512, 929 / 31 for 2048; at H 4096, rank 256, I 14336:
// 10.6 / 10.6, 14.3 / 11.0, 25.0 / 12.1, 68.9 / 13.2, 538 / 29, 2236 / 78.  Ranks above 512 do not fit the registers, and
// the 32 rows of x of a tile (64 where H allows it, launch_t) have to stay within 32-bit offsets.
bool predictor_mfma_supported(int dtype, int B, int H, int r)
{
    return dtype != ST_F32 && B > 8 && r <= 512 && H < (1 << 26);
}

// The second kernel alone.  What it switches on has to be off.
template <typename T, typename Tab>
static int launch_up_t(const Tab &tab, int layers, int B, int r, const void *Bm, int I, float thr, int cmp_ge, float *t_ws,
                       float *scores, uint8_t *mask, int round_storage, hipStream_t stream)
{
    // (the CUs a layer can count on when several share the launch)
    const int cus = (device_cu_count() + layers - 1) / layers;
    {
        ProfScope ps(ST_K_PRED_UP_MASK, stream);
        // resident: blocks a CU holds at once (registers, LDS).  One round of blocks: every further one would split its
        // rows of t into parts again.
        auto go = [&](auto kern, int ks, int wb, int waves, int resident) -> int {
            const int mt = (B + 16 * wb - 1) / (16 * wb), stages = (I + kPmStage - 1) / kPmStage;
            // (as many per XCD as its CUs hold: 19 splits of 12 row tiles, three on some XCDs, took two rounds there: 1536 rows,
            // rank 256, I 8192: both kernels 52 us, with two on each 34.9)
            const int per_xcd = resident * cus / (kXcds * mt);
            int splits = per_xcd > 0 ? per_xcd * kXcds : resident * cus / mt;
            if (splits < 1) splits = 1;
            int per = (stages + splits - 1) / splits;
            per = per < 256 ? per : 256;                     // (the LDS bytes of a block's indices)
            splits = (stages + per - 1) / per;
            if (splits > kXcds) splits = (splits + kXcds - 1) / kXcds * kXcds;
            const int lds = 2 * kPmStage * 4 * ks * 16 + per * kPmStage;
            const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), 2 * kPmStage * 4 * ks * 16 + 256 * kPmStage);
            if (rc != ST_OK) return rc;
            ST_LAUNCH(ps, kern, dim3(splits, mt, layers), dim3(waves * kWave), lds, stream, t_ws, static_cast<const T *>(Bm), B, r,
                      I, per, thr, (cmp_ge ? 1 : 0) | (round_storage ? 2 : 0), scores, mask, tab);
            return ST_OK;
        };
#define ST_PM_UP(KS, W, IG, RES) go(predictor_up_mfma_kernel<T, KS, W, IG, Tab>, KS, W / IG, W, RES)
#define ST_PM_UP4(KS, RES) (B <= 16 ? ST_PM_UP(KS, 4, 4, RES) : B <= 32 ? ST_PM_UP(KS, 4, 2, RES) : ST_PM_UP(KS, 4, 1, RES))
        int rc;
        // (eight waves share a stage once there are rows of x for them: 16 rows in blocks of eight waves 5.2 us, of four 4.4.
        // At ranks 257 to 384 their fp16 form spills 46 registers, most of them outside the loop: both kernels, 128 rows, rank
        // 384, fp16 / bf16 26.0 / 20.6 us)
        if (B <= 64) {
            if (r <= 128) rc = ST_PM_UP4(4, 4);
            else if (r <= 256) rc = ST_PM_UP4(8, 2);
            else if (r <= 384) rc = ST_PM_UP4(12, 1);
            else rc = ST_PM_UP4(16, 1);
        } else if (r <= 128) rc = ST_PM_UP(4, 8, 1, 2);
        else if (r <= 256) rc = ST_PM_UP(8, 8, 1, 1);
        else if (r <= 384) rc = ST_PM_UP(12, 8, 1, 1);
        else rc = ST_PM_UP(16, 4, 1, 1);   // (eight waves of 256 registers cannot hold its parts)
#undef ST_PM_UP4
#undef ST_PM_UP
        if (rc != ST_OK) return rc;
    }
    ST_HIP(hipGetLastError());
    return ST_OK;
}

template <typename T, typename Tab>
static int launch_t(const Tab &tab, int layers, const void *x, int B, int H, const void *A, int r, const void *Bm, int I,
                    float thr, int cmp_ge, float *t_ws, float *scores, uint8_t *mask, int round_storage, hipStream_t stream)
{
    {
        ProfScope ps(ST_K_PRED_DOWN, stream);
        auto go = [&](auto kern, int mi, int ni, int waves, int row_chunks) -> int {
            int mt = (B + 16 * mi - 1) / (16 * mi);
            const int nt = (r + 16 * ni - 1) / (16 * ni);
            // Tiles of x by XCD where x is the larger operand, unless their padded number takes the CUs of an XCD more rounds
            // than tiles dealt out evenly.  (Order only: the sums are the same.)  Both kernels, bf16, H 4096, tiles of x first
            // / of the rank first: 100 rows, rank 384, 21.3 / 19.6 us; 160 rows, rank 320, 27.2 / 23.3 (ten tiles: two rounds on
            // two XCDs); 400 rows, rank 320, 33.7 / 30.4; 1024 rows, rank 256, 32.8 / 37.4
            const int cus = device_cu_count(), xcd_cus = cus >= kXcds ? cus / kXcds : 1;
            const bool rank_first = B < r || (layers * ((mt + kXcds - 1) / kXcds) * nt + xcd_cus - 1) / xcd_cus >
                                                 (layers * mt * nt + cus - 1) / cus;
            if (!rank_first && mt > kXcds) mt = (mt + kXcds - 1) / kXcds * kXcds;
            const int gx = rank_first ? nt : mt, gy = rank_first ? mt : nt;
            const int lds = waves * 16 * (mi + ni) * row_chunks * 16;
            const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds);
            if (rc != ST_OK) return rc;
            ST_LAUNCH(ps, kern, dim3(gx, gy, layers), dim3(waves * kWave), lds, stream, static_cast<const T *>(x),
                      static_cast<const T *>(A), B, H, r, t_ws, mask, I, gx << 2 | (rank_first ? 2 : 0) | (round_storage ? 1 : 0),
                      mt * nt, tab);
            return ST_OK;
        };
        auto blocks = [&](int mi, int ni) { return ((B + 16 * mi - 1) / (16 * mi)) * ((r + 16 * ni - 1) / (16 * ni)); };
        // The largest tile of which there is one for three quarters of the CUs (by the shape alone: how many layers share the
        // launch must not change how the sums are split).  32 x 32 tiles have half the traffic from L2: 6.7 (16 x 16) against
        // 8.6 us with 64 of them (512 rows, H 3072, rank 128), 17.8 against 11.8 us with 224, 40 against 26 us with 512.  64 x
        // 32 tiles a quarter less again and 96 KB of loads in flight instead of 64, both kernels, 32 x 32 / 64 x 32: 33.7 / 35.0
        // us with 128 of them (1024 rows, H 4096, rank 256), 57.4 / 52.0 with 192, 54.9 / 48.4 with 256 (2048 rows).
        // (a tile's rows of x have to stay within 32-bit offsets: 64 of them up to H = 2^25, 32 for every H that is taken at all)
        const bool reach = (int64_t)64 * H * (int64_t)sizeof(T) <= (int64_t)1 << 32;
        const int want = 3 * device_cu_count();
        const int rc = reach && 4 * blocks(4, 2) >= want ? go(predictor_down_mfma_kernel<T, 4, 2, 4, 8, 3, Tab>, 4, 2, 4, 24)
                       : 4 * blocks(2, 2) >= want        ? go(predictor_down_mfma_kernel<T, 2, 2, 4, 16, 2, Tab>, 2, 2, 4, 32)
                                                         : go(predictor_down_mfma_kernel<T, 1, 1, 8, 16, 2, Tab>, 1, 1, 8, 32);
        if (rc != ST_OK) return rc;
    }
    ST_HIP(hipGetLastError());
    return launch_up_t<T>(tab, layers, B, r, Bm, I, thr, cmp_ge, t_ws, scores, mask, round_storage, stream);
}

int launch_predictor_mfma(int dtype, const void *x, int B, int H, const void *A, int r, const void *Bm, int I, float thr,
                          int cmp_ge, float *t_ws, float *scores, uint8_t *mask, int round_storage, hipStream_t stream)
{
    auto go = dtype == ST_F16 ? launch_t<f16_t, NoLayers> : launch_t<bf16_t, NoLayers>;
    return go(NoLayers{}, 1, x, B, H, A, r, Bm, I, thr, cmp_ge, t_ws, scores, mask, round_storage, stream);
}

int launch_predictor_mfma_layers(int dtype, const PredLayers &tab, int layers, const void *x, int B, int H, int r, int I,
                                 float *t_ws, int round_storage, hipStream_t stream)
{
    auto go = dtype == ST_F16 ? launch_t<f16_t, PredLayers> : launch_t<bf16_t, PredLayers>;
    return go(tab, layers, x, B, H, nullptr, r, nullptr, I, 0.f, 0, t_ws, nullptr, nullptr, round_storage, stream);
}

// Five to eight rows of bf16 at ranks of 129 to 256: the first map as for fewer rows (one wave of loads per rank row on the
// whole chip; 16-row tiles of x would be half empty), the second on the matrix cores once its multiplications outweigh
// splitting the rows of t into parts (by the shape alone, as above).  Both kernels, on the vector ALUs / so, us, H 3072, one
// layer | eight together, by millions of multiplications (rows, rank, I):
//    6.6 (5, 160, 8192)   8.29 / 8.71 | 25.2 / 19.5       14.1 (5, 256, 11008)  9.27 / 9.16 | 32.3 / 24.1
//    9.2 (5, 224, 8192)   8.81 / 8.90 | 28.4 / 22.3       18.4 (8, 160, 14336) 10.21 / 9.53 | 38.3 / 22.9
//   10.5 (8, 160, 8192)   9.25 / 9.02 | 28.6 / 20.0       25.7 (8, 224, 14336) 10.82 / 9.85 | 40.4 / 25.0
// fp16 also scales the rows of t, which a single layer does not earn back (18.4 million, 5 rows of rank 256: 9.36 / 10.69; 29.4
// million, 8 rows: 10.20 / 10.94; eight layers together 33.4 / 26.7, 38.0 / 27.3).  Ranks of 320 to 512 (H 4096, single layers
// of bf16): 22.9 million, rank 320, 12.7 / 11.6; 15.7, rank 384, 11.5 / 11.3; 21.0, rank 512, 12.0 / 12.4.
bool predictor_up_mfma_supported(int dtype, int B, int r, int I)
{
    return dtype == ST_BF16 && B >= 5 && B <= 8 && r > 128 && r <= 256 && (int64_t)B * r * I >= 10000000;
}

template <typename Tab>
int launch_predictor_up_mfma(int dtype, const Tab &tab, int layers, int B, int r, const void *Bm, int I, float thr, int cmp_ge,
                             float *t_ws, float *scores, uint8_t *mask, int round_storage, hipStream_t stream)
{
    auto go = dtype == ST_F16 ? launch_up_t<f16_t, Tab> : launch_up_t<bf16_t, Tab>;
    return go(tab, layers, B, r, Bm, I, thr, cmp_ge, t_ws, scores, mask, round_storage, stream);
}
template int launch_predictor_up_mfma<NoLayers>(int, const NoLayers &, int, int, int, const void *, int, float, int, float *, float *,
                                                uint8_t *, int, hipStream_t);
template int launch_predictor_up_mfma<PredLayers>(int, const PredLayers &, int, int, int, const void *, int, float, int, float *,
                                                  float *, uint8_t *, int, hipStream_t);

}  // namespace st
