// Sparse MLP over the active set for a small batch of rows of x (3 <= B <= 32):
// still bound by the HBM stream of the active rows, but with B rows of x the
// multiply-adds no longer fit beside it on the vector ALUs, so they go to the
// matrix cores (fp16 / bf16 MFMA 16x16x32, fp32 16x16x4; fp32 accumulate).  16 rows of x form
// the N (kernel 1) / M (kernel 2) dimension of one tile; both kernels take up
// to two such tiles in one pass over the weights, more rows (fp32, hidden sizes the GEMM
// kernels do not take) in passes of 32.
//
//   kernel 1  h[b][j] = act(x_b . gate_j) * (x_b . up_j)
//             one block per CU owns a contiguous range of active rows and works
//             through it in tiles of 32 rows.  The 8 waves split the hidden
//             dimension: weight fragments go from HBM straight into MFMA
//             operand registers (16 rows x 64 bytes per load instruction, which
//             streams as fast as fully coalesced loads on this chip), x comes
//             from LDS where it fits or from registers, and the 8 partial tiles are
//             summed through LDS.
//   kernel 2  out[b][:] = sum_j h[b][j] * down_j[:]
//             K runs down the rows of the packed down matrix, so the operand
//             has to be transposed: blocks own (column group, row split), each
//             wave stages 32 rows x 64 columns in LDS and reads the fragment
//             with the transposing LDS load (fp32 needs neither).  Split-K partial rows are summed in a fixed order
//             by kernel 3.
// Unlike a per-CU fused kernel this writes no per-CU partial [B,H] rows (which
// would cost B * 3 MB of extra traffic); h (B * n elements) is the only
// intermediate.
//
// Each kernel has two forms: for the hidden sizes 2048, 3072 and 4096 of the 2-byte types, and for any other.
// The second, whole forward, us, before (streaming kernel in passes of eight rows; two passes of 16 rows at multiples of 256) /
// now: bf16, H 1664, 1230 active, 9 rows 32.7 / 13.2; H 3200, 5000, 22 rows 180 / 45.6; H 4736, 6000, 25 rows 441 / 72.5; fp16,
// H 4480, 3000, 4 rows 42.9 / 29.0; H 2560, 3000, 24 rows 38.4 / 25.7; fp32, H 2816, 2200, 6 rows 55.0 / 28.2; H 2048, 2500, 64 rows 268 / 66.
// Relative error against float64 before / now: bf16 and fp16 the same to six digits where h is fp32 (1.655777e-3, 2.0769e-4),
// fp32 1.93e-7 / 1.85e-7 (H 2048), 2.09e-7 / 1.94e-7 (H 4096, 3500 active).
//
// Same contraction as sparse_mlp_forward_cpu
// (sparse_transformers/csrc/sparse_mlp_op.cpp:151-161,181-186) and
// SkipMLP._forward_sparse_weight_cache (src/modeling_skip.py:114-117).
#include "st_mfma.h"

#include <atomic>
#include <type_traits>

namespace st {

constexpr int kBtThreads = 512;
constexpr int kBtWaves = kBtThreads / kWave;
constexpr int kBtRows = 16;                      // rows of x per MFMA tile (kernel 1 takes two tiles per pass)
constexpr int kBtXPad = 8;                       // padding elements per x row in LDS (spreads the banks)
constexpr int kBtTile = 32;                      // active rows per tile / K per MFMA in kernel 2
constexpr int kBtRedFloats = kBtWaves * 2 * 256; // kernel 1: 8 waves x (g,u) x 16x16, one subtile at a time
constexpr int kBtStagePitch = 72;                // kernel 2: elements per staged row (64 + 8 pad)
constexpr int kBtStageBytes = kBtTile * kBtStagePitch * 2;

typedef short bt_v4i16_t __attribute__((ext_vector_type(4)));

// Orders this wave's LDS traffic for the compiler (the hardware executes one wave's LDS operations in order).
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// kernel 1.  KSW = MFMA k-steps per wave = H / 256; HG = gated; NT = tiles of 16 rows of x (1 or 2).
// h is written as hbuf[b * ldh + row] for all 16 NT b (rows of x past B are zeros).
// ---------------------------------------------------------------------------
template <typename T, int KSW, bool HG, int NT>
__global__ __launch_bounds__(kBtThreads) void batch_gateup_kernel(
    const T *__restrict__ x, int B, int G, const T *__restrict__ gate, const T *__restrict__ up, int n_host,
    const int *__restrict__ n_dev, T *__restrict__ hbuf, int ldh, T *__restrict__ combined, long ldc, int act)
{
    constexpr int H = KSW * 256;
    // k-steps of weight loads in flight per wave (the x fragments take 4 NT KSW registers)
    constexpr int DEPTH = NT == 1 ? (KSW < 6 ? KSW : 6) : (KSW > 12 ? 4 : 5);
    // One tile of x (NT == 1) is staged in LDS by the whole block with full-line loads and read from there;
    // two tiles do not fit, so every wave keeps the fragments of its K slice in registers (measured 0.4-1.2 us
    // slower per launch for one tile: a fragment load touches 16 half lines).
    constexpr bool XREG = NT > 1;
    constexpr int XP = H + kBtXPad;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    T *xs = reinterpret_cast<T *>(lds_raw);                                                      // [16][XP]
    float *red = reinterpret_cast<float *>(lds_raw + (XREG ? 0 : (size_t)kBtRows * XP * 2));     // [NT][8][2][4][64]

    const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int blk = blockIdx.x;  // G: the grid's size, an argument so that it arrives preloaded

    const int n = device_count(n_host, n_dev);
    const int R = (n + G - 1) / G;             // rows per block
    const int row0 = blk * R;
    const int jcount = n - row0 < R ? n - row0 : R;
    if (jcount <= 0) return;

    const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
    const int ntile = (jcount + kBtTile - 1) / kBtTile;

    // this lane's weight rows in the two 16-row subtiles of tile t
    bool v0, v1;
    size_t o0, o1;
    auto setup = [&](int t) __attribute__((always_inline)) {
        const int j0 = t * kBtTile + r, j1 = j0 + 16;
        v0 = j0 < jcount; v1 = j1 < jcount;
        o0 = (size_t)(row0 + (v0 ? j0 : 0)) * H + 8 * q + 32 * w;
        o1 = (size_t)(row0 + (v1 ? j1 : 0)) * H + 8 * q + 32 * w;
    };
    uint4 g0[KSW], u0[KSW], g1[KSW], u1[KSW];
    auto issue = [&](int j) __attribute__((always_inline)) {
        const int col = 256 * j;   // step j of wave w covers columns 32 * (8 j + w) ..
        u0[j] = zero4; u1[j] = zero4;
        if (HG) { g0[j] = zero4; g1[j] = zero4; }
        if (v0) {                  // lanes without a row request nothing
            u0[j] = ld16(up + o0 + col);
            if (HG) g0[j] = ld16(gate + o0 + col);
        }
        if (v1) {
            u1[j] = ld16(up + o1 + col);
            if (HG) g1[j] = ld16(gate + o1 + col);
        }
    };

    // x is requested first, then the first weight loads.  XREG: lane (r, q) of wave w holds columns
    // 256 j + 32 w + 8 q .. + 7 of row 16 t + r (rows past B are zeros).
    const T *xfrag = xs + (size_t)r * XP + 8 * q + 32 * w;
    uint4 xr[XREG ? NT : 1][XREG ? KSW : 1];
    if constexpr (XREG) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const bool ok = 16 * t + r < B;
            const T *xp = x + (size_t)(ok ? 16 * t + r : 0) * H + 8 * q + 32 * w;
#pragma unroll
            for (int j = 0; j < KSW; ++j) {
                xr[t][j] = zero4;
                if (ok) xr[t][j] = ld16(xp + 256 * j);
            }
        }
        setup(0);
#pragma unroll
        for (int j = 0; j < DEPTH; ++j) issue(j);
    } else {
        // 16 rows x H/8 chunks = KSW chunks per thread; staging x waits for x alone
        constexpr int chunks = H / 8;
        uint4 xv[KSW];
#pragma unroll
        for (int i = 0; i < KSW; ++i) {
            const int idx = tid + kBtThreads * i;
            const int b = idx / chunks, c = idx - b * chunks;
            xv[i] = zero4;
            if (b < B) xv[i] = ld16(x + (size_t)b * H + c * 8);
        }
        setup(0);
#pragma unroll
        for (int j = 0; j < DEPTH; ++j) issue(j);
#pragma unroll
        for (int i = 0; i < KSW; ++i) {
            const int idx = tid + kBtThreads * i;
            const int b = idx / chunks, c = idx - b * chunks;
            *reinterpret_cast<uint4 *>(xs + (size_t)b * XP + c * 8) = xv[i];
        }
        __syncthreads();
    }

    for (int t = 0; t < ntile; ++t) {
        if (t > 0) {
            setup(t);
#pragma unroll
            for (int j = 0; j < DEPTH; ++j) issue(j);
        }

        f32x4_t dg0[NT], du0[NT], dg1[NT], du1[NT];
#pragma unroll
        for (int xt = 0; xt < NT; ++xt) {
            dg0[xt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            du0[xt] = dg0[xt]; dg1[xt] = dg0[xt]; du1[xt] = dg0[xt];
        }
#pragma unroll
        for (int j = 0; j < KSW; ++j) {
#pragma unroll
            for (int xt = 0; xt < NT; ++xt) {
                uint4 xf;
                if constexpr (XREG) xf = xr[xt][j];
                else xf = *reinterpret_cast<const uint4 *>(xfrag + 256 * j);
                du0[xt] = Mfma<T>::run(u0[j], xf, du0[xt]);
                if (HG) dg0[xt] = Mfma<T>::run(g0[j], xf, dg0[xt]);
                du1[xt] = Mfma<T>::run(u1[j], xf, du1[xt]);
                if (HG) dg1[xt] = Mfma<T>::run(g1[j], xf, dg1[xt]);
            }
            if (j + DEPTH < KSW) issue(j + DEPTH);
        }

        // sum the 8 waves' partial tiles, one 16-row subtile at a time: red[xt][w][g|u][e][lane]
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (s == 1 && jcount - t * kBtTile <= 16) break;   // the second subtile is empty (uniform)
#pragma unroll
            for (int xt = 0; xt < NT; ++xt) {
                float *mine = red + (size_t)(xt * kBtWaves + w) * 512 + lane;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (HG) mine[e * 64] = s == 0 ? dg0[xt][e] : dg1[xt][e];
                    mine[(4 + e) * 64] = s == 0 ? du0[xt][e] : du1[xt][e];
                }
            }
            __syncthreads();
            if (tid < 256 * NT) {
                // thread -> one element of a 16x16 tile: D register e of D lane dl of x tile xt
                const int xt = tid >> 8, e = (tid >> 6) & 3, dl = tid & 63;
                float sg = 0.f, su = 0.f;
#pragma unroll
                for (int ww = 0; ww < kBtWaves; ++ww) {
                    if (HG) sg += red[(size_t)(xt * kBtWaves + ww) * 512 + e * 64 + dl];
                    su += red[(size_t)(xt * kBtWaves + ww) * 512 + (4 + e) * 64 + dl];
                }
                const int j = t * kBtTile + 16 * s + 4 * (dl >> 4) + e;   // D rows are 4 * (lane / 16) + e
                const int b = 16 * xt + (dl & 15);
                if (j < jcount) {
                    const float hv = HG ? activate(sg, act) * su : activate(su, act);
                    const int row = row0 + j;
                    hbuf[(size_t)b * ldh + row] = from_float<T>(hv);
                    if (combined && b < B) {
                        combined[(size_t)b * ldc + row] = from_float<T>(hv);
                        if (HG) combined[(size_t)b * ldc + n + row] = from_float<T>(su);
                    }
                }
            }
            __syncthreads();   // red is rewritten by the next subtile / tile
        }
    }
}

// ---------------------------------------------------------------------------
// Any other hidden size: multiples of 64, and of 16 in fp32.  Where it is no multiple of 256, h stays in fp32 between the
// kernels, as it does inside the streaming kernel, which takes such shapes in passes of eight rows: HT.
//
// A step's products: D += A * B over the 16-byte chunk of the rows of A and B that each lane holds.  One MFMA for the 2-byte
// types; four of 16x16x4 for fp32 (the i-th takes element i of every lane's chunk; the sum does not mind which k share an
// instruction), summed by themselves first, in two pairs: short chains of roundings.
template <typename T> __device__ __forceinline__ f32x4_t mfma_chunk(const uint4 &a, const uint4 &b, f32x4_t c)
{
    if constexpr (__is_same(T, float)) {
        const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
        f32x4_t p = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.x), __uint_as_float(b.x), zero, 0, 0, 0);
        f32x4_t o = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.y), __uint_as_float(b.y), zero, 0, 0, 0);
        p = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.z), __uint_as_float(b.z), p, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.w), __uint_as_float(b.w), o, 0, 0, 0);
        return c + (p + o);
    } else {
        return Mfma<T>::run(a, b, c);
    }
}

// ((v0 + v1) + (v2 + v3)) + ((v4 + v5) + (v6 + v7)) of the 8 waves' values `pitch` floats apart
__device__ __forceinline__ float sum_of_waves(const float *v, int pitch)
{
    static_assert(kBtWaves == 8, "a tree of eight");
    float a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = v[(size_t)i * pitch];
    return ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
}

// Block barrier that orders LDS traffic only: loads in flight stay in flight.
__device__ __forceinline__ void bt_lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// kernel 1: the decomposition of batch_gateup_kernel (a block owns a contiguous range of active rows, its waves split the
// hidden dimension in steps of 64 bytes), the number of steps a run-time value.  SUB = 16-row subtiles per tile: one where
// a block has 16 rows at most.  Weight fragments go through a ring of register slots whose loads are unconditional (a
// branch around a load makes the compiler wait for everything in flight): lanes without a row read their block's first
// row, steps past the wave's last one read one 16-byte piece.  The ring runs on into the next tile while a tile is summed.
// XLDS: x comes from LDS; otherwise its fragments go through the ring too.
template <typename T, typename HT, bool HG, int NT, bool XLDS, int SUB>
__device__ __forceinline__ void gateup_any(const T *__restrict__ x, int B, int H, const T *__restrict__ gate,
                                           const T *__restrict__ up, int n, int row0, int jcount, HT *__restrict__ hbuf,
                                           int ldh, T *__restrict__ combined, long ldc, int act, unsigned char *lds_raw)
{
    constexpr int V = Elem<T>::kVec, W = 4 * V;                 // elements of a 16-byte chunk, of a 64-byte step
    constexpr int RING = SUB == 1 ? 6 : 4;
    constexpr int TROWS = 16 * SUB;
    constexpr int NACC = __is_same(T, float) ? 2 : 1;           // fp32: even and odd steps apart, for shorter chains of roundings
    const int XP = H + V;                                       // 16 bytes of padding per row of x in LDS spread the banks
    T *xs = reinterpret_cast<T *>(lds_raw);                                                                    // [16 NT][XP]
    float *red = reinterpret_cast<float *>(lds_raw + (XLDS ? (size_t)kBtRows * NT * XP * sizeof(T) : 0));      // [8][NT][SUB][2][4][64]

    const int tid = threadIdx.x, lane = tid & (kWave - 1), w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int steps = H / W;
    const int KS = (steps - w + kBtWaves - 1) / kBtWaves;       // of this wave (0 where there are fewer steps than waves)
    const int ntile = (jcount + TROWS - 1) / TROWS;

    uint4 wg[RING][SUB], wu[RING][SUB], xr[XLDS ? 1 : RING][XLDS ? 1 : NT];
    size_t wo[SUB];                                             // this lane's row of each subtile, elements
    auto rows_of = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < SUB; ++s) {
            const int j = t * TROWS + 16 * s + r;
            wo[s] = (size_t)(row0 + (j < jcount ? j : 0)) * H + V * q + W * w;
        }
    };
    size_t xo[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) xo[t] = (size_t)(16 * t + r < B ? 16 * t + r : 0) * H + V * q + W * w;
    auto issue = [&](int slot, int j) __attribute__((always_inline)) {
        const bool ok = j < KS;
        const size_t col = (size_t)(kBtWaves * W) * j;
#pragma unroll
        for (int s = 0; s < SUB; ++s) {
            const size_t o = ok ? wo[s] + col : (size_t)row0 * H;
            wu[slot][s] = ld16(up + o);
            if (HG) wg[slot][s] = ld16(gate + o);
        }
        if constexpr (!XLDS) {
#pragma unroll
            for (int t = 0; t < NT; ++t) xr[slot][t] = ld16(x + (ok ? xo[t] + col : 0));
        }
        __builtin_amdgcn_sched_barrier(0);                      // slots in order: the waits count on it
    };

    rows_of(0);
    if constexpr (XLDS) {
        // x first (staging waits for it alone): up to 16 chunks per thread, in groups of four
        const int chunks = H / V, total = chunks * (NT * kBtRows < B ? NT * kBtRows : B);
        uint4 xv[4][4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (4 * g * kBtThreads >= total) break;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = tid + kBtThreads * (4 * g + k);
                xv[g][k] = ld16(x + (size_t)(i < total ? i : 0) * V);
            }
        }
#pragma unroll
        for (int sl = 0; sl < RING; ++sl) issue(sl, sl);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (4 * g * kBtThreads >= total) break;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = tid + kBtThreads * (4 * g + k);
                if (i < total) *reinterpret_cast<uint4 *>(xs + (size_t)(i / chunks) * XP + (i % chunks) * V) = xv[g][k];
            }
        }
        bt_lds_barrier();
    } else {
#pragma unroll
        for (int sl = 0; sl < RING; ++sl) issue(sl, sl);
    }
    const T *xfrag = xs + (size_t)r * XP + V * q + W * w;       // rows of x past B: whatever LDS holds, for columns nobody reads

    for (int t = 0; t < ntile; ++t) {
        f32x4_t dg[NT][SUB][NACC], du[NT][SUB][NACC];
#pragma unroll
        for (int xt = 0; xt < NT; ++xt)
#pragma unroll
            for (int s = 0; s < SUB; ++s)
#pragma unroll
                for (int a = 0; a < NACC; ++a) dg[xt][s][a] = du[xt][s][a] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        for (int jb = 0; jb < KS; jb += RING) {
            const bool last = jb + RING >= KS;                  // the slots' next contents are the next tile's first steps
            if (last) rows_of(t + 1 < ntile ? t + 1 : t);
#pragma unroll
            for (int sl = 0; sl < RING; ++sl) {
                const int j = jb + sl;
                if (j < KS) {                                   // uniform; no load inside
#pragma unroll
                    for (int xt = 0; xt < NT; ++xt) {
                        uint4 xf;
                        if constexpr (XLDS) xf = *reinterpret_cast<const uint4 *>(xfrag + (size_t)16 * xt * XP + kBtWaves * W * j);
                        else xf = xr[sl][xt];
#pragma unroll
                        for (int s = 0; s < SUB; ++s) {
                            du[xt][s][sl % NACC] = mfma_chunk<T>(wu[sl][s], xf, du[xt][s][sl % NACC]);
                            if (HG) dg[xt][s][sl % NACC] = mfma_chunk<T>(wg[sl][s], xf, dg[xt][s][sl % NACC]);
                        }
                    }
                }
                issue(sl, last ? (t + 1 < ntile ? sl : KS) : j + RING);
            }
        }

        // sum the 8 waves' partial tiles: red[w][xt][s][g|u][e][lane]
        float *mine = red + (size_t)w * (NT * SUB * 512) + lane;
#pragma unroll
        for (int xt = 0; xt < NT; ++xt)
#pragma unroll
            for (int s = 0; s < SUB; ++s)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float *m = mine + (xt * SUB + s) * 512 + e * 64;
                    if constexpr (NACC == 2) {
                        if (HG) m[0] = dg[xt][s][0][e] + dg[xt][s][NACC - 1][e];
                        m[256] = du[xt][s][0][e] + du[xt][s][NACC - 1][e];
                    } else {
                        if (HG) m[0] = dg[xt][s][0][e];
                        m[256] = du[xt][s][0][e];
                    }
                }
        bt_lds_barrier();
        for (int i = tid; i < NT * SUB * 256; i += kBtThreads) {
            // one element of a 16x16 tile: D register e of D lane dl of (x tile, subtile)
            const int tile = i >> 8, xt = tile / SUB, s = tile % SUB, e = (i >> 6) & 3, dl = i & 63;
            const float *m = red + tile * 512 + e * 64 + dl;
            const float sg = HG ? sum_of_waves(m, NT * SUB * 512) : 0.f, su = sum_of_waves(m + 256, NT * SUB * 512);
            const int j = t * TROWS + 16 * s + 4 * (dl >> 4) + e;
            const int b = 16 * xt + (dl & 15);
            if (j < jcount && b < B) {
                const float hv = HG ? activate(sg, act) * su : activate(su, act);
                const int row = row0 + j;
                hbuf[(size_t)b * ldh + row] = from_float<HT>(hv);
                if (combined) {
                    combined[(size_t)b * ldc + row] = from_float<T>(hv);
                    if (HG) combined[(size_t)b * ldc + n + row] = from_float<T>(su);
                }
            }
        }
        if (t + 1 < ntile) bt_lds_barrier();                    // red is rewritten by the next tile
    }
}

template <typename T, typename HT, bool HG, int NT, bool XLDS>
__global__ __launch_bounds__(kBtThreads) void batch_gateup_any_kernel(
    const T *__restrict__ x, int B, int H, int G, const T *__restrict__ gate, const T *__restrict__ up, int n_host,
    const int *__restrict__ n_dev, HT *__restrict__ hbuf, int ldh, T *__restrict__ combined, long ldc, int act)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int n = device_count(n_host, n_dev);
    const int R = (n + G - 1) / G;
    const int row0 = (int)blockIdx.x * R;
    const int jcount = n - row0 < R ? n - row0 : R;
    if (jcount <= 0) return;
    if (R <= 16) gateup_any<T, HT, HG, NT, XLDS, 1>(x, B, H, gate, up, n, row0, jcount, hbuf, ldh, combined, ldc, act, lds_raw);
    else gateup_any<T, HT, HG, NT, XLDS, 2>(x, B, H, gate, up, n, row0, jcount, hbuf, ldh, combined, ldc, act, lds_raw);
}

// kernel 2 for fp32, on MFMAs of 16x16x4: K runs down the rows of the packed down matrix, and an instruction takes one element
// of every lane's 16-byte chunk, so that the operand needs no transposition: lane (c, q) holds four columns from 4 c on of one
// of four rows, the i-th MFMA multiplies the columns 4 c + i of the four.  Block = (64 columns, row split); a wave takes chunks
// of 16 rows, kBtDownRing of them in flight, and sums each by itself first (the chain of roundings is then as long as a wave
// has chunks).  partial[(rs * B + b) * H + col].
constexpr int kBtDownRing = 4, kBtDownRows = 16;

template <int NT>
__global__ __launch_bounds__(kBtThreads) void batch_down_f32_kernel(
    const float *__restrict__ hbuf, int ldh, int B, const float *__restrict__ down, int H, int n_host,
    const int *__restrict__ n_dev, float *__restrict__ partial, int CG, int RS)
{
    constexpr int V = 4, COLS = 16 * V;
    constexpr int PITCH = 256 + 16;                             // floats per element of a chunk: spreads the banks
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15, q = lane >> 4;
    const int cg = blockIdx.x % CG, rs = blockIdx.x / CG;
    const int col0 = cg * COLS;

    const int n = device_count(n_host, n_dev);
    const int NC = (n + kBtDownRows - 1) / kBtDownRows;
    const int CPS = (NC + RS - 1) / RS;
    const int c_begin = rs * CPS;
    const int c_end = c_begin + CPS < NC ? c_begin + CPS : NC;

    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t acc[NT][V];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < V; ++i) acc[t][i] = zero;

    if (c_begin + w < c_end) {
        uint4 d[kBtDownRing][4];
        float hv[kBtDownRing][NT][4];
        const int col = col0 + V * c16 < H ? col0 + V * c16 : 0;     // lanes past the last column read the first and store nothing
        const float *hp[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) hp[t] = hbuf + (size_t)(16 * t + c16 < B ? 16 * t + c16 : 0) * ldh + 4 * q;
        // lane (c, q) takes rows 4 q .. 4 q + 3 of a chunk; chunks past the split's last one read one 16-byte piece
        auto issue = [&](int slot, int c) __attribute__((always_inline)) {
            const bool ok = c < c_end;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                int row = c * kBtDownRows + 4 * q + k;
                row = row < n ? row : n - 1;
                d[slot][k] = ld16(down + (ok ? (size_t)row * H + col : 0));
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const float4 v = *reinterpret_cast<const float4 *>(hp[t] + (ok ? c * kBtDownRows : 0));
                hv[slot][t][0] = v.x; hv[slot][t][1] = v.y; hv[slot][t][2] = v.z; hv[slot][t][3] = v.w;
            }
            __builtin_amdgcn_sched_barrier(0);                  // slots in order: the waits count on it
        };
#pragma unroll
        for (int sl = 0; sl < kBtDownRing; ++sl) issue(sl, c_begin + w + kBtWaves * sl);
        for (int cb = c_begin + w; cb < c_end; cb += kBtWaves * kBtDownRing) {
#pragma unroll
            for (int sl = 0; sl < kBtDownRing; ++sl) {
                const int c = cb + kBtWaves * sl;
                if (c < c_end) {                                // uniform; no load inside
                    if ((c + 1) * kBtDownRows > n) {            // rows past the count: neither h nor the weights hold anything
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            if (c * kBtDownRows + 4 * q + k >= n) {
                                d[sl][k] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
                                for (int t = 0; t < NT; ++t) hv[sl][t][k] = 0.f;
                            }
                        }
                    }
                    f32x4_t p[2][NT][V];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float f[V] = {__uint_as_float(d[sl][k].x), __uint_as_float(d[sl][k].y),
                                            __uint_as_float(d[sl][k].z), __uint_as_float(d[sl][k].w)};
#pragma unroll
                        for (int i = 0; i < V; ++i)
#pragma unroll
                            for (int t = 0; t < NT; ++t)
                                p[k & 1][t][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(hv[sl][t][k], f[i], k > 1 ? p[k & 1][t][i] : zero, 0, 0, 0);
                    }
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int i = 0; i < V; ++i) acc[t][i] += p[0][t][i] + p[1][t][i];
                }
                issue(sl, c + kBtWaves * kBtDownRing);
            }
        }
    }

    // sum the 8 waves' accumulators through LDS: red[w][t][i][e][lane]; D rows are the rows of x
    float *red = reinterpret_cast<float *>(lds_raw);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < V; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[(((size_t)w * NT + t) * V + i) * PITCH + e * 64 + lane] = acc[t][i][e];
    bt_lds_barrier();
#pragma unroll
    for (int m = 0; m < NT * 16 * COLS / kBtThreads; ++m) {
        const int idx = tid + kBtThreads * m;
        const int b = idx / COLS, cc = idx % COLS, i = cc % V, c = cc / V;
        if (b < B && col0 + cc < H)
            partial[((size_t)rs * B + b) * H + col0 + cc] =
                sum_of_waves(red + ((b >> 4) * V + i) * PITCH + (b & 3) * 64 + 16 * ((b & 15) >> 2) + c, NT * V * PITCH);
    }
}

// Eight fp32 values of h as three 16-bit operands each that sum to them, for the MFMAs of kernel 2.  bf16 has fp32's range:
// three parts of eight bits are the value.  fp16 has not: each row of x is scaled, chunk by chunk, by a power of two that puts
// its largest finite exponent at 2^14 (one multiply-add per result takes it back), where three parts hold all 24 bits of
// what is within 2^16 of the row's largest element and 2^-39 of the largest below that.  An infinity or NaN is its own first part.
template <typename T> struct SplitH;
template <> struct SplitH<bf16_t> {
    static constexpr bool kScaled = false;
    static __device__ __forceinline__ void run(const float (&h)[8], float, uint4 (&part)[3])
    {
        uint32_t w[3][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t b[2][3];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const float v = h[2 * i + k];
                const bool fin = (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u;
                b[k][0] = fin ? __float_as_uint(v) & 0xffff0000u : (uint32_t)from_float<bf16_t>(v).bits << 16;
                const float r1 = fin ? v - __uint_as_float(b[k][0]) : 0.f;
                b[k][1] = __float_as_uint(r1) & 0xffff0000u;
                b[k][2] = __float_as_uint(r1 - __uint_as_float(b[k][1]));
            }
#pragma unroll
            for (int p = 0; p < 3; ++p) w[p][i] = __builtin_amdgcn_perm(b[1][p], b[0][p], 0x07060302u);   // the high halves
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) part[p] = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
    }
};
template <> struct SplitH<f16_t> {
    static constexpr bool kScaled = true;
    static __device__ __forceinline__ void run(const float (&h)[8], float scale, uint4 (&part)[3])
    {
        uint32_t w[3][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            _Float16 b[2][3];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const float v = h[2 * i + k] * scale;
                const bool fin = (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u;
                b[k][0] = (_Float16)v;
                // (what is too small for a part keeps its sign, for an infinite weight to meet)
                if (b[k][0] == (_Float16)0.f && h[2 * i + k] != 0.f) b[k][0] = (_Float16)copysignf(0x1p-24f, h[2 * i + k]);
                const float r1 = fin ? v - (float)b[k][0] : 0.f;
                b[k][1] = (_Float16)r1;
                b[k][2] = (_Float16)(r1 - (float)b[k][1]);
            }
#pragma unroll
            for (int p = 0; p < 3; ++p)
                w[p][i] = (uint32_t)__builtin_bit_cast(uint16_t, b[0][p]) | (uint32_t)__builtin_bit_cast(uint16_t, b[1][p]) << 16;
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) part[p] = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
    }
};

// largest value over the four lanes that hold one row of an MFMA operand (lane % 16)
__device__ __forceinline__ uint32_t row_max_u32(uint32_t v)
{
    const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v = a[0] > a[1] ? a[0] : a[1];
    const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return b[0] > b[1] ? b[0] : b[1];
}

// ---------------------------------------------------------------------------
// kernel 2.  Block = (column group cg, row split rs); NP = 64-column pieces per
// block; NX = tiles of 16 rows of x; HT = the type h is held in (the storage type behind
// batch_gateup_kernel, fp32 behind batch_gateup_any_kernel: three MFMAs per tile and chunk of rows then).  Where h is scaled
// (fp16) the operands change places: a row of x is then a column of D, whose scale is the lane's own.  With fp32 h two forms do not
// fit the registers beside two chunks in flight: bf16 with two tiles of x keeps 112 bytes a lane of the chunks' h in scratch,
// fp16 with two pieces spills 12 registers (of batch_gateup_any_kernel, fp32 with two tiles and x from memory three).
// partial[(rs * ldb + b) * H + col], fp32.
// ---------------------------------------------------------------------------
template <typename T, typename HT, int NP, int NX>
__global__ __launch_bounds__(kBtThreads) void batch_down_kernel(
    const HT *__restrict__ hbuf, int ldh, int B, const T *__restrict__ down, int H, int n_host,
    const int *__restrict__ n_dev, float *__restrict__ partial, int CG, int RS, int ldb)
{
    constexpr int NT = NP * 4;   // 16-column tiles per block
    constexpr bool WIDE = __is_same(HT, float), SCALED = WIDE && SplitH<T>::kScaled;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid >> 6;
    const int c16 = lane & 15, q = lane >> 4;
    const int cg = blockIdx.x % CG, rs = blockIdx.x / CG;
    const int col0 = cg * NP * 64;

    const int n = device_count(n_host, n_dev);
    const int NC = (n + kBtTile - 1) / kBtTile;        // chunks of 32 rows
    const int CPS = (NC + RS - 1) / RS;
    const int c_begin = rs * CPS;
    const int c_end = c_begin + CPS < NC ? c_begin + CPS : NC;

    T *stage = reinterpret_cast<T *>(lds_raw + (size_t)w * kBtStageBytes);

    // WIDE: the lower parts' products by themselves, and left out where they are not finite: an infinite weight meets zeros
    // there, and what it makes of the result shows in the first parts' products
    f32x4_t acc[NX][NT], low[WIDE ? NX : 1][WIDE ? NT : 1];
#pragma unroll
    for (int t = 0; t < NX; ++t)
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            acc[t][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            if constexpr (WIDE) low[t][i] = acc[t][i];
        }

    typedef typename std::conditional<WIDE, uint4, uint2>::type HVec;   // four values of h
    struct Chunk { uint4 d[NP][4]; HVec hlo[NX], hhi[NX]; };
    // 8 rows x 128 bytes per load instruction
    auto load_chunk = [&](Chunk &k, int c) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            int row = c * kBtTile + (lane >> 3) + 8 * kk;
            row = row < n ? row : n - 1;
            const T *rp = down + (size_t)row * H + col0 + 8 * (lane & 7);
#pragma unroll
            for (int p = 0; p < NP; ++p) k.d[p][kk] = ld16(rp + 64 * p);
        }
        // h fragment: k-slots 0..3 <-> rows 4q..4q+3, slots 4..7 <-> rows 16+4q..16+4q+3 of the chunk
#pragma unroll
        for (int t = 0; t < NX; ++t) {
            const int b = 16 * t + c16 < B ? 16 * t + c16 : 0;
            const HT *hp = hbuf + (size_t)b * ldh + c * kBtTile + 4 * q;
            k.hlo[t] = *reinterpret_cast<const HVec *>(hp);
            k.hhi[t] = *reinterpret_cast<const HVec *>(hp + 16);
        }
    };
    auto process = [&](Chunk &k, int c) __attribute__((always_inline)) {
        if (c * kBtTile + kBtTile > n) {   // rows past the count: neither h nor the clamped weights count
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
                if (c * kBtTile + (lane >> 3) + 8 * kk >= n) {
#pragma unroll
                    for (int p = 0; p < NP; ++p) k.d[p][kk] = make_uint4(0u, 0u, 0u, 0u);
                }
        }
        constexpr int PARTS = WIDE ? 3 : 1;
        uint4 hf[NX][PARTS];
        float unscale[NX];
        if constexpr (WIDE) {
            float hv[NX][8];
#pragma unroll
            for (int t = 0; t < NX; ++t) {
                const uint32_t a[8] = {k.hlo[t].x, k.hlo[t].y, k.hlo[t].z, k.hlo[t].w, k.hhi[t].x, k.hhi[t].y, k.hhi[t].z, k.hhi[t].w};
#pragma unroll
                for (int i = 0; i < 8; ++i) hv[t][i] = __uint_as_float(a[i]);
            }
            if (c * kBtTile + kBtTile > n) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (c * kBtTile + (i < 4 ? 4 * q + i : 12 + 4 * q + i) >= n) {
#pragma unroll
                        for (int t = 0; t < NX; ++t) hv[t][i] = 0.f;
                    }
            }
#pragma unroll
            for (int t = 0; t < NX; ++t) {
                float scale = 1.f;
                if constexpr (SCALED) {
                    uint32_t e = 15u << 23;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        uint32_t x = __float_as_uint(hv[t][i]) & 0x7f800000u;
                        x = x == 0x7f800000u ? 0u : x;
                        e = e > x ? e : x;
                    }
                    e = row_max_u32(e);
                    scale = __uint_as_float((268u << 23) - e);      // 2^(141 - E)
                    unscale[t] = __uint_as_float(e - (14u << 23));  // 2^(E - 141)
                }
                SplitH<T>::run(hv[t], scale, hf[t]);
            }
        } else {
#pragma unroll
            for (int t = 0; t < NX; ++t) {
                uint32_t a[4] = {k.hlo[t].x, k.hlo[t].y, k.hhi[t].x, k.hhi[t].y};
                if (c * kBtTile + kBtTile > n) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int rlo = c * kBtTile + (i < 2 ? 4 * q + 2 * i : 16 + 4 * q + 2 * (i - 2));
                        if (rlo >= n) a[i] = 0u;
                        else if (rlo + 1 >= n) a[i] &= 0xffffu;
                    }
                }
                hf[t][0] = make_uint4(a[0], a[1], a[2], a[3]);
            }
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            wave_lds_fence();   // the previous piece's reads come first
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
                *reinterpret_cast<uint4 *>(stage + ((lane >> 3) + 8 * kk) * kBtStagePitch + 8 * (lane & 7)) = k.d[p][kk];
            wave_lds_fence();
            uint4 bf[4];
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) {
                // transposing LDS read: in its group of 16 lanes, lane j hands in four columns of row j / 4 and
                // lane i receives column i of the four rows (rows 4q.. and 16 + 4q.. of the staged piece)
                const uint16_t *sp = reinterpret_cast<const uint16_t *>(stage) +
                                     (4 * q + (c16 >> 2)) * kBtStagePitch + 16 * ct + 4 * (c16 & 3);
                const bt_v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) bt_v4i16_t *)sp);
                const bt_v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) bt_v4i16_t *)(sp + 16 * kBtStagePitch));
                bf[ct] = make_uint4((uint16_t)lo[0] | ((uint32_t)(uint16_t)lo[1] << 16),
                                    (uint16_t)lo[2] | ((uint32_t)(uint16_t)lo[3] << 16),
                                    (uint16_t)hi[0] | ((uint32_t)(uint16_t)hi[1] << 16),
                                    (uint16_t)hi[2] | ((uint32_t)(uint16_t)hi[3] << 16));
                if constexpr (!WIDE) {
#pragma unroll
                    for (int t = 0; t < NX; ++t) acc[t][p * 4 + ct] = Mfma<T>::run(hf[t][0], bf[ct], acc[t][p * 4 + ct]);
                }
            }
            if constexpr (WIDE) {
                const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
                f32x4_t d[2][NX][4];
#pragma unroll
                for (int part = PARTS - 1; part >= 0; --part)
#pragma unroll
                    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                        for (int t = 0; t < NX; ++t) {
                            const int lo = part > 0;
                            f32x4_t &sum = SCALED ? d[lo][t][ct] : lo ? low[t][p * 4 + ct] : acc[t][p * 4 + ct];
                            sum = SCALED ? Mfma<T>::run(bf[ct], hf[t][part], part != 1 ? zero : sum) : Mfma<T>::run(hf[t][part], bf[ct], sum);
                        }
                if constexpr (SCALED) {
#pragma unroll
                    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                        for (int t = 0; t < NX; ++t)
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                acc[t][p * 4 + ct][e] = fmaf(d[0][t][ct][e], unscale[t], acc[t][p * 4 + ct][e]);
                                low[t][p * 4 + ct][e] = fmaf(d[1][t][ct][e], unscale[t], low[t][p * 4 + ct][e]);
                            }
                }
            }
        }
    };

    Chunk ka, kb;
    int c = c_begin + w;
    if (c < c_end) load_chunk(ka, c);
    while (c < c_end) {
        int cn = c + kBtWaves;
        if (cn < c_end) load_chunk(kb, cn);
        process(ka, c);
        c = cn;
        if (c >= c_end) break;
        cn = c + kBtWaves;
        if (cn < c_end) load_chunk(ka, cn);
        process(kb, c);
        c = cn;
    }

    if constexpr (WIDE) {
#pragma unroll
        for (int t = 0; t < NX; ++t)
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float l = low[t][i][e];
                    acc[t][i][e] += (__float_as_uint(l) & 0x7f800000u) == 0x7f800000u ? 0.f : l;
                }
    }

    // sum the 8 waves' accumulators through LDS (reuses the staging area), one tile of x at a time
#pragma unroll
    for (int t = 0; t < NX; ++t) {
        __syncthreads();
        if constexpr (SCALED) {   // a lane holds four neighbouring columns of row lane % 16
            f32x4_t *red = reinterpret_cast<f32x4_t *>(lds_raw);   // [8][NT][64]
#pragma unroll
            for (int i = 0; i < NT; ++i) red[(w * NT + i) * 64 + lane] = acc[t][i];
            __syncthreads();
            for (int idx = tid; idx < NT * 64; idx += kBtThreads) {
                f32x4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ww = 0; ww < kBtWaves; ++ww) s += red[ww * NT * 64 + idx];
                const int tile = idx >> 6, dl = idx & 63, b = 16 * t + (dl & 15);
                if (b < B) *reinterpret_cast<f32x4_t *>(partial + ((size_t)rs * ldb + b) * H + col0 + 16 * tile + 4 * (dl >> 4)) = s;
            }
        } else {
            float *red = reinterpret_cast<float *>(lds_raw);   // [8][NT][4][64]
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) red[((size_t)(w * NT + i) * 4 + e) * 64 + lane] = acc[t][i][e];
            __syncthreads();
#pragma unroll
            for (int m = 0; m < NT * 256 / kBtThreads; ++m) {
                const int idx = tid + kBtThreads * m;
                float s = 0.f;
#pragma unroll
                for (int ww = 0; ww < kBtWaves; ++ww) s += red[(size_t)ww * NT * 256 + idx];
                const int tile = idx >> 8, e = (idx >> 6) & 3, dl = idx & 63;
                const int b = 16 * t + 4 * (dl >> 4) + e;   // D rows are the rows of x
                if (b < B) partial[((size_t)rs * ldb + b) * H + col0 + 16 * tile + (dl & 15)] = s;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// kernel 3, and the GEMM kernels' third: the splits' partial rows, in their order (more than sixteen: first the z-th and the
// (z + U)-th).  A round trip and little else: a thread takes four neighbouring results and has all splits' loads of them in flight
// (U: how many, 16 at most at once).  Before, the batch kernels' went through mlp_reduce_kernel, whose blocks deal 256 partial
// rows to sixteen groups of threads, and the GEMM kernels' through a loop that waited for each split.
// Whole forward, us, before / now: batch kernels, 8 rows, H 4096, 3584 active 26.6 / 25.5; 16 rows, H 3072, 5900 33.3 / 32.4; 30
// rows, H 4096, 2500 31.1 / 28.9; fp32, 8 rows, H 2048, 2500 24.6 / 23.0; GEMM kernels, 77 rows, H 2560, twelve splits 34.0 / 32.7,
// 39 x 1920, sixteen 22.0 / 21.0.  Fewer than 16384 results are too few threads for that (4 rows, H 3072 24.9 / 25.1; 3 rows,
// H 1152 11.7 / 11.9): the batch kernels keep the dealt form there.
// ---------------------------------------------------------------------------
template <typename T, int U>
__global__ __launch_bounds__(256) void split_reduce_kernel(const float *__restrict__ partials, int splits, size_t stride,
                                                           size_t total, int threads, T *__restrict__ out)
{
    const size_t i4 = ((size_t)blockIdx.x * threads + threadIdx.x) * 4;
    if (i4 >= total) return;
    const float *const p = partials + i4;
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const float4 *>(p + (size_t)(u < splits ? u : splits - 1) * stride);
    if (splits > U) {
        float4 w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = *reinterpret_cast<const float4 *>(p + (size_t)(U + u < splits ? U + u : splits - 1) * stride);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = U + u < splits;
            v[u].x = in ? v[u].x + w[u].x : v[u].x; v[u].y = in ? v[u].y + w[u].y : v[u].y;
            v[u].z = in ? v[u].z + w[u].z : v[u].z; v[u].w = in ? v[u].w + w[u].w : v[u].w;
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    float4 s = v[0];
#pragma unroll
    for (int u = 1; u < U; ++u) {   // (selects: with branches the last loads go out behind the first sums)
        const bool in = u < splits;
        s.x = in ? s.x + v[u].x : s.x; s.y = in ? s.y + v[u].y : s.y;
        s.z = in ? s.z + v[u].z : s.z; s.w = in ? s.w + v[u].w : s.w;
    }
    T *const o = out + i4;
    if constexpr (sizeof(T) == 2) {
        if ((reinterpret_cast<uintptr_t>(out) & 7) == 0) {
            const uint32_t lo = (uint32_t)from_float<T>(s.x).bits | ((uint32_t)from_float<T>(s.y).bits << 16);
            const uint32_t hi = (uint32_t)from_float<T>(s.z).bits | ((uint32_t)from_float<T>(s.w).bits << 16);
            *reinterpret_cast<uint2 *>(o) = make_uint2(lo, hi);
            return;
        }
    }
    o[0] = from_float<T>(s.x); o[1] = from_float<T>(s.y); o[2] = from_float<T>(s.z); o[3] = from_float<T>(s.w);
}

template <typename T>
static int split_reduce_t(const float *partials, int splits, size_t stride, size_t total, void *out, hipStream_t stream)
{
    ProfScope ps(ST_K_MLP_REDUCE, stream);
    const size_t quads = total / 4;
    const int threads = quads >= (size_t)256 * device_cu_count() || splits <= 4 ? 256 : 64;   // (no CU without a block)
    auto go = [&](auto kern) {
        ST_LAUNCH(ps, kern, dim3((unsigned)((quads + threads - 1) / threads)), dim3(threads), 0, stream, partials, splits, stride,
                  total, threads, static_cast<T *>(out));
    };
    const int u = splits <= 16 ? splits : (splits + 1) / 2;   // (32 splits at most; a load too many reads the last split again)
    if (u <= 2) go(split_reduce_kernel<T, 2>);
    else if (u <= 3) go(split_reduce_kernel<T, 3>);
    else if (u <= 4) go(split_reduce_kernel<T, 4>);
    else if (u <= 5) go(split_reduce_kernel<T, 5>);
    else if (u <= 6) go(split_reduce_kernel<T, 6>);
    else if (u <= 8) go(split_reduce_kernel<T, 8>);
    else if (u <= 10) go(split_reduce_kernel<T, 10>);
    else if (u <= 12) go(split_reduce_kernel<T, 12>);
    else go(split_reduce_kernel<T, 16>);
    ST_HIP(hipGetLastError());
    return ST_OK;
}

int launch_split_reduce(int dtype, const float *partials, int splits, size_t stride, size_t total, void *out, hipStream_t stream)
{
    return dtype == ST_F32   ? split_reduce_t<float>(partials, splits, stride, total, out, stream)
           : dtype == ST_F16 ? split_reduce_t<f16_t>(partials, splits, stride, total, out, stream)
                             : split_reduce_t<bf16_t>(partials, splits, stride, total, out, stream);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct BatchShape { int ksw, np, cg, rs; bool special; };
constexpr int kBtMaxH = 16384;   // 2-byte elements; 8192 in fp32

// Hidden sizes with kernels of their own (2048 / 3072 / 4096, 2-byte types: what follows describes their launches), and any
// other that is a multiple of 64 (16 in fp32).
static bool batch_shape(int dtype, int H, BatchShape &s)
{
    const int row = H * (dtype == ST_F32 ? 4 : 2);
    if (row % (dtype == ST_F32 ? 64 : 128) != 0 || H < 16 || row > 2 * kBtMaxH) return false;
    s.ksw = H / 256;
    s.special = dtype != ST_F32 && H % 256 == 0 && (s.ksw == 8 || s.ksw == 12 || s.ksw == 16);
    const int pieces = H / 64;
    s.np = pieces % 3 == 0 ? 3 : 2;   // 4 pieces with two chunks in flight would not fit the register file
    s.cg = pieces / s.np;
    s.rs = s.cg ? device_cu_count() / s.cg : 1;
    if (s.rs < 1) s.rs = 1;
    if (s.rs > 32) s.rs = 32;
    return true;
}

// Few rows at small hidden sizes stay with the streaming kernel, which takes four rows of 16 bits, or eight of fp32, in one pass
// and is one launch (2.5 us of the host's, who sets the pace there) less.  Whole forward, us, streaming / batch kernels: fp16,
// three rows, H 384, 768 active 11.0 / 11.2; H 640, 1280 11.6 / 11.5; H 896, 1760 12.4 / 12.1; H 1152, 2304 16.1 / 12.7; five
// rows, H 384 13.3 / 11.3.  fp32, three or four rows, H 1024, 1500 active 12.8 / 15.3; H 1536, 1200 16.5 / 17.0; H 1792, 1280
// 17.5 / 18.9; H 2048, 2500 26.4 / 23.5; seven, H 512, 1024 12.2 / 11.7; H 1024, 672 14.4 / 13.7 (three layers of a module
// with their masks: 84.9 / 93.0 from the host); H 1536, 1002 20.3 / 17.5; twelve, H 512, 1024 21.8 / 11.9.
bool batch_supported(int dtype, int B, int H)
{
    BatchShape s;
    if (!batch_shape(dtype, H, s)) return false;
    if (dtype == ST_F32) return !(B <= 4 && H < 2048) && !(B <= 8 && H <= 1024);
    return s.special || !(B <= 4 && H < 1024);
}

static int64_t batch_ldh(int64_t n) { return (n + kBtTile - 1) / kBtTile * kBtTile; }

// h of up to 32 rows of x, fp32
static int64_t batch_h_bytes(int64_t n) { return ((int64_t)2 * kBtRows * batch_ldh(n) * 4 + 255) & ~(int64_t)255; }

int64_t batch_workspace_bytes(int64_t H, int64_t n)
{
    return batch_h_bytes(n) + (int64_t)32 * 2 * kBtRows * H * 4;   // and as many row splits of their partial rows
}

template <typename T, int KSW, bool HG, int NT>
static int launch_gateup(const T *x, int B, const T *gate, const T *up, int n, const int *n_dev, T *hbuf, int ldh,
                         T *comb, long ldc, int act, hipStream_t stream)
{
    auto kern = batch_gateup_kernel<T, KSW, HG, NT>;
    const size_t lds = (NT == 1 ? (size_t)kBtRows * (KSW * 256 + kBtXPad) * 2 : 0) + (size_t)NT * kBtRedFloats * 4;
    static std::atomic<bool> attr_set{false};   // (setting the attribute twice from two threads is harmless)
    if (!attr_set.load(std::memory_order_acquire)) {
        ST_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)lds));
        attr_set.store(true, std::memory_order_release);
    }
    ProfScope ps(ST_K_MLP_BATCH_GATEUP, stream);
    const int G = device_cu_count();
    ST_LAUNCH(ps, kern, dim3(G), dim3(kBtThreads), lds, stream, x, B, G, gate, up, n, n_dev, hbuf,
                       ldh, comb, ldc, act);
    return ST_OK;
}

// LDS of kernel 1 for any hidden size: the sums, and x where both fit
constexpr int kBtMaxLds = 160 * 1024;
static size_t any_red_bytes(int nt) { return (size_t)kBtWaves * nt * 2 * 512 * 4; }

template <typename T, typename HT, bool HG, int NT, bool XLDS>
static int launch_gateup_any(const T *x, int B, int H, const T *gate, const T *up, int n, const int *n_dev, HT *hbuf,
                             int ldh, T *comb, long ldc, int act, hipStream_t stream)
{
    auto kern = batch_gateup_any_kernel<T, HT, HG, NT, XLDS>;
    const size_t lds = any_red_bytes(NT) + (XLDS ? (size_t)kBtRows * NT * (H * sizeof(T) + 16) : 0);
    const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), kBtMaxLds);
    if (rc != ST_OK) return rc;
    ProfScope ps(ST_K_MLP_BATCH_GATEUP, stream);
    const int G = device_cu_count();
    ST_LAUNCH(ps, kern, dim3(G), dim3(kBtThreads), lds, stream, x, B, H, G, gate, up, n, n_dev, hbuf, ldh, comb, ldc, act);
    ST_HIP(hipGetLastError());
    return ST_OK;
}

template <typename T, typename HT, int NP, int NX>
static int launch_down(const HT *hbuf, int ldh, int B, const T *down, int H, int n, const int *n_dev, float *partial,
                       int cg, int rs, int ldb, hipStream_t stream)
{
    auto kern = batch_down_kernel<T, HT, NP, NX>;
    const size_t red = (size_t)kBtWaves * NP * 4 * 256 * 4, stage = (size_t)kBtWaves * kBtStageBytes;
    const size_t lds = red > stage ? red : stage;
    const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), kBtMaxLds);
    if (rc != ST_OK) return rc;
    ProfScope ps(ST_K_MLP_BATCH_DOWN, stream);
    ST_LAUNCH(ps, kern, dim3(cg * rs), dim3(kBtThreads), lds, stream, hbuf, ldh, B, down, H, n, n_dev, partial, cg, rs, ldb);
    ST_HIP(hipGetLastError());
    return ST_OK;
}

template <int NT>
static int launch_down_f32(const float *hbuf, int ldh, int B, const float *down, int H, int n, const int *n_dev,
                           float *partial, int cg, int rs, hipStream_t stream)
{
    auto kern = batch_down_f32_kernel<NT>;
    const size_t lds = (size_t)kBtWaves * NT * 4 * (256 + 16) * 4;
    const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), kBtMaxLds);
    if (rc != ST_OK) return rc;
    ProfScope ps(ST_K_MLP_BATCH_DOWN, stream);
    ST_LAUNCH(ps, kern, dim3(cg * rs), dim3(kBtThreads), lds, stream, hbuf, ldh, B, down, H, n, n_dev, partial, cg, rs);
    ST_HIP(hipGetLastError());
    return ST_OK;
}

template <typename T, typename HT, int NT>
static int launch_any_pass(const T *x, int B, int H, const T *gate, const T *up, const T *down, int n, const int *n_dev,
                           HT *hbuf, int ldh, float *partial, T *comb, long ldc, int act, int has_gate, int *splits,
                           hipStream_t stream)
{
    const bool xlds = any_red_bytes(NT) + (size_t)kBtRows * NT * (H * sizeof(T) + 16) <= (size_t)kBtMaxLds;
    int rc;
    if (xlds)
        rc = has_gate ? launch_gateup_any<T, HT, true, NT, true>(x, B, H, gate, up, n, n_dev, hbuf, ldh, comb, ldc, act, stream)
                      : launch_gateup_any<T, HT, false, NT, true>(x, B, H, gate, up, n, n_dev, hbuf, ldh, comb, ldc, act, stream);
    else
        rc = has_gate ? launch_gateup_any<T, HT, true, NT, false>(x, B, H, gate, up, n, n_dev, hbuf, ldh, comb, ldc, act, stream)
                      : launch_gateup_any<T, HT, false, NT, false>(x, B, H, gate, up, n, n_dev, hbuf, ldh, comb, ldc, act, stream);
    if (rc != ST_OK) return rc;
    // 64-column pieces per block: what the registers hold beside the accumulators
    const int pieces = (H + 63) / 64;
    const int np = __is_same(T, float) ? 1 : __is_same(HT, float) ? (NT == 1 && pieces % 2 == 0 ? 2 : 1)
                                                                  : NT == 1 && pieces % 3 == 0 ? 3 : 2;
    const int cg = pieces / np;
    int rs = device_cu_count() / cg;
    rs = *splits = rs < 1 ? 1 : rs > 32 ? 32 : rs;
    if constexpr (__is_same(T, float)) {
        return launch_down_f32<NT>(hbuf, ldh, B, down, H, n, n_dev, partial, cg, rs, stream);
    } else if constexpr (__is_same(HT, float)) {
        return np == 2 ? launch_down<T, HT, NT == 1 ? 2 : 1, NT>(hbuf, ldh, B, down, H, n, n_dev, partial, cg, rs, B, stream)
                       : launch_down<T, HT, 1, NT>(hbuf, ldh, B, down, H, n, n_dev, partial, cg, rs, B, stream);
    } else {
        return np == 3 ? launch_down<T, HT, NT == 1 ? 3 : 2, NT>(hbuf, ldh, B, down, H, n, n_dev, partial, cg, rs, B, stream)
                       : launch_down<T, HT, 2, NT>(hbuf, ldh, B, down, H, n, n_dev, partial, cg, rs, B, stream);
    }
}

// Kernel 3 for rows [rs][ldb][H].
static int launch_batch_reduce(int dtype, const float *partial, int rs, int ldb, int B, int H, void *out, hipStream_t stream)
{
    if ((size_t)B * H < 16384) return launch_mlp_reduce(dtype, partial, rs, ldb, B, H, out, stream);
    return launch_split_reduce(dtype, partial, rs, (size_t)ldb * H, (size_t)B * H, out, stream);
}

// One pass over the weights per 32 rows of x; HT: the type h is held in.
template <typename T, typename HT>
static int launch_batch_any(const void *x_, int B, int H, const void *gate_, const void *up_, const void *down_, int n,
                            const int *n_dev, void *out_, void *comb_, long ldc, void *workspace, int act, int has_gate,
                            hipStream_t stream)
{
    const int ldh = (int)batch_ldh(n);
    HT *hbuf = static_cast<HT *>(workspace);
    float *partial = reinterpret_cast<float *>(static_cast<unsigned char *>(workspace) + batch_h_bytes(n));
    const T *gate = static_cast<const T *>(gate_), *up = static_cast<const T *>(up_), *down = static_cast<const T *>(down_);
    const int dtype = __is_same(T, float) ? ST_F32 : __is_same(T, f16_t) ? ST_F16 : ST_BF16;
    for (int b0 = 0; b0 < B; b0 += 2 * kBtRows) {
        const int bc = B - b0 < 2 * kBtRows ? B - b0 : 2 * kBtRows;
        const T *x = static_cast<const T *>(x_) + (size_t)b0 * H;
        T *comb = comb_ ? static_cast<T *>(comb_) + (size_t)b0 * ldc : nullptr;
        int rs = 1;
        int rc = bc > kBtRows ? launch_any_pass<T, HT, 2>(x, bc, H, gate, up, down, n, n_dev, hbuf, ldh, partial, comb, ldc, act,
                                                          has_gate, &rs, stream)
                              : launch_any_pass<T, HT, 1>(x, bc, H, gate, up, down, n, n_dev, hbuf, ldh, partial, comb, ldc, act,
                                                          has_gate, &rs, stream);
        if (rc != ST_OK) return rc;
        rc = launch_batch_reduce(dtype, partial, rs, bc, bc, H, static_cast<T *>(out_) + (size_t)b0 * H, stream);
        if (rc != ST_OK) return rc;
    }
    return ST_OK;
}

template <typename T>
static int launch_batch_t(const void *x_, int B, int H, const void *gate_, const void *up_, const void *down_, int n,
                          const int *n_dev, void *out_, void *comb_, long ldc, void *workspace, int act, int has_gate,
                          hipStream_t stream)
{
    BatchShape s;
    constexpr int dtype = __is_same(T, f16_t) ? ST_F16 : ST_BF16;
    ST_REQUIRE(batch_shape(dtype, H, s), "st_mlp_forward: hidden size %d is not supported by the batch kernels", H);
    if (!s.special)
        return H % 256 == 0 ? launch_batch_any<T, T>(x_, B, H, gate_, up_, down_, n, n_dev, out_, comb_, ldc, workspace, act,
                                                     has_gate, stream)
                            : launch_batch_any<T, float>(x_, B, H, gate_, up_, down_, n, n_dev, out_, comb_, ldc, workspace, act,
                                                         has_gate, stream);
    const int ldh = (int)batch_ldh(n);
    T *hbuf = static_cast<T *>(workspace);
    float *partial = reinterpret_cast<float *>(static_cast<unsigned char *>(workspace) + batch_h_bytes(n));
    const T *gate = static_cast<const T *>(gate_), *up = static_cast<const T *>(up_);
    const T *down = static_cast<const T *>(down_);
    const int pass_rows = 2 * kBtRows;   // one pass over the weights per 32 rows of x
    for (int b0 = 0; b0 < B; b0 += pass_rows) {
        const int bc = B - b0 < pass_rows ? B - b0 : pass_rows;
        const T *x = static_cast<const T *>(x_) + (size_t)b0 * H;
        T *comb = comb_ ? static_cast<T *>(comb_) + (size_t)b0 * ldc : nullptr;
        int rc;
#define ST_BT_GATEUP(KSW)                                                                                              \
    rc = bc > kBtRows                                                                                                 \
             ? (has_gate ? launch_gateup<T, KSW, true, 2>(x, bc, gate, up, n, n_dev, hbuf, ldh, comb, ldc, act, stream)   \
                         : launch_gateup<T, KSW, false, 2>(x, bc, gate, up, n, n_dev, hbuf, ldh, comb, ldc, act, stream)) \
             : (has_gate ? launch_gateup<T, KSW, true, 1>(x, bc, gate, up, n, n_dev, hbuf, ldh, comb, ldc, act, stream)   \
                         : launch_gateup<T, KSW, false, 1>(x, bc, gate, up, n, n_dev, hbuf, ldh, comb, ldc, act, stream))
        if (s.ksw == 8) ST_BT_GATEUP(8);
        else if (s.ksw == 12) ST_BT_GATEUP(12);
        else ST_BT_GATEUP(16);
#undef ST_BT_GATEUP
        if (rc != ST_OK) return rc;
        ST_HIP(hipGetLastError());
        // kernel 2 takes both tiles of x in one pass with two 64-column pieces per block (three would not leave
        // registers for a second set of accumulators); kernel 3 sums the row splits' partial rows
        // [rs][16 or 32][H] in a fixed order
        T *out = static_cast<T *>(out_) + (size_t)b0 * H;
        int rs = s.rs, nbrows = kBtRows;
        if (bc > kBtRows) {
            const int cg = H / 128;
            rs = device_cu_count() / cg;
            rs = rs < 1 ? 1 : (rs > 16 ? 16 : rs);
            nbrows = 2 * kBtRows;
            rc = launch_down<T, T, 2, 2>(hbuf, ldh, bc, down, H, n, n_dev, partial, cg, rs, nbrows, stream);
        } else {
            rc = s.np == 3 ? launch_down<T, T, 3, 1>(hbuf, ldh, bc, down, H, n, n_dev, partial, s.cg, s.rs, nbrows, stream)
                           : launch_down<T, T, 2, 1>(hbuf, ldh, bc, down, H, n, n_dev, partial, s.cg, s.rs, nbrows, stream);
        }
        if (rc != ST_OK) return rc;
        ST_HIP(hipGetLastError());
        rc = launch_batch_reduce(dtype, partial, rs, nbrows, bc, H, out, stream);
        if (rc != ST_OK) return rc;
    }
    return ST_OK;
}

int launch_batch(int dtype, const void *x, int B, int H, const void *gate, const void *up, const void *down, int n,
                 const int *n_dev, void *out, void *comb, long ldc, void *workspace, int act, int has_gate,
                 hipStream_t stream)
{
    if (dtype == ST_F32)
        return launch_batch_any<float, float>(x, B, H, gate, up, down, n, n_dev, out, comb, ldc, workspace, act, has_gate, stream);
    if (dtype == ST_F16)
        return launch_batch_t<f16_t>(x, B, H, gate, up, down, n, n_dev, out, comb, ldc, workspace, act, has_gate, stream);
    return launch_batch_t<bf16_t>(x, B, H, gate, up, down, n, n_dev, out, comb, ldc, workspace, act, has_gate, stream);
}

}  // namespace st
