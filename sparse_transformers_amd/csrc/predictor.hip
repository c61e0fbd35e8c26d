// LoRA importance predictor -> threshold mask -> union over the batch rows.
//
//   kernel 1  t[b,k]   = <x[b,:], A[k,:]>            one wave per rank row k
//   kernel 2  s[b,i]   = <t[b,:], Bm[i,:]>           LPR lanes per row i
//             mask[i]  = any_b( s[b,i] >= thr )      written as one byte per i
//
// The rank-r intermediate stays in fp32.  Replaces FastLoRAProjection.forward
// (src/modeling_skip.py:52-53) and the "naive" branch + any(dim=0) of
// SkipDecoderLayer._compute_binary_mask (src/modeling_skip.py:204-207,214).
#include "st_common.h"

namespace st {

constexpr int kPredBTile = 8;
constexpr int kPredDownThreads = 256;
constexpr int kPredDownUnroll = 2;  // chunks per thread issued together

// One block per rank row k: all loads of the row (and of x) are issued before
// any arithmetic, so the kernel costs one memory round trip.
// BT = rows of x per pass (1 for single-row decode, so that nothing is requested twice).
// (tab: several layers of equal shape at once, grid dimension y; x [layers,B,H], t [layers,B,r])
// CLEAR: the mask too, for a second kernel that only switches bytes of it on.  A form of its own: as a run-time case in the
// eight-row form this kernel took 4.4 and 3.8 us on two machines (H 3072, rank 128, four rows), without it 3.8 and 3.6.
template <typename T, int BT, bool CLEAR, typename Tab>
__global__ __launch_bounds__(kPredDownThreads) void predictor_down_kernel(const T *__restrict__ x, int B, int H,
                                                                          const T *__restrict__ A, int r,
                                                                          float *__restrict__ t, int round_storage,
                                                                          uint8_t *__restrict__ mask, int I, Tab tab)
{
    if constexpr (Tab::kLayers) {
        A = static_cast<const T *>(tab.l[blockIdx.y].A);
        if (CLEAR) mask = tab.l[blockIdx.y].mask;
        x += (size_t)blockIdx.y * B * H;
        t += (size_t)blockIdx.y * B * r;
    }
    constexpr int VEC = Elem<T>::kVec;
    __shared__ float red[kPredDownThreads / kWave][BT];
    const int k = blockIdx.x, tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const int chunks = H / VEC;
    const T *row = A + (size_t)k * H;
    const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
    if constexpr (CLEAR)   // (r blocks)
        for (int i = k * kPredDownThreads + tid; i < I; i += r * kPredDownThreads) mask[i] = 0;
    for (int b0 = 0; b0 < B; b0 += BT) {
        float acc[BT];
#pragma unroll
        for (int b = 0; b < BT; ++b) acc[b] = 0.f;
        for (int c0 = 0; c0 < chunks; c0 += kPredDownThreads * kPredDownUnroll) {
            uint4 w[kPredDownUnroll];
#pragma unroll
            for (int u = 0; u < kPredDownUnroll; ++u) {
                const int c = c0 + u * kPredDownThreads + tid;
                w[u] = c < chunks ? ld16(row + (size_t)c * VEC) : zero4;
            }
            // x for every row of the tile is requested together (clamped row: the surplus sums are dropped)
            uint4 xv[BT][kPredDownUnroll];
#pragma unroll
            for (int b = 0; b < BT; ++b) {
                const int bb = b0 + b < B ? b0 + b : B - 1;
#pragma unroll
                for (int u = 0; u < kPredDownUnroll; ++u) {
                    const int c = c0 + u * kPredDownThreads + tid;
                    xv[b][u] = ld16(x + (size_t)bb * H + (size_t)(c < chunks ? c : 0) * VEC);
                }
            }
#pragma unroll
            for (int u = 0; u < kPredDownUnroll; ++u) {
                float fw[VEC];
                unpack<T>(w[u], fw);   // zeros past the row end
#pragma unroll
                for (int b = 0; b < BT; ++b) {
                    float fx[VEC];
                    unpack<T>(xv[b][u], fx);
#pragma unroll
                    for (int e = 0; e < VEC; ++e) acc[b] = fmaf(fw[e], fx[e], acc[b]);
                }
            }
        }
#pragma unroll
        for (int b = 0; b < BT; ++b) {
            const float s = wave_sum_dpp(acc[b]);
            if (lane == 0) red[wave][b] = s;
        }
        __syncthreads();
        if (tid < BT && b0 + tid < B) {
            float s = 0.f;
#pragma unroll
            for (int w2 = 0; w2 < kPredDownThreads / kWave; ++w2) s += red[w2][tid];
            // (round_storage: the rank-r intermediate as a module in the storage type would hand it on)
            t[(size_t)(b0 + tid) * r + k] = round_storage ? to_float<T>(from_float<T>(s)) : s;
        }
        __syncthreads();
    }
}

constexpr int kPredUpThreads = 256;   // (128-thread blocks measure the same)
// Rows of Bm a wave owns: as few as keep every lane busy for one pass (four rows of 16 chunks, two of 32 or
// 64).  More rows per wave mean fewer blocks, and the layer measures slower: 16 rows per wave (128 blocks at
// I = 8192) cost 1 us per layer against 4, and 4 against 2 cost 1.2 us at r = 256 and 0.7 us at r = 440.
constexpr int pred_rows_per_wave(int lpr) { return lpr >= 32 ? 2 : 4; }
constexpr int kPredUpBTile = 8;

// LPR lanes share one row of Bm (LPR >= r/VEC unless the row needs several
// passes); a wave owns RPW consecutive rows and issues the loads of all of them
// before the rank-r intermediate is staged in LDS.  BT: rows of x per pass.  Single-row decode has a form of
// its own (BT 1): tests of the row count around every sum, and sums kept for eight rows, took 81 instead of 57 us for the
// 310 MB of 32 layers at I 11008, rank 440 (3.0 instead of 2.9 us for one layer at I 8192, rank 128).
template <typename T, int LPR, int RPW, int BT, typename Tab>
__global__ __launch_bounds__(kPredUpThreads) void predictor_up_mask_kernel(const float *__restrict__ t,
                                                                  const T *__restrict__ Bm,
                                                                  float *__restrict__ scores,
                                                                  uint8_t *__restrict__ mask, int B, int r, int I,
                                                                  float thr, int flags, Tab tab)
{
    if constexpr (Tab::kLayers) {
        const st_predictor_layer &ly = tab.l[blockIdx.y];
        Bm = static_cast<const T *>(ly.Bm);
        mask = ly.mask;
        thr = ly.thr;
        flags = (flags & ~1) | (ly.cmp_ge ? 1 : 0);
        t += (size_t)blockIdx.y * B * r;
    }
    // (13 dwords of arguments, all of them in scalar registers when the wave starts; the three switches share one)
    const int cmp_ge = flags & 1, round_storage = (flags >> 1) & 1, accumulate = (flags >> 2) & 1;
    constexpr int VEC = Elem<T>::kVec;
    constexpr int RPI = kWave / LPR;                                          // rows per iteration
    constexpr int NIT = RPW / RPI > 0 ? RPW / RPI : 1;  // iterations per tile
    extern __shared__ __align__(16) unsigned char smem[];
    float *ts = reinterpret_cast<float *>(smem);  // [B][r]
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const int chunks = r / VEC;
    const int cl = lane & (LPR - 1), gidx = lane / LPR;
    const int tile = (blockIdx.x * (kPredUpThreads / kWave) + wave) * RPW;
    const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);

    float s[NIT][BT];
    bool any[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it) any[it] = false;

    for (int b0 = 0; b0 < B || b0 == 0; b0 += BT) {
#pragma unroll
        for (int it = 0; it < NIT; ++it)
#pragma unroll
            for (int b = 0; b < BT; ++b) s[it][b] = 0.f;
        for (int c = cl; c < chunks || c == cl; c += LPR) {  // one pass unless r/VEC > LPR
            uint4 w[NIT];
#pragma unroll
            for (int it = 0; it < NIT; ++it) {
                const int ro = it * RPI + gidx;
                const int row = tile + ro;
                w[it] = (c < chunks && ro < RPW && row < I) ? ld16(Bm + (size_t)row * r + (size_t)c * VEC)
                                                                        : zero4;
            }
            if (b0 == 0 && c == cl) {  // stage t after the row loads are in flight
                // 16-byte pieces, two per thread requested together: one memory round trip per 8 KB
                // (a scalar copy loop pays one round trip per 256 bytes)
                const float4 *t4 = reinterpret_cast<const float4 *>(t);
                float4 *ts4 = reinterpret_cast<float4 *>(ts);
                const int n4 = (B * r) >> 2;
                for (int i0 = 0; i0 < n4; i0 += kPredUpThreads * 2) {
                    float4 v[2];
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const int i = i0 + u * kPredUpThreads + tid;
                        v[u] = t4[i < n4 ? i : n4 - 1];
                    }
#pragma unroll
                    for (int u = 0; u < 2; ++u)   // unconditional: the staging buffer is padded to whole batches
                        ts4[i0 + u * kPredUpThreads + tid] = v[u];
                }
                __syncthreads();
            }
            if (c < chunks) {
#pragma unroll
                for (int it = 0; it < NIT; ++it) {
                    float fw[VEC];
                    unpack<T>(w[it], fw);
#pragma unroll
                    for (int b = 0; b < BT; ++b) {
                        if (BT == 1 || b0 + b < B) {
                            const float *tp = ts + (size_t)(b0 + b) * r + c * VEC;
#pragma unroll
                            for (int e = 0; e < VEC; ++e) s[it][b] = fmaf(fw[e], tp[e], s[it][b]);
                        }
                    }
                }
            }
            if (c + LPR >= chunks) break;
        }
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
            const int ro = it * RPI + gidx;
            const int row = tile + ro;
            const bool row_ok = ro < RPW && row < I;
#pragma unroll
            for (int b = 0; b < BT; ++b) {
                if (BT == 1 || b0 + b < B) {  // uniform across the wave
                    float v = group_sum_dpp<LPR>(s[it][b]);
                    if (round_storage) v = to_float<T>(from_float<T>(v));
                    any[it] = any[it] || (cmp_ge ? (v >= thr) : (v > thr));
                    if (scores && cl == 0 && row_ok) scores[(size_t)(b0 + b) * I + row] = v;
                }
            }
        }
        if (b0 + BT >= B) break;
    }
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        const int ro = it * RPI + gidx;
        const int row = tile + ro;
        // (accumulate: a later pass over more rows of x only ever switches bytes on)
        if (cl == 0 && ro < RPW && row < I && (any[it] || !accumulate)) mask[row] = any[it] ? 1 : 0;
    }
}

// Several rows of x (B > 1), rank rows of at most LPR chunks: a lane keeps its chunk of t for eight rows of x
// in registers and reuses it for the NITER rows of Bm it visits, so the LDS is read once per lane instead of
// once per (row of Bm, row of x) -- the first form of the kernel was bound by exactly those reads (32-byte
// strides, half the banks idle) and took 1.3 us per additional row of x at r = 256.  All NITER row loads of a
// wave are issued before anything else.
template <typename T, int LPR, int NITER, typename Tab>
__global__ __launch_bounds__(kPredUpThreads) void predictor_up_mask_rows_kernel(const float *__restrict__ t,
                                                                       const T *__restrict__ Bm,
                                                                       float *__restrict__ scores,
                                                                       uint8_t *__restrict__ mask, int B, int r, int I,
                                                                       float thr, int flags, Tab tab)
{
    if constexpr (Tab::kLayers) {
        const st_predictor_layer &ly = tab.l[blockIdx.y];
        Bm = static_cast<const T *>(ly.Bm);
        mask = ly.mask;
        thr = ly.thr;
        flags = (flags & ~1) | (ly.cmp_ge ? 1 : 0);
        t += (size_t)blockIdx.y * B * r;
    }
    const int cmp_ge = flags & 1, round_storage = (flags >> 1) & 1, accumulate = (flags >> 2) & 1;   // (as above)
    constexpr int VEC = Elem<T>::kVec;
    constexpr int RPI = kWave / LPR;   // rows per iteration
    extern __shared__ __align__(16) unsigned char smem[];
    float *ts = reinterpret_cast<float *>(smem);  // [B][r]
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const int chunks = r / VEC;
    const int cl = lane & (LPR - 1), gidx = lane / LPR;
    const int tile = (blockIdx.x * (kPredUpThreads / kWave) + wave) * (RPI * NITER);
    const bool has_chunk = cl < chunks;

    uint4 w[NITER];
#pragma unroll
    for (int it = 0; it < NITER; ++it) {
        const int row = tile + it * RPI + gidx;
        w[it] = ld16(Bm + (size_t)(row < I ? row : I - 1) * r + (size_t)(has_chunk ? cl : 0) * VEC);
    }
    {   // stage t: 16-byte pieces, two per thread requested together (the buffer is padded to whole batches)
        const float4 *t4 = reinterpret_cast<const float4 *>(t);
        float4 *ts4 = reinterpret_cast<float4 *>(ts);
        const int n4 = (B * r) >> 2;
        for (int i0 = 0; i0 < n4; i0 += kPredUpThreads * 2) {
            float4 v[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int i = i0 + u * kPredUpThreads + tid;
                v[u] = t4[i < n4 ? i : n4 - 1];
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) ts4[i0 + u * kPredUpThreads + tid] = v[u];
        }
        __syncthreads();
    }
    unsigned any = 0u;   // bit per iteration
    for (int b0 = 0; b0 < B; b0 += kPredUpBTile) {
        float tr[kPredUpBTile][VEC];
#pragma unroll
        for (int b = 0; b < kPredUpBTile; ++b) {
            const float *tp = ts + (size_t)(b0 + b < B ? b0 + b : B - 1) * r + (has_chunk ? cl : 0) * VEC;
#pragma unroll
            for (int e = 0; e < VEC; e += 4) {
                const float4 q = *reinterpret_cast<const float4 *>(tp + e);
                tr[b][e] = q.x; tr[b][e + 1] = q.y; tr[b][e + 2] = q.z; tr[b][e + 3] = q.w;
            }
        }
#pragma unroll
        for (int it = 0; it < NITER; ++it) {
            const int row = tile + it * RPI + gidx;
            float fw[VEC];
            unpack<T>(w[it], fw);
#pragma unroll
            for (int b = 0; b < kPredUpBTile; ++b) {
                if (b0 + b < B) {   // uniform
                    float acc = 0.f;
#pragma unroll
                    for (int e = 0; e < VEC; ++e) acc = fmaf(fw[e], tr[b][e], acc);
                    // (lanes without a chunk multiplied the first one: not by zero weights, which an infinity makes NaN of)
                    float v = group_sum_dpp<LPR>(has_chunk ? acc : 0.f);
                    if (round_storage) v = to_float<T>(from_float<T>(v));
                    if (cmp_ge ? (v >= thr) : (v > thr)) any |= 1u << it;
                    if (scores && cl == 0 && row < I) scores[(size_t)(b0 + b) * I + row] = v;
                }
            }
        }
    }
#pragma unroll
    for (int it = 0; it < NITER; ++it) {
        const int row = tile + it * RPI + gidx;
        if (cl == 0 && row < I && (((any >> it) & 1u) || !accumulate)) mask[row] = (any >> it) & 1u;
    }
}

// What the two kernels of one call (one layer, or several of equal shape) are launched with.
struct PredLaunch {
    const void *x; int B, H; const void *A; int r; const void *Bm; int I;
    float thr; int flags;   // bit 0: >=, bit 1: round to storage, bit 2: later pass
    float *t_ws, *scores; uint8_t *mask;
    int layers; hipStream_t stream;
};

template <typename T, int LPR, typename Tab>
static void launch_up(ProfScope &ps, const PredLaunch &a, const Tab &tab)
{
    constexpr size_t batch = (size_t)kPredUpThreads * 2 * 16;   // the staging buffer is padded to whole batches
    const size_t lds = ((size_t)a.B * a.r * sizeof(float) + batch - 1) / batch * batch;
    auto go = [&](auto kern, int rows) {
        ST_LAUNCH(ps, kern, dim3((a.I + rows - 1) / rows, a.layers), dim3(kPredUpThreads), lds, a.stream, a.t_ws,
                  static_cast<const T *>(a.Bm), a.scores, a.mask, a.B, a.r, a.I, a.thr, a.flags, tab);
    };
    constexpr int NITER = LPR >= 16 ? LPR / 16 : 1;   // about four rows of Bm per wave (measured against 1, 2 and 8 per lane)
    constexpr int RPW = pred_rows_per_wave(LPR);
    const int up_rows = RPW * (kPredUpThreads / kWave);
    if (a.B == 1) go(predictor_up_mask_kernel<T, LPR, RPW, 1, Tab>, up_rows);
    else if (a.r / Elem<T>::kVec > LPR) go(predictor_up_mask_kernel<T, LPR, RPW, kPredUpBTile, Tab>, up_rows);
    else go(predictor_up_mask_rows_kernel<T, LPR, NITER, Tab>, (kWave / LPR) * NITER * (kPredUpThreads / kWave));
}

template <typename T, typename Tab>
static int launch_predictor(const PredLaunch &a, const Tab &tab)
{
    constexpr int dtype = Elem<T>::kBytes == 4 ? ST_F32 : __is_same(T, f16_t) ? ST_F16 : ST_BF16;
    // (not a later pass over more rows of x, which must not clear what an earlier one switched on: those have up to 64 rows each)
    const bool up_mfma = (a.flags & 4) == 0 && predictor_up_mfma_supported(dtype, a.B, a.r, a.I);
    {
        ProfScope ps(ST_K_PRED_DOWN, a.stream);
        auto go = [&](auto kern) {
            ST_LAUNCH(ps, kern, dim3(a.r, a.layers), dim3(kPredDownThreads), 0, a.stream, static_cast<const T *>(a.x), a.B,
                      a.H, static_cast<const T *>(a.A), a.r, a.t_ws, (a.flags >> 1) & 1, a.mask, a.I, tab);
        };
        if (a.B == 1) go(predictor_down_kernel<T, 1, false, Tab>);
        else if (up_mfma) go(predictor_down_kernel<T, kPredBTile, dtype == ST_BF16, Tab>);   // (up_mfma: bf16 only)
        else if (a.B <= kPredBTile) go(predictor_down_kernel<T, kPredBTile, false, Tab>);
        else go(predictor_down_kernel<T, 2 * kPredBTile, false, Tab>);   // 9 to 16 rows of x in one pass (one memory round trip instead of two)
    }
    ST_HIP(hipGetLastError());
    if (up_mfma)
        return launch_predictor_up_mfma(dtype, tab, a.layers, a.B, a.r, a.Bm, a.I, a.thr, a.flags & 1, a.t_ws, a.scores, a.mask,
                                        (a.flags >> 1) & 1, a.stream);
    const int chunks = a.r / Elem<T>::kVec;
    {
        ProfScope ps(ST_K_PRED_UP_MASK, a.stream);
        if (chunks <= 4) launch_up<T, 4>(ps, a, tab);
        else if (chunks <= 8) launch_up<T, 8>(ps, a, tab);
        else if (chunks <= 16) launch_up<T, 16>(ps, a, tab);
        else if (chunks <= 32) launch_up<T, 32>(ps, a, tab);
        else launch_up<T, 64>(ps, a, tab);
    }
    ST_HIP(hipGetLastError());
    return ST_OK;
}

template <typename Tab> static int launch_predictor_dtype(int dtype, const PredLaunch &a, const Tab &tab)
{
    switch (dtype) {
    case ST_F32: return launch_predictor<float>(a, tab);
    case ST_F16: return launch_predictor<f16_t>(a, tab);
    default: return launch_predictor<bf16_t>(a, tab);
    }
}

// Rows of x per pass of these kernels: what the staging buffer of the second one holds, 64 at most.
static int64_t pred_rows_per_pass(int64_t r)
{
    const int64_t per = (56 * 1024) / (r * 4);
    return per > 64 ? 64 : per;
}

static int check_predictor_args(const char *who, int64_t B, int64_t H, int64_t r, int64_t I, int dtype, int flags)
{
    ST_REQUIRE(dtype >= ST_F32 && dtype <= ST_BF16, "%s: unknown dtype %d", who, dtype);
    const int esz = dtype == ST_F32 ? 4 : 2;
    ST_REQUIRE(B >= 1 && B <= (1 << 20), "%s: B=%lld out of range", who, (long long)B);
    ST_REQUIRE(H >= 1 && (H * esz) % 16 == 0, "%s: H=%lld rows are not 16-byte multiples", who, (long long)H);
    ST_REQUIRE(r >= 1 && (r * esz) % 16 == 0, "%s: rank %lld rows are not 16-byte multiples", who, (long long)r);
    ST_REQUIRE(I >= 1 && I <= (1 << 24), "%s: I=%lld out of range", who, (long long)I);
    ST_REQUIRE(r * 4 <= 56 * 1024, "%s: rank %lld too large for the LDS staging buffer", who, (long long)r);
    ST_REQUIRE((flags & ~ST_PRED_ROUND_STORAGE) == 0, "%s: unknown flags %d", who, flags);
    return ST_OK;
}

}  // namespace st

extern "C" int st_predictor_mask_ex(const void *x, int64_t B, int64_t H, const void *A, int64_t r, const void *Bm,
                                    int64_t I, int dtype, float thr, int cmp_ge, int flags, float *t_ws, float *scores,
                                    uint8_t *mask, void *stream)
{
    using namespace st;
    ST_REQUIRE(x && A && Bm && t_ws && mask, "st_predictor_mask_ex: null pointer");
    const int arc = check_predictor_args("st_predictor_mask_ex", B, H, r, I, dtype, flags);
    if (arc != ST_OK) return arc;
    const int esz = dtype == ST_F32 ? 4 : 2;
    const uintptr_t align = (uintptr_t)x | (uintptr_t)A | (uintptr_t)Bm;
    ST_REQUIRE((align & 15) == 0, "st_predictor_mask_ex: pointers must be 16-byte aligned");
    const int round_storage = (flags & ST_PRED_ROUND_STORAGE) && dtype != ST_F32 ? 1 : 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (predictor_mfma_supported(dtype, (int)B, (int)H, (int)r))
        return launch_predictor_mfma(dtype, x, (int)B, (int)H, A, (int)r, Bm, (int)I, thr, cmp_ge, t_ws, scores, mask,
                                     round_storage, s);
    // Further passes reuse the front of t_ws (the launches are ordered on the stream) and only ever switch mask bytes on.
    const int64_t per = pred_rows_per_pass(r);
    for (int64_t b0 = 0; b0 < B; b0 += per) {
        PredLaunch a;
        a.x = static_cast<const unsigned char *>(x) + (size_t)b0 * H * esz;
        a.B = (int)(B - b0 < per ? B - b0 : per);
        a.H = (int)H; a.A = A; a.r = (int)r; a.Bm = Bm; a.I = (int)I;
        a.thr = thr;
        a.flags = (cmp_ge ? 1 : 0) | (round_storage ? 2 : 0) | (b0 > 0 ? 4 : 0);
        a.t_ws = t_ws;
        a.scores = scores ? scores + (size_t)b0 * I : nullptr;
        a.mask = mask; a.layers = 1; a.stream = s;
        const int rc = launch_predictor_dtype(dtype, a, NoLayers{});
        if (rc != ST_OK) return rc;
    }
    return ST_OK;
}

extern "C" int st_predictor_mask_layers(const st_predictor_layer *layers, int64_t L, const void *x, int64_t B, int64_t H,
                                        int64_t r, int64_t I, int dtype, int flags, float *t_ws, void *stream)
{
    using namespace st;
    ST_REQUIRE(layers && x && t_ws && L >= 1, "st_predictor_mask_layers: null pointer or no layers");
    const int arc = check_predictor_args("st_predictor_mask_layers", B, H, r, I, dtype, flags);
    if (arc != ST_OK) return arc;
    const int esz = dtype == ST_F32 ? 4 : 2;
    uintptr_t align = (uintptr_t)x | (uintptr_t)((size_t)B * H * esz) | (uintptr_t)t_ws;
    for (int64_t l = 0; l < L; ++l) {
        ST_REQUIRE(layers[l].A && layers[l].Bm && layers[l].mask, "st_predictor_mask_layers: null pointer in layer %lld", (long long)l);
        align |= (uintptr_t)layers[l].A | (uintptr_t)layers[l].Bm;
    }
    ST_REQUIRE((align & 15) == 0, "st_predictor_mask_layers: pointers must be 16-byte aligned");
    const int round_storage = (flags & ST_PRED_ROUND_STORAGE) && dtype != ST_F32 ? 1 : 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool mfma = predictor_mfma_supported(dtype, (int)B, (int)H, (int)r);
    if (!mfma && B > pred_rows_per_pass(r)) {   // several passes per layer: one layer at a time
        for (int64_t l = 0; l < L; ++l) {
            const st_predictor_layer &y = layers[l];
            const int rc = st_predictor_mask_ex(static_cast<const unsigned char *>(x) + (size_t)l * B * H * esz, B, H, y.A, r,
                                                y.Bm, I, dtype, y.thr, y.cmp_ge, flags, t_ws, nullptr, y.mask, stream);
            if (rc != ST_OK) return rc;
        }
        return ST_OK;
    }
    for (int64_t l0 = 0; l0 < L; l0 += kMaxLayers) {
        PredLayers tab;
        const int nl = (int)(L - l0 < kMaxLayers ? L - l0 : kMaxLayers);
        for (int l = 0; l < kMaxLayers; ++l) tab.l[l] = layers[l0 + (l < nl ? l : 0)];
        const void *xl = static_cast<const unsigned char *>(x) + (size_t)l0 * B * H * esz;
        float *tl = t_ws + (size_t)l0 * B * r;
        int rc;
        if (mfma) {
            rc = launch_predictor_mfma_layers(dtype, tab, nl, xl, (int)B, (int)H, (int)r, (int)I, tl, round_storage, s);
        } else {
            PredLaunch a;
            a.x = xl; a.B = (int)B; a.H = (int)H; a.A = nullptr; a.r = (int)r; a.Bm = nullptr; a.I = (int)I;
            a.thr = 0.f; a.flags = round_storage ? 2 : 0;
            a.t_ws = tl; a.scores = nullptr; a.mask = nullptr; a.layers = nl; a.stream = s;
            rc = launch_predictor_dtype(dtype, a, tab);
        }
        if (rc != ST_OK) return rc;
    }
    return ST_OK;
}

extern "C" int st_predictor_mask(const void *x, int64_t B, int64_t H, const void *A, int64_t r, const void *Bm,
                                 int64_t I, int dtype, float thr, int cmp_ge, float *t_ws, float *scores,
                                 uint8_t *mask, void *stream)
{
    return st_predictor_mask_ex(x, B, H, A, r, Bm, I, dtype, thr, cmp_ge, 0, t_ws, scores, mask, stream);
}
