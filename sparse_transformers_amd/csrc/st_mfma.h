// Matrix-core helpers shared by the MFMA translation units (fp16 / bf16 16x16x32, fp32 accumulate).
//
// Operand layout of v_mfma_f32_16x16x32 on a 64-lane wave, D[m][n] += sum_k A[m][k] * B[k][n]:
//   A: lane l holds row m = l % 16, the 8 consecutive k of slice l / 16
//   B: lane l holds column n = l % 16, the 8 consecutive k of slice l / 16
//   D: lane l holds column n = l % 16, rows m = 4 * (l / 16) + e for e = 0..3
#pragma once

#include "st_common.h"

namespace st {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <typename T> struct Mfma;
template <> struct Mfma<f16_t> {
    static __device__ __forceinline__ f32x4_t run(const uint4 &a, const uint4 &b, f32x4_t c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b),
                                                      c, 0, 0, 0);
    }
};
template <> struct Mfma<bf16_t> {
    static __device__ __forceinline__ f32x4_t run(const uint4 &a, const uint4 &b, f32x4_t c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
};

constexpr int kXcds = 8;

// Workgroups are handed to the 8 XCDs round-robin by their linear id, and each XCD has its own L2.
// This maps the linear id to a tile id such that every XCD works through one contiguous range of tile
// ids; tile ids are ordered so that neighbours share an operand tile (the same weight rows for all row
// tiles of x), which then comes from that XCD's L2 instead of HBM.  Returns -1 for the padding ids.
__device__ __forceinline__ int xcd_tile_id(int bid, int ntiles)
{
    const int per = (ntiles + kXcds - 1) / kXcds;
    const int t = (bid % kXcds) * per + bid / kXcds;
    return (bid / kXcds < per && t < ntiles) ? t : -1;
}

// s_waitcnt immediate: vmcnt in bits 3:0 (and 15:14), expcnt 6:4 left at "no wait", lgkmcnt 11:8 = 0
#define ST_WAIT_VM_LGKM0(vm) __builtin_amdgcn_s_waitcnt(((vm) & 15) | (7 << 4) | (0 << 8) | (((vm) >> 4) << 14))

// 64 lanes x 16 bytes from `base + off` (uniform base, per-lane byte offset) to the 1 KB of LDS at byte address
// `dst` (uniform), lane i's 16 bytes at dst + 16 i.  The instruction takes the LDS address from M0; the compiler is not
// told about M0 (it is a reserved register for inline assembly), so its value is put back, and the write of M0 is
// followed by the wait state the instruction needs before it may read it.
__device__ __forceinline__ void load_to_lds(unsigned dst, unsigned off, const char *base)
{
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "s"(dst), "v"(off), "s"(base)
                 : "memory");
}

__device__ __forceinline__ int device_count(int n_host, const int *n_dev)
{
    int n = n_host;
    if (n_dev) {
        const int nd = *n_dev;
        n = nd < n ? nd : n;
        if (n < 0) n = 0;
    }
    return n;
}

}  // namespace st
