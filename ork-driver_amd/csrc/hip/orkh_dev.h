// orkh_dev.h -- device helpers shared by the matmul kernels on resident panels (orkh_kernels.hip, orkh_big.hip,
// orkh_grouped.hip): the panel kinds, nibble and NF4 decode, MFMA, raw buffer loads, direct-to-LDS loads, write-through
// stores.
#ifndef ORKH_DEV_H
#define ORKH_DEV_H
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <atomic>

#include "orkh.h"

extern thread_local char g_lerr[256]; // why the last launch call on this thread refused its plan (orkh_launch_error)

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <int KIND> struct KT;
template <> struct KT<ORKH_I8> {
    static constexpr int KPB = 64, STEPS = 1, ESZ = 1;
    typedef v4i acc_t;
    typedef int32_t c_t;
};
template <> struct KT<ORKH_I4U> {
    static constexpr int KPB = 128, STEPS = 2, ESZ = 1;
    typedef v4i acc_t;
    typedef int32_t c_t;
};
template <> struct KT<ORKH_NF4> {
    static constexpr int KPB = 128, STEPS = 2, ESZ = 1;
    typedef v4i acc_t;
    typedef int32_t c_t;
};
template <> struct KT<ORKH_F16> {
    static constexpr int KPB = 32, STEPS = 1, ESZ = 2;
    typedef v4f acc_t;
    typedef float c_t;
};

// First k (within a K-block) of the 16-byte A chunk that lane group g feeds to MFMA step s. Must match
// the B byte -> k assignment of the panel layout.
template <int KIND> __device__ __forceinline__ int a_koff(int s, int g) {
    if constexpr (KIND == ORKH_I8) return g * 16;
    else if constexpr (KIND == ORKH_F16) return g * 8;
    else return g * 32 + s * 16;
}

struct Lut { uint32_t l0, l1, l2, l3; };

// One dword of NF4 codes (8 nibbles) -> the int8 codebook values of its low nibbles (lo) and of its high
// nibbles (hi), byte for byte. Both 8-entry halves of the codebook are looked up with the code's low 3 bits
// (v_perm: selector bytes 0-3 pick from its second operand, 4-7 from its first), then a third v_perm takes
// byte j from the upper half where bit 3 of code j is set: its selector byte is j + 4 * bit3. Six VALU
// operations per four codes (the select mask built from bit 3 by shift-and-subtract took eight).
__device__ __forceinline__ void nf4_map8(uint32_t x, const Lut &L, uint32_t &lo, uint32_t &hi) {
    const uint32_t i0 = x & 0x07070707u, i1 = (x >> 4) & 0x07070707u;
    const uint32_t s0 = ((x >> 1) & 0x04040404u) | 0x03020100u; // bit 3 of each low nibble -> byte select
    const uint32_t s1 = ((x >> 5) & 0x04040404u) | 0x03020100u; // bit 7 (bit 3 of the high nibble)
    lo = __builtin_amdgcn_perm(__builtin_amdgcn_perm(L.l3, L.l2, i0), __builtin_amdgcn_perm(L.l1, L.l0, i0), s0);
    hi = __builtin_amdgcn_perm(__builtin_amdgcn_perm(L.l3, L.l2, i1), __builtin_amdgcn_perm(L.l1, L.l0, i1), s1);
}

// Raw 16-byte panel chunk -> STEPS MFMA B operands.
template <int KIND> __device__ __forceinline__ void decode(v4i raw, v4i *op, const Lut &L) {
    if constexpr (KIND == ORKH_I8 || KIND == ORKH_F16) {
        op[0] = raw;
    } else if constexpr (KIND == ORKH_I4U) {
        const uint32_t x0 = raw.x, x1 = raw.y, x2 = raw.z, x3 = raw.w;
        op[0] = v4i{(int)((x0 << 4) & 0xf0f0f0f0u), (int)(x0 & 0xf0f0f0f0u),
                    (int)((x1 << 4) & 0xf0f0f0f0u), (int)(x1 & 0xf0f0f0f0u)};
        op[1] = v4i{(int)((x2 << 4) & 0xf0f0f0f0u), (int)(x2 & 0xf0f0f0f0u),
                    (int)((x3 << 4) & 0xf0f0f0f0u), (int)(x3 & 0xf0f0f0f0u)};
    } else {
        uint32_t a0, b0, a1, b1, a2, b2, a3, b3;
        nf4_map8((uint32_t)raw.x, L, a0, b0);
        nf4_map8((uint32_t)raw.y, L, a1, b1);
        nf4_map8((uint32_t)raw.z, L, a2, b2);
        nf4_map8((uint32_t)raw.w, L, a3, b3);
        op[0] = v4i{(int)a0, (int)b0, (int)a1, (int)b1};
        op[1] = v4i{(int)a2, (int)b2, (int)a3, (int)b3};
    }
}

__device__ __forceinline__ v4i mma(v4i a, v4i b, v4i c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4f mma(v4i a, v4i b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

template <int KIND> __device__ __forceinline__ typename KT<KIND>::c_t finish(typename KT<KIND>::c_t v) {
    if constexpr (KIND == ORKH_I4U) return v >> 4;  // exact: every partial is 16 * integer
    else return v;
}

// ------------------------------------------------------------------------------------------------
// Raw buffer loads: the hardware returns 0 for any byte offset >= num_records, so out-of-range rows,
// K tails and stages past the end cost no clamping or select instructions, and can never fault.
typedef unsigned v4u __attribute__((ext_vector_type(4)));
constexpr uint32_t OOB = 0x80000000u;  // an offset past every buffer this path addresses (< 2 GiB)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ v4i bload(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return (v4i)__builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
}

// Write-through vector stores at device scope (global_store_* ... sc1): the L2 passes the data on to memory as it
// comes instead of holding it dirty until the end of the kernel. Written as asm because the compiler merges a store
// that carries a cache-policy modifier with an otherwise identical plain store on the other side of a branch, and
// drops the modifier.
__device__ __forceinline__ void store_wt(int *p, int v) {
    asm volatile("global_store_dword %0, %1, off sc1" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void store_wt(float *p, float v) {
    asm volatile("global_store_dword %0, %1, off sc1" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void store_wt4(void *p, v4i v) {
    asm volatile("global_store_dwordx4 %0, %1, off sc1" ::"v"(p), "v"(v) : "memory");
}
// Direct-to-LDS loads. M0 carries the LDS destination; nothing else in these kernels uses M0 (checked in the ISA), so the
// clobber of that reserved register is safe and its warning is silenced here.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// SITE only numbers the call site in an asm comment: identical asm at several sites lets the compiler merge them
// through a phi it may place in a VGPR, which the "s" operand cannot take.
template <int SITE = 0>
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t lds_byte) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds ; site %3" ::"s"(lds_byte),
                 "v"(voff), "s"(r), "i"(SITE)
                 : "memory", "m0");
}
// At a per-lane offset plus a scalar one, 16 and 4 bytes a lane (the range check covers the per-lane offset only: a lane
// whose sum would leave the resource carries OOB)
__device__ __forceinline__ void lds_dma16s(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, uint32_t lds_byte) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds_byte), "v"(voff), "s"(r),
                 "s"(soff)
                 : "memory", "m0");
}
__device__ __forceinline__ void lds_dma4s(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, uint32_t lds_byte) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"s"(lds_byte), "v"(voff), "s"(r),
                 "s"(soff)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
template <int VM> __device__ __forceinline__ void wait_vmcnt() {
    static_assert(VM >= 0 && VM < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Quotient and remainder of a wave-uniform x / d (0 <= x, 1 <= d, both < 2^24) on the VALU: the correctly
// rounded float quotient is within one of the integer one, and one correction fixes it. A scalar integer
// division is ~35 instructions on the scalar unit, which a workgroup's 16 waves share; two of them per wave
// in a tiled kernel's prologue queue ~1,000 cycles there.
__device__ __forceinline__ void udivmod(int x, int d, int &q, int &r) {
    int qq = (int)((float)x / (float)d);
    int rr = x - qq * d;
    if (rr < 0) { qq--; rr += d; }
    else if (rr >= d) { qq++; rr -= d; }
    q = __builtin_amdgcn_readfirstlane(qq);
    r = __builtin_amdgcn_readfirstlane(rr);
}

// Raise a kernel's dynamic-LDS limit once per (kernel, device): hipFuncSetAttribute holds per device, so the
// flags are per device, and atomic, since contexts may launch from several threads.
constexpr int ORKH_MAX_DEV = 64;
typedef std::atomic<bool> lds_flags[ORKH_MAX_DEV];
inline int lds_limit(const void *kern, int bytes, lds_flags &done) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= ORKH_MAX_DEV) {
        snprintf(g_lerr, sizeof g_lerr, "LDS limit: no current device below %d", ORKH_MAX_DEV);
        return -1;
    }
    if (done[dev].load(std::memory_order_acquire)) return 0;
    const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) {
        snprintf(g_lerr, sizeof g_lerr, "hipFuncSetAttribute(%d B of LDS): %s", bytes, hipGetErrorString(e));
        return -1;
    }
    done[dev].store(true, std::memory_order_release);
    return 0;
}

} // namespace
#endif
