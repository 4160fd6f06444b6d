// Device-side helpers shared by the SDDMM kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sddmm {

constexpr int WAVE = 64;
constexpr int NUM_XCD = 8;  // MI355X: 8 accelerator complex dies, one L2 each

// ---- cross-lane -----------------------------------------------------------
// DPP control words (gfx9 encoding)
constexpr int DPP_QUAD_XOR1 = 0xB1;        // quad_perm:[1,0,3,2]
constexpr int DPP_QUAD_XOR2 = 0x4E;        // quad_perm:[2,3,0,1]
constexpr int DPP_ROW_HALF_MIRROR = 0x141; // lane i <-> 7-i inside each 8
constexpr int DPP_ROW_MIRROR = 0x140;      // lane i <-> 15-i inside each 16

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
    // old = 0 with bound_ctrl lets the compiler fold the move into the consuming
    // VALU instruction (v_add_f32_dpp); every pattern used here reads a valid lane
    int i = __builtin_bit_cast(int, v);
    i = __builtin_amdgcn_update_dpp(0, i, CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(float, i);
}

// Sum over aligned groups of LPN lanes; every lane of the group ends with the
// total.  The addition tree is fixed (1,2,4,8,16,32), so the value does not
// depend on which kernel calls it.
template <int LPN>
__device__ __forceinline__ float group_sum(float v) {
    if constexpr (LPN >= 2) v += dpp_f32<DPP_QUAD_XOR1>(v);
    if constexpr (LPN >= 4) v += dpp_f32<DPP_QUAD_XOR2>(v);
    if constexpr (LPN >= 8) v += dpp_f32<DPP_ROW_HALF_MIRROR>(v);
    if constexpr (LPN >= 16) v += dpp_f32<DPP_ROW_MIRROR>(v);
    if constexpr (LPN >= 32) {
        // swap the two 16-lane halves of each 32: ds_swizzle bit mode, xor 0x10
        int i = __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), 0x401F);
        v += __builtin_bit_cast(float, i);
    }
    if constexpr (LPN >= 64) v += __shfl_xor(v, 32, WAVE);
    return v;
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & (WAVE - 1); }
__device__ __forceinline__ int waves_in_block() { return (int)(blockDim.x >> 6); }
// index of the wavefront inside its workgroup, as a scalar
__device__ __forceinline__ int wave_in_block() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// ---- 16-lane helpers (a strip is walked by 16 neighbouring lanes) -------------
template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
    return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xF, 0xF, false);
}
__device__ __forceinline__ int min16(int v) {
    int o;
    o = dpp_i32<DPP_QUAD_XOR1>(v); v = o < v ? o : v;
    o = dpp_i32<DPP_QUAD_XOR2>(v); v = o < v ? o : v;
    o = dpp_i32<DPP_ROW_HALF_MIRROR>(v); v = o < v ? o : v;
    o = dpp_i32<DPP_ROW_MIRROR>(v); v = o < v ? o : v;
    return v;
}
__device__ __forceinline__ int sum16(int v) {
    v += dpp_i32<DPP_QUAD_XOR1>(v);
    v += dpp_i32<DPP_QUAD_XOR2>(v);
    v += dpp_i32<DPP_ROW_HALF_MIRROR>(v);
    v += dpp_i32<DPP_ROW_MIRROR>(v);
    return v;
}

// Sums over a wavefront in the vector unit, all 64 lanes active.  (As six __shfl steps through the LDS crossbar: k_own_rows of
// 29 000 rows 18.2 us, so 16.5; k_scan_jobs 5.8 and 5.2.)
__device__ __forceinline__ int wave_sum_i32(int v) {
    v = sum16(v);
    return (__builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16)) +
           (__builtin_amdgcn_readlane(v, 32) + __builtin_amdgcn_readlane(v, 48));
}
__device__ __forceinline__ int wave_inclusive_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);       // row_shr:1, 2, 4, 8: within 16 lanes
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);       // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);       // row_bcast:31 into rows 2 and 3
    return v;
}

// LDS that only one wavefront touches: its LDS operations execute in program order, so a
// write followed by a read of another lane's slot needs no workgroup barrier, only that the
// compiler keeps the order.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Workgroups are handed to the 8 XCDs round-robin by id.  Give every XCD one
// contiguous eighth of the logical work so that neighbouring row panels (which
// touch neighbouring B rows) share an L2.  Returns the logical index, or -1 for
// the padding blocks of the rounded-up grid.
__device__ __forceinline__ int64_t xcd_remap(int64_t bid, int64_t nblocks) {
    int64_t per = (nblocks + NUM_XCD - 1) / NUM_XCD;
    int64_t logical = (bid % NUM_XCD) * per + bid / NUM_XCD;
    return logical < nblocks ? logical : -1;
}
inline int64_t xcd_grid(int64_t nblocks) {
    return ((nblocks + NUM_XCD - 1) / NUM_XCD) * NUM_XCD;
}

// Streamed operands (column indices, S values, row indices, P) are touched once
// per run.  Marking them non-temporal (SDDMM_NT=1) was measured SLOWER on MI355X
// (FEM-banded K=32: 119 us vs 86 us; power-law unchanged): repeated runs find the
// index arrays in the last-level cache, and the hint gives that up.  Off by default.
#ifndef SDDMM_NT
#define SDDMM_NT 0
#endif
template <class T>
__device__ __forceinline__ T ld_stream(const T *p) {
#if SDDMM_NT
    return __builtin_nontemporal_load(p);
#else
    return *p;
#endif
}
template <class T>
__device__ __forceinline__ void st_stream(T *p, T v) {
#if SDDMM_NT
    __builtin_nontemporal_store(v, p);
#else
    *p = v;
#endif
}

// four consecutive values of an array that is only 4-byte aligned, as one access
struct __attribute__((packed, aligned(4))) I4u { int x, y, z, w; };
struct __attribute__((packed, aligned(4))) F4u { float x, y, z, w; };
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

// One work item of the wave-per-segment kernel: entries [start,end) of one row.
struct RowItem {
    int32_t row;
    int32_t start;
    int32_t end;
    int32_t extra;     // panels: where the first row starts; fused items: place of a cut row's piece (k_piece_places)
};

// ---- units of the K dimension ----------------------------------------------
// A "unit" is what one lane loads per step along K: 16 bytes where alignment
// allows (4 fp32, 8 bf16 or 8 fp16), one fp32 otherwise.  dot() extends an fp32
// accumulator with fused multiply-adds in element order.
// The kernels take the length of a row as a number of units, or of elements where rows hold no
// whole number of units (fp32, K % 4 != 0: rows are 4-byte aligned, which is all that 16-byte
// global loads need).  The last unit of such a row then ends with the row; its first elements
// are the unit's before it, and trim() zeroes them.
// element types of A and B as template arguments of the kernels
constexpr int DT_F32 = 0, DT_BF16 = 1, DT_F16 = 2;

template <class T_>
struct WholeUnits {
    using T = T_;
    static constexpr bool WHOLE = true;
    static __device__ __forceinline__ int units(int len) { return len; }
    static __device__ __forceinline__ uint32_t row_bytes(int len) { return (uint32_t)len * (uint32_t)sizeof(T); }
    static __device__ __forceinline__ uint32_t unit_off(int u, int) { return (uint32_t)u * (uint32_t)sizeof(T); }
    static __device__ __forceinline__ T load(const char *p) { return *reinterpret_cast<const T *>(p); }
    static __device__ __forceinline__ T trim(const T &v, int, int) { return v; }
};

struct UnitF32x4 : WholeUnits<float4> {
    static constexpr int DT = DT_F32;
    static constexpr int ELEMS = 4;
    static __device__ __forceinline__ T zero() { return make_float4(0.f, 0.f, 0.f, 0.f); }
    static __device__ __forceinline__ float dot(const T &a, const T &b, float acc) {
        acc = __builtin_fmaf(a.x, b.x, acc);
        acc = __builtin_fmaf(a.y, b.y, acc);
        acc = __builtin_fmaf(a.z, b.z, acc);
        acc = __builtin_fmaf(a.w, b.w, acc);
        return acc;
    }
    // acc[e] += p * (element e of b)
    static __device__ __forceinline__ void axpy(float p, const T &b, float (&acc)[ELEMS]) {
        acc[0] = __builtin_fmaf(p, b.x, acc[0]);
        acc[1] = __builtin_fmaf(p, b.y, acc[1]);
        acc[2] = __builtin_fmaf(p, b.z, acc[2]);
        acc[3] = __builtin_fmaf(p, b.w, acc[3]);
    }
};
struct UnitF32x4u : UnitF32x4 {
    static constexpr bool WHOLE = false;
    static __device__ __forceinline__ int units(int len) { return (len + 3) >> 2; }
    static __device__ __forceinline__ uint32_t row_bytes(int len) { return (uint32_t)len * 4u; }
    static __device__ __forceinline__ uint32_t unit_off(int u, int len) {
        const uint32_t at = (uint32_t)u * 16u, top = (uint32_t)len * 4u - 16u;
        return at < top ? at : top;
    }
    static __device__ __forceinline__ T load(const char *p) {
        return __builtin_bit_cast(T, *reinterpret_cast<const F4u *>(p));
    }
    static __device__ __forceinline__ T trim(const T &v, int u, int len) {
        const int n = units(len), cut = u == n - 1 ? 4 * n - len : 0;
        return make_float4(cut > 0 ? 0.f : v.x, cut > 1 ? 0.f : v.y, cut > 2 ? 0.f : v.z, v.w);
    }
};
struct UnitF32x1 : WholeUnits<float> {           // rows of fewer than four elements
    static constexpr int DT = DT_F32;
    static constexpr int ELEMS = 1;
    static __device__ __forceinline__ T zero() { return 0.f; }
    static __device__ __forceinline__ float dot(const T &a, const T &b, float acc) {
        return __builtin_fmaf(a, b, acc);
    }
};
struct UnitBF16x8 : WholeUnits<uint4> {
    static constexpr int DT = DT_BF16;
    // 8 bfloat16, two per 32-bit word, low half first
    static constexpr int ELEMS = 8;
    static __device__ __forceinline__ T zero() { return make_uint4(0u, 0u, 0u, 0u); }
    static __device__ __forceinline__ float lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
    static __device__ __forceinline__ float hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xFFFF0000u); }
    static __device__ __forceinline__ float dot(const T &a, const T &b, float acc) {
        acc = __builtin_fmaf(lo(a.x), lo(b.x), acc);
        acc = __builtin_fmaf(hi(a.x), hi(b.x), acc);
        acc = __builtin_fmaf(lo(a.y), lo(b.y), acc);
        acc = __builtin_fmaf(hi(a.y), hi(b.y), acc);
        acc = __builtin_fmaf(lo(a.z), lo(b.z), acc);
        acc = __builtin_fmaf(hi(a.z), hi(b.z), acc);
        acc = __builtin_fmaf(lo(a.w), lo(b.w), acc);
        acc = __builtin_fmaf(hi(a.w), hi(b.w), acc);
        return acc;
    }
    static __device__ __forceinline__ void axpy(float p, const T &b, float (&acc)[ELEMS]) {
        acc[0] = __builtin_fmaf(p, lo(b.x), acc[0]); acc[1] = __builtin_fmaf(p, hi(b.x), acc[1]);
        acc[2] = __builtin_fmaf(p, lo(b.y), acc[2]); acc[3] = __builtin_fmaf(p, hi(b.y), acc[3]);
        acc[4] = __builtin_fmaf(p, lo(b.z), acc[4]); acc[5] = __builtin_fmaf(p, hi(b.z), acc[5]);
        acc[6] = __builtin_fmaf(p, lo(b.w), acc[6]); acc[7] = __builtin_fmaf(p, hi(b.w), acc[7]);
    }
};

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
struct UnitF16x8 : WholeUnits<uint4> {
    static constexpr int DT = DT_F16;
    // 8 IEEE half floats, two per 32-bit word, low half first
    static constexpr int ELEMS = 8;
    static __device__ __forceinline__ T zero() { return make_uint4(0u, 0u, 0u, 0u); }
    // v_dot2c_f32_f16: acc + a.lo*b.lo + a.hi*b.hi with fp32 accumulation (products of
    // halves are exact in fp32)
    static __device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float acc) {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, a), __builtin_bit_cast(half2_t, b), acc, false);
    }
    static __device__ __forceinline__ float dot(const T &a, const T &b, float acc) {
        acc = dot2(a.x, b.x, acc);
        acc = dot2(a.y, b.y, acc);
        acc = dot2(a.z, b.z, acc);
        acc = dot2(a.w, b.w, acc);
        return acc;
    }
    static __device__ __forceinline__ float lo(uint32_t w) {
        const half2_t h = __builtin_bit_cast(half2_t, w);
        const _Float16 e = h[0];
        return (float)e;
    }
    static __device__ __forceinline__ float hi(uint32_t w) {
        const half2_t h = __builtin_bit_cast(half2_t, w);
        const _Float16 e = h[1];
        return (float)e;
    }
    static __device__ __forceinline__ void axpy(float p, const T &b, float (&acc)[ELEMS]) {
        acc[0] = __builtin_fmaf(p, lo(b.x), acc[0]); acc[1] = __builtin_fmaf(p, hi(b.x), acc[1]);
        acc[2] = __builtin_fmaf(p, lo(b.y), acc[2]); acc[3] = __builtin_fmaf(p, hi(b.y), acc[3]);
        acc[4] = __builtin_fmaf(p, lo(b.z), acc[4]); acc[5] = __builtin_fmaf(p, hi(b.z), acc[5]);
        acc[6] = __builtin_fmaf(p, lo(b.w), acc[6]); acc[7] = __builtin_fmaf(p, hi(b.w), acc[7]);
    }
};

}  // namespace sddmm
