// tile_common.h -- pieces shared by the MFMA tile attention kernels (gfx950):
// 16x16x32 MFMA wrappers, the swizzled LDS tile layout, the HBM -> LDS copy
// path and raw buffer loads.
#pragma once

#include "dsa_device.h"

typedef float dsa_f32x4 __attribute__((ext_vector_type(4)));
// Raw buffer loads (the LLVM intrinsics, bound by asm label, so declared
// outside any namespace).  They are typed as float on purpose: this
// toolchain's optimiser narrows the integer-vector forms (and the clang
// builtin __builtin_amdgcn_raw_buffer_load_b128) to a single dword and
// repeats it in every element.  Arguments: resource, byte offset (VGPR),
// SGPR offset, cache policy.
__device__ dsa_f32x4 buffer_load_f32x4(__amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.raw.ptr.buffer.load.v4f32");
__device__ float buffer_load_f32(__amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.raw.ptr.buffer.load.f32");
typedef float dsa_f32x2 __attribute__((ext_vector_type(2)));
__device__ dsa_f32x2 buffer_load_f32x2(__amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.raw.ptr.buffer.load.v2f32");

namespace dsa {
namespace {

constexpr int kTQ = 128;  // queries per block
constexpr int kKT = 64;   // keys per LDS tile
constexpr int kNT = 256;  // threads per block

template <typename Tag>
struct Mfma16x16x32;

template <>
struct Mfma16x16x32<BF16> {
  static __device__ __forceinline__ f32x4 run(const u32x4& a, const u32x4& b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static constexpr uint32_t kOnes = 0x3f803f80u;  // two bf16 1.0
  static __device__ __forceinline__ float dot2_ones(uint32_t w, float acc) {  // acc + w.lo + w.hi
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w),
                                           __builtin_bit_cast(bf16x2, kOnes), acc, false);
  }
  static __device__ __forceinline__ uint32_t pack(float lo, float hi) {  // one v_cvt_pk_bf16_f32
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
  }
};

template <>
struct Mfma16x16x32<F16> {
  static __device__ __forceinline__ f32x4 run(const u32x4& a, const u32x4& b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static constexpr uint32_t kOnes = 0x3c003c00u;  // two f16 1.0
  static __device__ __forceinline__ float dot2_ones(uint32_t w, float acc) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, w), __builtin_bit_cast(f16x2, kOnes), acc,
                                  false);
  }
  static __device__ __forceinline__ uint32_t pack(float lo, float hi) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), f16x2));
  }
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
#define DSA_LDS __attribute__((address_space(3)))

// One K or V tile in LDS: KT rows of D 16-bit elements, 16-byte chunk c of
// row r stored at chunk position c ^ swz(r).
template <int D, int KT = kKT>
struct TileLds {
  static constexpr int NCH = D / 8;  // 16-byte chunks per row
  static constexpr int BYTES = KT * D * 2;
  // K is read as 16-byte A fragments by 16 consecutive rows at one chunk:
  // row % NCH spreads them over NCH chunk positions.
  static __device__ __forceinline__ int swz_k(int r) { return r & (NCH - 1); }
  // V is read by the transposing 8-byte reads: 4 consecutive rows at one
  // chunk pair {2m, 2m+1} per 16-lane group; 2*(r % (NCH/2)) keeps the pair
  // together and moves it per row.
  static __device__ __forceinline__ int swz_v(int r) { return (2 * r) & (NCH - 1); }
};

// Buffer resource over one head's K or V rows from row s1 on (`head_base`
// is row 0 of this batch element at this head's columns): rows_rsrc, whose
// size ends at row T, so DMA reads of rows at or past T return zeros with no
// per-row clamp.  Those rows are never causal for any query, so they are
// masked to -inf and their zero V rows add 0.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const char* head_base, int s1, int T,
                                                          uint32_t rowbytes) {
  return rows_rsrc(head_base, s1, T, rowbytes);
}

// Issue this wave's share of the DMA of one 64-row tile into `dst`: PW
// 1 KiB instructions (buffer_load_dwordx4 ... lds: no registers, no LDS
// store instructions); off[i] is the lane's loop-invariant byte offset of
// its 16-byte chunk within the tile.  Completion is awaited with vmcnt
// before the barrier that publishes the tile.
template <int PW>
__device__ __forceinline__ void dma_tile(__amdgpu_buffer_rsrc_t rsrc, const uint32_t (&off)[PW],
                                         DSA_LDS uint8_t* dst, int wave) {
#pragma unroll
  for (int i = 0; i < PW; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, dst + (wave * PW + i) * 1024, 16,
                                             static_cast<int>(off[i]), 0, 0, 0);
}

// Wait until at most N vector-memory operations of this wave are
// outstanding: the ones issued last (a tile's score loads) may stay in
// flight, everything issued before them (the DMA) has completed.
template <int N>
__device__ __forceinline__ void wait_dma_keep() {
  __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

}  // namespace
}  // namespace dsa
