// Device helpers of the attention kernels: LDS swizzles, lane reductions,
// buffer descriptors and loads into LDS, division by launch constants.
#pragma once

#include <atomic>

#include "sage_common.h"

namespace sage {
namespace {

constexpr int kXcds = 8;                   // MI355X: workgroups are dealt round-robin to 8 XCDs
constexpr int kBufferWord3 = 0x00020000;   // gfx9 buffer descriptor word 3 (raw dword access)
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// Compute units of the current device, read once per device (256, the
// MI355X count, if the runtime cannot tell).
int device_cus() {
  constexpr int kDevs = 64;
  static std::atomic<int> cache[kDevs];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) {
    (void)hipGetLastError();
    return 256;
  }
  if (dev < kDevs) {
    const int v = cache[dev].load(std::memory_order_relaxed);
    if (v > 0) return v;
  }
  int v = 0;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) {
    (void)hipGetLastError();
    v = 256;
  }
  if (dev < kDevs) cache[dev].store(v, std::memory_order_relaxed);
  return v;
}

// Division of 0 <= n < 2^31 by a launch constant d >= 1 as a multiply and a
// shift: with l = ceil(log2 d) and m = floor(2^32 (2^l - d) / d) + 1, n / d =
// (hi32(m n) + n) >> l (Granlund and Montgomery).  The item decode divides by
// six of them; on wave-uniform operands this is four scalar instructions where
// the division is ~35 vector ones, which one wave issues at 5-8 cycles each.
struct FastDiv {
  uint32_t m, l;
};
inline FastDiv fast_div(int64_t d) {
  uint32_t l = 0;
  while ((int64_t{1} << l) < d) ++l;
  return {static_cast<uint32_t>((((uint64_t{1} << l) - static_cast<uint64_t>(d)) << 32) / static_cast<uint64_t>(d) + 1), l};
}
__host__ __device__ __forceinline__ int div_by(int n, FastDiv d) {
  const uint32_t u = static_cast<uint32_t>(n);
  return static_cast<int>((static_cast<uint32_t>((static_cast<uint64_t>(d.m) * u) >> 32) + u) >> d.l);
}

// LDS tiles are unpadded rows of 16-byte chunks; chunk c of row r is stored at
// chunk position c ^ swz(r).  gfx950's LDS serves 256 bytes (64 banks) per
// cycle, i.e. 16 lanes of a ds_read_b128; the 16 lanes of an MFMA operand read
// take one chunk each from 16 consecutive rows.  Rows r and r + 256/ROW_BYTES
// share banks, so the XOR key is the row's index among those: every 16-lane
// group then covers all 64 banks once.  The XOR is its own inverse, so the
// same function maps position -> chunk for the loads.
template <int ROW_BYTES>
__device__ __forceinline__ int swz(int row) {
  static_assert(ROW_BYTES == 256 || ROW_BYTES == 128 || ROW_BYTES == 64, "rows of 4, 8 or 16 chunks");
  constexpr int kRowsPerWindow = 256 / ROW_BYTES;
  constexpr int kChunks = ROW_BYTES / 16;
  return (row / kRowsPerWindow) & (kChunks - 1);
}

// Row-major V tiles (key rows of D fp16 values) are read with
// ds_read_b64_tr_b16, whose 16-lane groups each take 8 bytes from 4
// consecutive key rows at 4 column offsets 8 bytes apart (32 bytes of each
// row; two groups cover 64 bytes of the same 4 rows).  XOR-ing the chunk
// index with 4 * (the row's index among the 4) -- for 128-byte rows, among
// the 2 rows that share a bank window -- puts the 4 rows' 64 bytes in 4
// different quarters of the 64 banks.  The loads use the same XOR.
template <int D>
__device__ __forceinline__ int swz_vrow(int row) {
  static_assert(D == 128 || D == 64, "head_dim 64 or 128");
  return D == 128 ? 4 * (row & 3) : 4 * ((row & 3) >> 1);
}

// LDS row r of a K stage holds key kperm(r) of the tile (bits 2 and 3 swapped;
// an involution).
__device__ __forceinline__ int kperm(int r) { return (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1); }

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// max(x[lane], x[lane ^ 32]) / sum via v_permlane32_swap
__device__ __forceinline__ float xhalf_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __builtin_fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xhalf_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Log-sum-exp of a row (natural log) from its reference max m and sum l in
// log2 units: -inf without a live key (l = 0), NaN where the scores are.
__device__ __forceinline__ float row_lse(float m, float l) {
  return l == 0.0f ? -INFINITY : (m + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;
}

// Uniform 64-bit pointer (the compiler cannot always prove it).
template <typename T>
__device__ __forceinline__ const T* uniform_ptr(const T* ptr) {
  const uint64_t v = reinterpret_cast<uint64_t>(ptr);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return reinterpret_cast<const T*>((static_cast<uint64_t>(hi) << 32) | lo);
}

// Buffer descriptor over [base, base + bytes); reads past the end return 0.
// Both fields are made explicitly wave-uniform: a descriptor in VGPRs would
// turn every load into a waterfall loop.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(uniform_ptr(base)), static_cast<short>(0),
                                           static_cast<int>(__builtin_amdgcn_readfirstlane(bytes)), kBufferWord3);
}

// One 16-byte-per-lane buffer load straight into LDS (buffer_load_dwordx4
// ... lds): the wave's 64 lanes fill 1 KB at `lds_dst` + lane*16 from byte
// voffset + soffset of the buffer; lanes past the descriptor's end write
// zeros.  The builtin takes an LDS-address-space pointer, which only the
// device pass of this single-source file can form; in the host pass (which
// compiles no device code but would otherwise drop the kernels' launch stubs)
// the body is empty.
__device__ __forceinline__ void lds_direct_load16(__amdgpu_buffer_rsrc_t rsrc, char* lds_dst, uint32_t voffset,
                                                  uint32_t soffset) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(3))) void* lds_ptr;
  // the low 32 bits of a generic LDS address are the LDS offset
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, reinterpret_cast<lds_ptr>(reinterpret_cast<uintptr_t>(lds_dst)), 16,
                                           voffset, soffset, 0, 0);
#endif
}

// ds_read_b64_tr_b16 at a generic LDS address.  The restrict parameter gives
// the read an alias scope; without one the compiler assumes that it may read
// what any load into LDS still in flight writes, and waits for all of them
// (vmcnt(0)) before it, which undoes the ring's prefetch.  The kernels' own
// waits order the reads after the loads of their stage.
#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ uint2 lds_read_tr(const char* __restrict__ a) {
  typedef short short4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) short4_t* lds_s4;
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)a));
}
#endif

// Largest value over the 64 lanes, without LDS: DPP butterflies inside each
// 16-lane row, then the row and half-wave swaps.
__device__ __forceinline__ float wave_max64(float v) {
  v = __builtin_fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false)));
  v = __builtin_fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false)));
  v = __builtin_fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, false)));
  v = __builtin_fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, false)));
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __builtin_fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  return xhalf_max(v);
}

// fl(x * s) rounded half away from zero.  round_half_away_i8 without its
// clamp: x * s has a magnitude of at most 127 (1 + 2^-22) for finite x, as s =
// fl(127 / max|x|) (times Q's pre-scale, which max|x| includes), and the
// conversion turns NaN into 0.
__device__ __forceinline__ int quant1(float x, float s) {
#pragma clang fp contract(off)
  const float t = x * s;
  const float u = t + __builtin_copysignf(0.5f, t);
  int r;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(u));
  return r;
}

// 16 elements (8 dwords) -> 16 int8 (the MFMA operand of a lane)
template <bool BF16>
__device__ __forceinline__ int4_t quant16(const uint32_t (&w)[8], float s) {
  int4_t o;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float2_t a = unpack2<BF16>(w[2 * k]), b = unpack2<BF16>(w[2 * k + 1]);
    const uint32_t lo = __builtin_amdgcn_perm(quant1(a.y, s), quant1(a.x, s), 0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm(quant1(b.y, s), quant1(b.x, s), 0x04000c0cu);
    o[k] = static_cast<int>(lo | hi);
  }
  return o;
}

}  // namespace
}  // namespace sage
