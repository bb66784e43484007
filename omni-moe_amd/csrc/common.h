// Device-side helpers shared by the gfx950 kernels of the OmniMoE forward path.
// Wave size is 64 throughout; nothing here is written for any other target.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <type_traits>
#include <utility>

namespace omni {

constexpr int kWave = 64;

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Storage dtypes of the operator API (values match include/omni_moe_hip.h).
enum : int { kBF16 = 0, kF16 = 1, kF32 = 2 };

// ---- scalar conversions ----------------------------------------------------
__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) { return __uint_as_float(uint32_t(b) << 16); }
__device__ __forceinline__ float bf16_lo(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }

// two floats -> packed bf16 pair, round-to-nearest-even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  f32x2_t f = {lo, hi};
  bf16x2_t r = __builtin_convertvector(f, bf16x2_t);
  return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) { return uint16_t(pack_bf16(f, 0.f) & 0xffffu); }
__device__ __forceinline__ float round_to_bf16(float f) { return bf16_lo(pack_bf16(f, 0.f)); }

__device__ __forceinline__ float f16_bits_to_f32(uint16_t b) { return float(__builtin_bit_cast(_Float16, b)); }
__device__ __forceinline__ uint16_t f32_to_f16_bits(float f) { return __builtin_bit_cast(uint16_t, _Float16(f)); }
__device__ __forceinline__ uint32_t pack_f16(float lo, float hi) {
  return uint32_t(f32_to_f16_bits(lo)) | (uint32_t(f32_to_f16_bits(hi)) << 16);
}

// Per-dtype element traits used by the bandwidth-bound kernels.
template <int DT> struct Elem;
template <> struct Elem<kBF16> {
  typedef uint16_t store_t;
  static __device__ __forceinline__ float load(const void* p, int64_t i) { return bf16_bits_to_f32(((const uint16_t*)p)[i]); }
  static __device__ __forceinline__ void store(void* p, int64_t i, float v) { ((uint16_t*)p)[i] = f32_to_bf16_bits(v); }
  static __device__ __forceinline__ float round(float v) { return round_to_bf16(v); }
};
template <> struct Elem<kF16> {
  typedef uint16_t store_t;
  static __device__ __forceinline__ float load(const void* p, int64_t i) { return f16_bits_to_f32(((const uint16_t*)p)[i]); }
  static __device__ __forceinline__ void store(void* p, int64_t i, float v) { ((uint16_t*)p)[i] = f32_to_f16_bits(v); }
  static __device__ __forceinline__ float round(float v) { return float(_Float16(v)); }
};
template <> struct Elem<kF32> {
  typedef float store_t;
  static __device__ __forceinline__ float load(const void* p, int64_t i) { return ((const float*)p)[i]; }
  static __device__ __forceinline__ void store(void* p, int64_t i, float v) { ((float*)p)[i] = v; }
  static __device__ __forceinline__ float round(float v) { return v; }
};

// ---- wave-level primitives ---------------------------------------------------
__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

// Another lane's value by a DPP control under which every lane reads a lane that is there.  With no value to keep and no lane left out, the exchange becomes an
// operand of the instruction that takes it (where that has such a form), instead of a copy and a move in front of it.
template <int CTRL> __device__ __forceinline__ int dpp_i(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true); }
template <int CTRL> __device__ __forceinline__ float dpp_f(float v) { return __int_as_float(dpp_i<CTRL>(__float_as_int(v))); }
enum : int { kQuadXor1 = 0xB1, kQuadXor2 = 0x4E, kQuadXor3 = 0x1B, kRowRor4 = 0x124, kRowXor8 = 0x128, kRowXor15 = 0x140, kRowXor7 = 0x141 };      // quad_perm, row_ror, row_mirror, row_half_mirror

// Over all 64 lanes, in every lane: lane distances 32, 16, 8, 4, 2, 1.  The two swaps leave a lane with its own value and the other's in one order or the
// other; from distance 8 on a rotation inside 16 lanes reaches the partner, or one that holds the same.  Six steps of register exchanges: through
// ds_bpermute (__shfl_xor) each step is a round trip to LDS
// (the layer for one token 19.9 -> 19.2 us, for 48 24.4 -> 23.9, the router stage at 4096 tokens 20.5 -> 20.2).
__device__ __forceinline__ float wave_sum(float v) {
  const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = __int_as_float((int)s32[0]) + __int_as_float((int)s32[1]);
  const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = __int_as_float((int)s16[0]) + __int_as_float((int)s16[1]);
  v += dpp_f<kRowXor8>(v);
  v += dpp_f<kRowRor4>(v);
  v += dpp_f<kQuadXor2>(v);
  return v + dpp_f<kQuadXor1>(v);
}
// Spelled out: fmaxf is two instructions more a step, which quiet signalling NaNs (no arithmetic result is one).  The waits are what a DPP operand asks for behind the
// instruction that wrote it; the last one is for a DPP operand of the compiler's, who does not see what wrote this one.
__device__ __forceinline__ float wave_max(float v) {
  const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = fmaxf(__int_as_float((int)s32[0]), __int_as_float((int)s32[1]));
  const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = fmaxf(__int_as_float((int)s16[0]), __int_as_float((int)s16[1]));
  asm("s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\tv_max_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\tv_max_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\ts_nop 1" : "+v"(v));
  return v;
}

// Value of lane (lane ^ STRIDE) without touching LDS memory: DPP (1, 2, 8; 4 as 7 and 3), a ds_swizzle bit pattern (16), v_permlane32_swap (32).
template <int STRIDE>
__device__ __forceinline__ int xor_lane_i(int v, int lane) {
  if constexpr (STRIDE == 1) return dpp_i<kQuadXor1>(v);
  else if constexpr (STRIDE == 2) return dpp_i<kQuadXor2>(v);
  else if constexpr (STRIDE == 4) return dpp_i<kQuadXor3>(dpp_i<kRowXor7>(v));
  else if constexpr (STRIDE == 8) return dpp_i<kRowXor8>(v);
  else if constexpr (STRIDE == 16) return __builtin_amdgcn_ds_swizzle(v, 0x401F);
  else {
    const auto sw = __builtin_amdgcn_permlane32_swap(v, v, false, false);         // [lo,lo] and [hi,hi]
    return (lane & 32) ? (int)sw[0] : (int)sw[1];
  }
}
template <int STRIDE>
__device__ __forceinline__ float xor_lane_f(float v, int lane) {
  return __int_as_float(xor_lane_i<STRIDE>(__float_as_int(v), lane));
}

// ---- loads into LDS --------------------------------------------------------------
// 16 bytes per lane from base + off + more (zeros past `bytes`; the check counts both offsets) to 1 KiB of LDS.  Spelled out, so that the compiler does not take part in counting
// it: it would put a wait for ALL outstanding loads in front of every transposing read that follows one, because it cannot tell
// the two places in LDS apart (4096 x 1024 x 4096, both operands transposed, 256 x 256 tiles: 113 us so, 92 us without).  The kernels
// that use it do their own waiting.
template <int kAt>
__device__ __forceinline__ void load_to_lds(uint64_t base, int bytes, uint32_t lds_base, uint32_t off, int more) {
  const u32x4_t r = {(uint32_t)base, (uint32_t)(base >> 32), (uint32_t)bytes, 0x00020000u};
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds_base), "v"(off), "s"(r), "s"(more), "n"(kAt)
               : "memory", "scc");   // (and m0, which nothing else here uses)
}
__device__ __forceinline__ void lds_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
template <int N> __device__ __forceinline__ void vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// sigmoid(x), x*sigmoid(x) in fp32, IEEE division.
__device__ __forceinline__ float sigmoid_f32(float x) { return 1.0f / (1.0f + __expf(-x)); }
__device__ __forceinline__ float silu_f32(float x) { return x / (1.0f + __expf(-x)); }
// Same with the hardware reciprocal (1 ulp) and exp2: ~6 instructions.  For results that are
// rounded to a 16-bit type straight away.
__device__ __forceinline__ float silu_fast(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.4426950408889634f));
}

// f(0, 1, ...), with the numbers as types: what depends on them is decided at compile time
template <class F, int... I>
__device__ __forceinline__ void with_sequence(F& f, std::integer_sequence<int, I...>) { f(std::integral_constant<int, I>{}...); }

// ---- host side ---------------------------------------------------------------
// A kernel whose dynamic LDS exceeds the 64 KiB default needs its limit raised once per device (the
// attribute belongs to the device's copy of the kernel).  Every such kernel is one LdsKernel object with
// static storage: its constructor links it into a list at library load, so that omni_init() can raise all
// limits up front (a caller that captures HIP graphs wants no hipFuncSetAttribute inside a capture), and
// ensure() does it on first use for callers that never call omni_init().  `done` is the bit mask of devices
// already set up; concurrent callers at worst set the attribute twice.
struct LdsKernel;
inline LdsKernel*& lds_kernel_list() {
  static LdsKernel* head = nullptr;
  return head;
}
struct LdsKernel {
  const void* kernel;
  int bytes;
  std::atomic<uint64_t> done{0};
  LdsKernel* next;
  LdsKernel(const void* k, int b) : kernel(k), bytes(b), next(lds_kernel_list()) { lds_kernel_list() = this; }
  hipError_t ensure() {
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
    if (hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes); e != hipSuccess) return e;
    done.fetch_or(bit, std::memory_order_release);
    return hipSuccess;
  }
};

// The schedule's allocation-free entry point keeps a device array; this resolves its address on the
// current device (defined beside the array).
int schedule_scratch_prepare();

}  // namespace omni
