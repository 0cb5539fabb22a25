// stage_math.h -- device helpers shared by the ETD2 stage kernels: lane shifts,
// buffer addressing, phi factors.  Included inside the including file's unnamed
// namespace; everything here is wave64, FP64.
#pragma once

constexpr int WAVE = 64;

// Index of this wave in its workgroup, as a wave-uniform (scalar) value: the
// compiler cannot prove threadIdx.x / 64 uniform by itself, and values read
// through it (task fields, block ranges) would otherwise live in vector
// registers behind exec-masked branches.
__device__ __forceinline__ int wave_id() {
  return __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
}

// phi factor thresholds of the reference step (solvers/etd2.py:43-46)
constexpr double PHI1_SMALL = 1e-6;
constexpr double PHI2_SMALL = 1e-3;

__device__ __forceinline__ double shfl_or_zero(double v, int src, int d) {
  const double r = __shfl(v, src < 0 ? 0 : (src > 63 ? 63 : src), WAVE);
  return (src >= 0 && src < d) ? r : 0.0;
}

// Whole-wave lane shifts by one (DPP wave_shl:1 / wave_shr:1, VALU moves, no
// LDS): lane i receives lane i+1 (lane_next; lane 63 receives 0) or lane i-1
// (lane_prev; lane 0 receives 0).  Callers keep lanes >= d at zero, so a chain
// of shifts equals shfl_or_zero at offsets of one sign.  All 64 lanes must be
// active.
constexpr int DPP_WAVE_SHL1 = 0x130;
constexpr int DPP_WAVE_SHR1 = 0x138;
template <int CTRL>
__device__ __forceinline__ double lane_shift1(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double lane_next(double v) { return lane_shift1<DPP_WAVE_SHL1>(v); }
__device__ __forceinline__ double lane_prev(double v) { return lane_shift1<DPP_WAVE_SHR1>(v); }
// value of lane l (wave-uniform l) as a scalar
__device__ __forceinline__ double readlane_f64(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Buffer resource over `bytes` bytes from base (raw, no swizzle) and 64-bit
// loads / stores at a per-lane byte offset voff plus a wave-uniform soff: the
// address arithmetic stays in scalar registers.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const double* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(base), (short)0, bytes, 0x00020000);
}
__device__ __forceinline__ double tload(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
__device__ __forceinline__ void tstore(double v, __amdgpu_buffer_rsrc_t r, int voff, int soff) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, voff, soff, 0);
}

// diagonal phi factors (solvers/etd2.py:329-390)
__device__ __forceinline__ double phi1_of(double hd, double e) {
  return (fabs(hd) > PHI1_SMALL) ? (e - 1.0) / hd : (hd * (1.0 / 6.0) + 0.5) * hd + 1.0;
}
__device__ __forceinline__ double phi2_of(double hd, double e) {
  return (fabs(hd) > PHI2_SMALL) ? ((e - 1.0) - hd) / (hd * hd)
                                 : (hd * (1.0 / 24.0) + (1.0 / 6.0)) * hd + 0.5;
}
