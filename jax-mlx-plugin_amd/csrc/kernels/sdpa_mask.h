// Additive masks that vary along query rows, as the 16-bit matrix-core
// attention kernels read them: in runs of eight consecutive keys of the row
// of the query that a lane owns.
//
// Loading whole runs is what makes this kernel fast: one element at a time
// behind a branch on the type, each load waited for alone, a
// [1,16,1999,1999] bf16 bias took 1045 us a call on [4,16,1999,128] GQA;
// in runs, a tile's all in flight a tile ahead, 214 (187 with 2048 keys, whose
// rows start on a dword; 132 to 145 without a mask on the pipelined kernel).
// What is left is the mask's own vector work, 12 vector instructions a matrix
// instruction where there are 4.6 without a mask: the vector units are busy
// 51-56% of the time and the matrix cores 29-34%.  The backward of the same call
// from its residuals went from 2511 to 812 us (padding mask: 1444 to 754).
#pragma once

#include <type_traits>

#include "sdpa_elem.h"

namespace mfx {

// Mask code (beside mask_code's 1..3) of a mask of any type and key stride,
// read element by element.
constexpr int kAnyMask = 4;

// The code a kernel takes `p`'s mask with: runs need key stride 1 and a row
// of at least one run.
template <class Params>
inline int mask_run_code(const Params& p) {
  return !p.mask ? 0 : p.ms[3] != 1 || p.Tk < 8 ? kAnyMask : mask_code(p.mask_dtype);
}

// One lane's mask values of eight consecutive keys of its query row, as raw
// bits.  MT: mask_code of the mask's type.
template <int MT>
struct MaskRun {
  using Elem = std::conditional_t<MT == 1, uint32_t, uint16_t>;
  static constexpr int NW = MT == 1 ? 8 : 4;  // dwords
  // -inf throughout, which removes the keys.
  static constexpr uint32_t kOff = MT == 1 ? 0xFF800000u : MT == 2 ? 0xFF80FF80u : 0xFC00FC00u;
  uint32_t w[NW + (MT != 1)];

  // Keys key .. key + 7 of the row at `row` (key stride 1, at least eight
  // keys) as 16-byte loads on any 4-byte boundary.  A run that would pass the
  // row's end is moved back inside it; shift() undoes that.
  //
  // odd: some run may start on an odd 16-bit element.  Loads off a 4-byte
  // boundary are slow (259 against 179 us with a 1999- and a 2048-key bias),
  // so such runs load the five dwords that hold them and align() moves them
  // into place.  (No dword without a byte of the run is touched.)
  __device__ __forceinline__ void load(const Elem* row, int key, int Tk, bool odd) {
    load(row + min(key, Tk - 8), odd);
  }
  __device__ __forceinline__ void load(const Elem* at, bool odd) {
    typedef uint32_t run_t __attribute__((ext_vector_type(4), aligned(4)));
    // (Pointer arithmetic, not a cast from the rounded address: that would
    // make these flat loads, which also count as LDS operations, and the
    // backward kernels' counted LDS waits would no longer hold.)
    const int past = MT != 1 ? (int)(reinterpret_cast<uintptr_t>(at) & 2) : 0;
    const char* from = reinterpret_cast<const char*>(at) - past;
#pragma unroll
    for (int c = 0; c < NW / 4; ++c) {
      const run_t v = *reinterpret_cast<const run_t*>(from + c * 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) w[c * 4 + j] = v[j];
    }
    if constexpr (MT != 1)
      if (odd) w[4] = *reinterpret_cast<const uint32_t*>(from + 12 + 2 * past);
  }
  // After an odd load; par: 1 when the run began on an odd element.
  __device__ __forceinline__ void align(uint32_t par) {
    if constexpr (MT != 1)
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = __builtin_amdgcn_alignbit(w[j + 1], w[j], par * 16);
  }
  // At a ragged end: moves the run's first valid value back to slot 0 (the
  // slots past Tk keep something; the caller masks them).
  __device__ __forceinline__ void shift(int key, int Tk) {
    const int d = key - min(key, Tk - 8);
    if constexpr (MT == 1) {
#pragma unroll
      for (int by = 1; by < 8; by *= 2)
#pragma unroll
        for (int j = 0; j + by < 8; ++j) {
          const uint32_t a = w[j], b = w[j + by];
          w[j] = (d & by) ? b : a;
        }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t a = w[j], b = w[(j + 1) & 3];
        w[j] = (d & 1) ? a >> 16 | b << 16 : a;
      }
#pragma unroll
      for (int by = 1; by < 4; by *= 2)
#pragma unroll
        for (int j = 0; j + by < 4; ++j) {
          const uint32_t a = w[j], b = w[j + by];
          w[j] = (d & 2 * by) ? b : a;
        }
    }
  }
  __device__ __forceinline__ float get(int j) const {
    if constexpr (MT == 1) return __uint_as_float(w[j]);
    else if constexpr (MT == 2) return __uint_as_float((j & 1) ? w[j >> 1] & 0xFFFF0000u : w[j >> 1] << 16);
    else return (j & 1) ? f16_hi(w[j >> 1]) : f16_lo(w[j >> 1]);
  }
};

// Whether a run of a 16-bit mask may start on an odd element (a row does, or
// the last run of a row of odd length, moved back inside it).
template <int MT, class Params>
__device__ __forceinline__ bool mask_runs_odd(const Params& p) {
  return MT != 1 && (((reinterpret_cast<uintptr_t>(p.mask) >> 1) | p.ms[0] | p.ms[1] | p.ms[2] | p.Tk) & 1) != 0;
}

// N loaded runs, the g-th at key + g*16, put in place; ragged: they may pass Tk.
template <int MT, int N>
__device__ __forceinline__ void place_runs(MaskRun<MT> (&run)[N], const typename MaskRun<MT>::Elem* row, int key, int Tk,
                                           bool odd, bool ragged) {
  const uint32_t par = (uint32_t)(reinterpret_cast<uintptr_t>(row) >> 1) & 1;
#pragma unroll
  for (int g = 0; g < N; ++g) {
    if (odd) run[g].align(par ^ (ragged ? min(key + g * 16, Tk - 8) & 1 : 0));
    if (ragged) run[g].shift(key + g * 16, Tk);
  }
}

// Whether every lane's every value is -inf.  The first value decides for
// nearly every tile that is not.
template <int MT, int N>
__device__ __forceinline__ bool runs_all_off(const MaskRun<MT> (&run)[N]) {
  constexpr uint32_t off = MaskRun<MT>::kOff;
  if (__ballot(run[0].w[0] != off)) return false;
  uint32_t d = 0;
#pragma unroll
  for (int g = 0; g < N; ++g)
#pragma unroll
    for (int j = 0; j < MaskRun<MT>::NW; ++j) d |= run[g].w[j] ^ off;
  return __ballot(d != 0) == 0;
}

}  // namespace mfx
