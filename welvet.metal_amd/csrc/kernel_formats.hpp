// kernel_formats.hpp — the storage formats as the product kernels read them:
// kernel formats, the chunks lanes load, their decode, and the small device
// helpers the kernels of dense.hip and ragged.hpp share.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "codec.hpp"
#include "kernels.hpp"

namespace wh {
namespace {

// Kernel formats: dtypes sharing a body layout and decode share a kernel.
// FL* decode through an LDS table of 2^bits exact values; FL4P is the 4-bit
// layout read through a 256-entry table of value pairs (one read per byte);
// FE4 / FE5 decode FP8 E4M3 / E5M2 with the hardware converts, reading the
// store's decode-ready copy (codec.hpp kcode: the reference's quirks applied
// at encode / SGD time); FI8 decodes Int8 by integer conversion; FF4 decodes
// FP4 E2M1 with the hardware converts (exact for all 16 codes, no scale).
enum Fmt {
  FL1, FL2, FL3, FL4, FL5, FL6, FL8, FH16, FB16, FI16, FU16, FF32, FI32, FU32, FI64, FU64, FC64,
  FC128, FF64, FE4, FE5, FI8, FL4P, FF4, kNumFmt
};

int fmt_of(int dt) {
  switch (dt) {
  case kFloat64: return FF64;
  case kFloat32: return FF32;
  case kFloat16: return FH16;
  case kBFloat16: return FB16;
  case kFP8E4M3: case kFP8E5M2: case kInt8: case kUint8: return FL8;
  case kInt64: case kInt: return FI64;
  case kInt32: return FI32;
  case kInt16: return FI16;
  case kUint64: case kUint: case kUintptr: return FU64;
  case kUint32: return FU32;
  case kUint16: return FU16;
  case kInt4: case kUint4: case kFP4: case kNF4: return FL4;
  case kInt2: case kUint2: case kTernary: return FL2;
  case kBinary: return FL1;
  case kComplex64: return FC64;
  case kComplex128: return FC128;
  case kFP6: case kInt6: case kUint6: return FL6;
  case kInt5: case kUint5: return FL5;
  case kInt3: case kUint3: return FL3;
  }
  return -1;
}

// Chunk = the unit one lane loads: kE elements in kW dwords.
template <int F>
struct FI {
  static constexpr int kBits = F == FL1 ? 1 : F == FL2 ? 2 : F == FL3 ? 3 : (F == FL4 || F == FL4P || F == FF4) ? 4
                             : F == FL5 ? 5 : F == FL6 ? 6 : (F == FL8 || F == FE4 || F == FE5 || F == FI8) ? 8
                             : (F == FH16 || F == FB16 || F == FI16 || F == FU16) ? 16
                             : (F == FF32 || F == FI32 || F == FU32) ? 32 : F == FC128 ? 128 : 64;
  static constexpr bool kLut = (kBits <= 8 && F != FE4 && F != FE5 && F != FI8 && F != FF4) || F == FL4P;
  static constexpr bool kPair = F == FL4P;
  // floats of LDS table: 2^bits values, or 256 value pairs
  static constexpr int kTable = kPair ? 512 : (kLut ? (1 << kBits) : 1);
  static constexpr int kE = kBits <= 6 ? 32 : 128 / kBits;
  static constexpr int kW = kBits <= 6 ? kBits : 4;
  using Acc = std::conditional_t<F == FF64, double, float>;
  // decodes that can be Inf or NaN (float codes; 8-bit tables include E5M2)
  static constexpr bool kMayBeNonFinite = F == FE5 || F == FL8 || F == FH16 || F == FB16 ||
                                          F == FF32 || F == FF64 || F == FC64 || F == FC128;
};

// Fills the block's LDS table from the store's 2^bits decoded values.
template <int F>
__device__ inline void fill_table(float *tab, const float *lut, int tid, int nthreads) {
  using I = FI<F>;
  if constexpr (I::kPair) {
    for (int b = tid; b < 256; b += nthreads) {
      tab[2 * b] = lut[b & 15];
      tab[2 * b + 1] = lut[b >> 4];
    }
  } else if constexpr (I::kLut) {
    for (int i = tid; i < (1 << I::kBits); i += nthreads) tab[i] = lut[i];
  }
}

int fmt_chunk_elems(int f) {
  switch (f) {
  case FL1: case FL2: case FL3: case FL4: case FL5: case FL6: return 32;
  case FL8: case FE4: case FE5: case FI8: return 16;
  case FL4P: case FF4: return 32;
  case FH16: case FB16: case FI16: case FU16: return 8;
  case FF32: case FI32: case FU32: return 4;
  case FC128: return 1;
  default: return 2;
  }
}
int fmt_chunk_bytes(int f) {
  switch (f) {
  case FL1: return 4;
  case FL2: return 8;
  case FL3: return 12;
  case FL5: return 20;
  case FL6: return 24;
  default: return 16;
  }
}

template <int W>
__device__ inline void load_words(const uint8_t *__restrict__ p, uint32_t (&w)[W]) {
  if constexpr (W == 4) {
    const uint4 v = *(const uint4 *)p;
    w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
  } else if constexpr (W == 2) {
    const uint2 v = *(const uint2 *)p;
    w[0] = v.x; w[1] = v.y;
  } else {
#pragma unroll
    for (int i = 0; i < W; ++i) w[i] = ((const uint32_t *)p)[i];
  }
}

// Workgroup barrier for LDS hand-offs only: this wave's LDS operations are
// complete (lgkmcnt 0) and its global loads stay in flight, where
// __syncthreads' fence would also wait for every outstanding load (on this
// target one counter covers vector-memory loads and stores).  The empty asm
// statements keep the compiler from moving memory accesses across it.
__device__ inline void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0); vmcnt and expcnt at their maxima
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// load_words with the non-temporal hint (streamed weights, read once).
template <int W>
__device__ inline void load_words_nt(const uint8_t *__restrict__ p, uint32_t (&w)[W]) {
  typedef uint32_t u4v __attribute__((ext_vector_type(4)));
  typedef uint32_t u2v __attribute__((ext_vector_type(2)));
  if constexpr (W == 4) {
    const u4v v = __builtin_nontemporal_load((const u4v *)p);
    w[0] = v[0]; w[1] = v[1]; w[2] = v[2]; w[3] = v[3];
  } else if constexpr (W == 2) {
    const u2v v = __builtin_nontemporal_load((const u2v *)p);
    w[0] = v[0]; w[1] = v[1];
  } else {
#pragma unroll
    for (int i = 0; i < W; ++i) w[i] = __builtin_nontemporal_load((const uint32_t *)p + i);
  }
}

// Code of element e of a chunk (LSB-first bitstream over little-endian words).
template <int BITS, int W>
__device__ inline uint32_t chunk_code(const uint32_t (&w)[W], int e) {
  const int bit = e * BITS, word = bit >> 5, off = bit & 31;
  uint32_t v = w[word] >> off;
  if (off + BITS > 32) v |= w[word + 1] << (32 - off);
  return v & ((1u << BITS) - 1);
}

// Decoded value of element e (exact decode of the reference, widened later).
template <int F>
__device__ inline typename FI<F>::Acc chunk_value(const uint32_t (&w)[FI<F>::kW], int e,
                                                  const float *lut, float scale, float minv) {
  using I = FI<F>;
  typedef float f2 __attribute__((ext_vector_type(2)));
  if constexpr (F == FL4P) {
    const uint32_t b = (w[e >> 3] >> (8 * ((e >> 1) & 3))) & 0xffu;
    return lut[2 * b + (e & 1)];
  } else if constexpr (I::kLut) return lut[chunk_code<I::kBits, I::kW>(w, e)];
  else if constexpr (F == FF4) {
    const f2 p = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[e >> 3] >> (8 * ((e >> 1) & 3)), 1.0f, 0);
    return (e & 1) ? p[1] : p[0];
  } else if constexpr (F == FE4 || F == FE5) {
    const uint32_t q = w[e >> 2];
    f2 p;
    if (F == FE4) p = (e & 2) ? __builtin_amdgcn_cvt_pk_f32_fp8(q, true) : __builtin_amdgcn_cvt_pk_f32_fp8(q, false);
    else p = (e & 2) ? __builtin_amdgcn_cvt_pk_f32_bf8(q, true) : __builtin_amdgcn_cvt_pk_f32_bf8(q, false);
    return (e & 1) ? p[1] : p[0];
  } else if constexpr (F == FI8) return (float)(int8_t)(uint8_t)(w[e >> 2] >> (8 * (e & 3))) * scale;
  else if constexpr (F == FH16) {
    const uint16_t h = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
    return (float)__builtin_bit_cast(_Float16, h);
  } else if constexpr (F == FB16) return u2f((w[e >> 1] >> (16 * (e & 1))) << 16);
  else if constexpr (F == FI16) return (float)(int16_t)(uint16_t)(w[e >> 1] >> (16 * (e & 1))) * scale;
  else if constexpr (F == FU16) return (float)(w[e >> 1] >> (16 * (e & 1)) & 0xffffu) * scale + minv;
  else if constexpr (F == FF32) return u2f(w[e]);
  else if constexpr (F == FI32) return (float)(int32_t)w[e] * scale;
  else if constexpr (F == FU32) return (float)w[e] * scale + minv;
  else if constexpr (F == FI64) return (float)(int64_t)((uint64_t)w[2 * e] | ((uint64_t)w[2 * e + 1] << 32)) * scale;
  else if constexpr (F == FU64) return (float)((uint64_t)w[2 * e] | ((uint64_t)w[2 * e + 1] << 32)) * scale + minv;
  else if constexpr (F == FC64) return u2f(w[2 * e]);
  else if constexpr (F == FC128) return (float)u2d((uint64_t)w[0] | ((uint64_t)w[1] << 32));
  else return u2d((uint64_t)w[2 * e] | ((uint64_t)w[2 * e + 1] << 32));  // FF64
}

// All E values of a chunk, decoded before any of them is used so the table
// reads (or converts) of a chunk are independent and issue back to back.
template <int F>
__device__ inline void decode_chunk(const uint32_t (&w)[FI<F>::kW], typename FI<F>::Acc (&v)[FI<F>::kE],
                                    const float *tab, float scale, float minv) {
  using I = FI<F>;
  typedef float f2 __attribute__((ext_vector_type(2)));
  if constexpr (F == FE4 || F == FE5) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f2 lo, hi;
      if constexpr (F == FE4) {
        lo = __builtin_amdgcn_cvt_pk_f32_fp8(w[i], false);
        hi = __builtin_amdgcn_cvt_pk_f32_fp8(w[i], true);
      } else {
        lo = __builtin_amdgcn_cvt_pk_f32_bf8(w[i], false);
        hi = __builtin_amdgcn_cvt_pk_f32_bf8(w[i], true);
      }
      v[4 * i] = lo[0];
      v[4 * i + 1] = lo[1];
      v[4 * i + 2] = hi[0];
      v[4 * i + 3] = hi[1];
    }
  } else if constexpr (F == FL4P) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const uint32_t b = (w[j >> 2] >> (8 * (j & 3))) & 0xffu;
      const f2 p = ((const f2 *)tab)[b];
      v[2 * j] = p[0];
      v[2 * j + 1] = p[1];
    }
  } else if constexpr (F == FF4) {
    // byte j of the chunk holds elements 2j (low nibble) and 2j + 1
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f2 p[4] = {__builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[i], 1.0f, 0),
                       __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[i], 1.0f, 1),
                       __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[i], 1.0f, 2),
                       __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[i], 1.0f, 3)};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[8 * i + 2 * j] = p[j][0];
        v[8 * i + 2 * j + 1] = p[j][1];
      }
    }
  } else {
#pragma unroll
    for (int e = 0; e < I::kE; ++e) v[e] = chunk_value<F>(w, e, tab, scale, minv);
  }
}

template <int E>
__device__ inline void load_x(const float *__restrict__ p, float (&v)[E]) {
  if constexpr (E >= 4) {
#pragma unroll
    for (int i = 0; i < E; i += 4) {
      const float4 q = *(const float4 *)(p + i);
      v[i] = q.x; v[i + 1] = q.y; v[i + 2] = q.z; v[i + 3] = q.w;
    }
  } else if constexpr (E == 2) {
    const float2 q = *(const float2 *)p;
    v[0] = q.x; v[1] = q.y;
  } else {
    v[0] = p[0];
  }
}

template <typename T>
__device__ inline T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// A GEMV block's LDS decode table, in two steps around the weight loads:
// load() before them (so the wait for the table covers no weight load) and
// store() + lds_barrier() after they are issued.  Thread t < 64 of the block
// copies float4 entries t and t + 64 of the store's table (the pair table for
// FL4P: 128 entries; other tables have at most 64); the loads read clamped
// in-range entries.  Two named registers, no array: an array here is placed
// in LDS by the compiler.
template <int F>
struct TabCopy {
  static constexpr int kFloats = FI<F>::kTable;
  static constexpr int kQ = (kFloats + 3) / 4;
  static_assert(kQ <= 128, "two float4 per thread cover the table");
  float4 q0, q1;
  __device__ void load(const float *lut, int tid) {
    const float4 *src = (const float4 *)(FI<F>::kPair ? lut + kPairLut : lut);
    q0 = src[min(tid & 63, kQ - 1)];
    if constexpr (kQ > 64) q1 = src[min((tid & 63) + 64, kQ - 1)];
  }
  __device__ void store(float *tab, int tid) const {
    if (tid < 64 && tid < kQ) put(tab, tid, q0);
    if constexpr (kQ > 64)
      if (tid < 64 && tid + 64 < kQ) put(tab, tid + 64, q1);
  }
  __device__ static void put(float *tab, int i, float4 v) {
    if constexpr (kFloats % 4 == 0) {
      ((float4 *)tab)[i] = v;
    } else {  // tables of 2 floats (1-bit formats)
      if (4 * i < kFloats) tab[4 * i] = v.x;
      if (4 * i + 1 < kFloats) tab[4 * i + 1] = v.y;
    }
  }
};

// Kernel format of a dtype: FP8 and FP4 through the hardware converters
// (FP8 from the decode-ready copy), Int8 by integer conversion, the other
// 4-bit formats through the byte-pair table, the rest as fmt_of.
int kernel_fmt(int dt) {
  if (dt == kFP8E4M3) return FE4;
  if (dt == kFP8E5M2) return FE5;
  if (dt == kInt8) return FI8;
  if (dt == kFP4) return FF4;
  const int f = fmt_of(dt);
  return f == FL4 ? FL4P : f;
}

// Payload a kernel format reads: the decode-ready copy for the formats
// decoded by the FP8 converters (null when the store has none).
const uint8_t *kernel_body(const DevStore &w, int f) {
  return (f == FE4 || f == FE5) ? w.kbody : w.body;
}

int64_t row_bytes_of(const DevStore &w) {
  return (int64_t)w.cols * dtype_bits(w.dtype) / 8;
}

int num_cus() {
  static int n = [] {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, 0) != hipSuccess || v <= 0)
      v = 256;
    return v;
  }();
  return n;
}

#define WH_FMT_SWITCH(f, F)                                                                          \
  switch (f) {                                                                                       \
  case FL1: F(FL1); case FL2: F(FL2); case FL3: F(FL3); case FL5: F(FL5);                            \
  case FL6: F(FL6); case FL8: F(FL8); case FH16: F(FH16); case FB16: F(FB16); case FI16: F(FI16);    \
  case FU16: F(FU16); case FF32: F(FF32); case FI32: F(FI32); case FU32: F(FU32); case FI64: F(FI64); \
  case FU64: F(FU64); case FC64: F(FC64); case FC128: F(FC128); case FF64: F(FF64);                  \
  case FE4: F(FE4); case FE5: F(FE5); case FI8: F(FI8); case FL4P: F(FL4P); case FF4: F(FF4);        \
  default: return hipErrorInvalidValue;                                                              \
  }

}  // namespace
}  // namespace wh
