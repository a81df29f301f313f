// Device-side building blocks of the GRPO loss-head kernels (gfx950, wave64).
//
// Element codecs, vector row I/O, the online (max, sum-exp) pair and its wave /
// workgroup merge, and the per-token GRPO math shared by every kernel.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pcp_grpo.h"

namespace pcp {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr float kLog2e = 1.44269504088896340736f;
constexpr float kLn2 = 0.69314718055994530942f;
constexpr float kNegInf = -__builtin_inff();

// Device error conditions, raised in the context's host page (slot i for bit 1 << i); the
// host maps them to pcp_status codes after the stream is synchronised.
constexpr int kErrTokenRange = 1;
constexpr int kErrNonFinite = 2;
constexpr int kErrBadRagged = 4;   // rollout packing: offsets decrease or run past the token array
constexpr int kErrBadBase64 = 8;   // base64: a character outside the alphabet or misplaced padding
constexpr int kErrListedRow = 16;  // a row listed live by live_rows_kernel was not live in the row kernel

// A store of 1 to the condition's own slot, not an atomic OR: the page is host memory, and
// the link to the host carries no OR.
__device__ __forceinline__ void raise_error(int* err, int bit) {
  __hip_atomic_store(err + __builtin_ctz(static_cast<unsigned>(bit)), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// v_exp_f32: 2^x. Used only for the per-element softmax terms, where results
// below the fp32 normal range are irrelevant (they multiply a coefficient < 1).
__device__ __forceinline__ float hw_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// ---------------------------------------------------------------------------
// Element codecs. `unpack(w, j)` reads element j of a packed little-endian word
// array; `load1` reads one element of a row.
// ---------------------------------------------------------------------------
struct F32T {
  static constexpr int kBytes = 4;
  __device__ static __forceinline__ float unpack(const uint32_t* w, int j) {
    return __uint_as_float(w[j]);
  }
  __device__ static __forceinline__ float load1(const void* p, int64_t i) {
    return static_cast<const float*>(p)[i];
  }
};

struct BF16T {
  static constexpr int kBytes = 2;
  __device__ static __forceinline__ float unpack(const uint32_t* w, int j) {
    const uint32_t x = w[j >> 1];
    return __uint_as_float((j & 1) ? (x & 0xffff0000u) : (x << 16));
  }
  __device__ static __forceinline__ float load1(const void* p, int64_t i) {
    return __uint_as_float(static_cast<uint32_t>(static_cast<const uint16_t*>(p)[i]) << 16);
  }
};

struct F16T {
  static constexpr int kBytes = 2;
  __device__ static __forceinline__ float unpack(const uint32_t* w, int j) {
    const uint32_t x = w[j >> 1];
    const uint16_t h = (j & 1) ? static_cast<uint16_t>(x >> 16) : static_cast<uint16_t>(x & 0xffffu);
    return static_cast<float>(__builtin_bit_cast(_Float16, h));
  }
  __device__ static __forceinline__ float load1(const void* p, int64_t i) {
    return static_cast<float>(static_cast<const _Float16*>(p)[i]);
  }
};

// Pack two floats into one 32-bit word of the output element type (RNE).
template <typename TO>
__device__ __forceinline__ uint32_t pack2(float lo, float hi);
template <>
__device__ __forceinline__ uint32_t pack2<BF16T>(float lo, float hi) {
  f32x2 f = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));  // v_cvt_pk_bf16_f32
}
template <>
__device__ __forceinline__ uint32_t pack2<F16T>(float lo, float hi) {
  f32x2 f = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
}

template <typename TO>
__device__ __forceinline__ void store1(void* p, int64_t i, float v);
template <>
__device__ __forceinline__ void store1<F32T>(void* p, int64_t i, float v) {
  static_cast<float*>(p)[i] = v;
}
template <>
__device__ __forceinline__ void store1<BF16T>(void* p, int64_t i, float v) {
  static_cast<__bf16*>(p)[i] = static_cast<__bf16>(v);
}
template <>
__device__ __forceinline__ void store1<F16T>(void* p, int64_t i, float v) {
  static_cast<_Float16*>(p)[i] = static_cast<_Float16>(v);
}

// Load one 16-byte vector (kBytes*EPV == 16) of a row; `nt` selects the
// non-temporal (streaming) cache policy.
template <bool NT>
__device__ __forceinline__ u32x4 ld16(const void* base, int64_t vec_idx) {
  const u32x4* p = static_cast<const u32x4*>(base) + vec_idx;
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}

// Raw buffer resource over one row (base, size in bytes). The hardware range check
// of a raw buffer access compares the lane (VGPR) offset with num_records (the
// SGPR offset is not checked), so every access passes its full byte offset in the
// VGPR: reads past the row end return 0 and writes past it are dropped. No lane
// then needs a branch around its access (a branch around a load makes the
// compiler wait for the pending load before the other path writes the same
// registers, serialising the row), and the descriptor stays in SGPRs.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const void* p, uint32_t nbytes) {
  // dword3 0x00020000: untyped 32-bit data format, as for any raw buffer access on gfx9.
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), static_cast<short>(0),
                                           static_cast<int>(nbytes), 0x00020000);
}

// Byte offset base + add, formed at the point of use by an opaque v_add_u32. Left to
// itself the compiler computes the NCH chunk offsets of a row once and keeps them
// live from the first load to the last store (19 VGPRs at V = 151936), which pushes
// the resident kernel past its 128-VGPR budget.
__device__ __forceinline__ uint32_t fresh_off(uint32_t base, uint32_t add) {
  uint32_t r;
  asm volatile("v_add_u32 %0, %1, %2" : "=v"(r) : "s"(add), "v"(base));
  return r;
}

// Cache-policy bits of buffer accesses: 2 = NT (streaming, not retained).
constexpr int kBufNT = 2;
// sc0 | sc1 | nt: nontemporal at system scope (stores written through to memory).
constexpr int kBufNTSystem = 19;

// 16-byte load / store at byte offset `off` of a row buffer (range-checked).
template <bool NT>
__device__ __forceinline__ u32x4 buf_ld16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, NT ? kBufNT : 0));
}

template <bool NT>
__device__ __forceinline__ u32x2 buf_ld8(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, NT ? kBufNT : 0));
}

// Global streaming stores at system scope (sc0 sc1 nt: written through to memory), for
// kernels that write each byte once and whose output the next launch reads back. No
// builtin sets these bits on a global store, hence the inline assembly; the compiler
// does not track these stores, which is safe as nothing in the kernel reads them back.
__device__ __forceinline__ void store_nt_sys(u32x4 v, void* p) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1 nt" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void store_nt_sys(u32x2 v, void* p) {
  asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1 nt" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void store_nt_sys(uint32_t v, void* p) {
  asm volatile("global_store_dword %0, %1, off sc0 sc1 nt" ::"v"(p), "v"(v) : "memory");
}

// POL: the cache policy of an NT access (kBufNT or kBufNTSystem).
template <bool NT, int POL = kBufNT>
__device__ __forceinline__ void buf_st16(__amdgpu_buffer_rsrc_t r, u32x4 v, uint32_t off) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, v), r, off, 0, NT ? POL : 0);
}

// Store one output element at byte offset `off` of a row buffer (range-checked).
template <typename TO, bool NT, int POL = kBufNT>
__device__ __forceinline__ void buf_store1(__amdgpu_buffer_rsrc_t r, uint32_t off, float v) {
  if constexpr (TO::kBytes == 4) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, off, 0, NT ? POL : 0);
  } else {
    __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(pack2<TO>(v, 0.f) & 0xffffu), r, off, 0,
                                          NT ? POL : 0);
  }
}

// Pack N floats into N output elements (N * kBytes = 16 or 32 bytes) and store them
// through a row buffer at byte offset `off` (range-checked).
template <typename TO, int N, bool NT, int POL = kBufNT>
__device__ __forceinline__ void buf_store_vals(__amdgpu_buffer_rsrc_t r, uint32_t off, const float (&v)[N]) {
  if constexpr (TO::kBytes == 4) {
    static_assert(N % 4 == 0, "f32 output stores whole 16-byte vectors");
#pragma unroll
    for (int q = 0; q < N / 4; ++q) {
      u32x4 w = {__float_as_uint(v[4 * q]), __float_as_uint(v[4 * q + 1]), __float_as_uint(v[4 * q + 2]),
                 __float_as_uint(v[4 * q + 3])};
      buf_st16<NT, POL>(r, w, off + 16 * q);
    }
  } else {
    static_assert(N % 8 == 0, "16-bit output stores whole 16-byte vectors");
#pragma unroll
    for (int q = 0; q < N / 8; ++q) {
      u32x4 w = {pack2<TO>(v[8 * q], v[8 * q + 1]), pack2<TO>(v[8 * q + 2], v[8 * q + 3]),
                 pack2<TO>(v[8 * q + 4], v[8 * q + 5]), pack2<TO>(v[8 * q + 6], v[8 * q + 7])};
      buf_st16<NT, POL>(r, w, off + 16 * q);
    }
  }
}

// Store N floats as N output elements at element offset `elem` of `base`.
// N * kBytes is 8, 16 or 32 bytes; `base + elem` is aligned to that size.
template <typename TO, int N, bool NT>
__device__ __forceinline__ void store_vals(void* base, int64_t elem, const float (&v)[N]) {
  if constexpr (TO::kBytes == 4) {
    static_assert(N % 4 == 0, "f32 output stores whole 16-byte vectors");
    u32x4* p = reinterpret_cast<u32x4*>(static_cast<float*>(base) + elem);
#pragma unroll
    for (int q = 0; q < N / 4; ++q) {
      u32x4 w = {__float_as_uint(v[4 * q]), __float_as_uint(v[4 * q + 1]),
                 __float_as_uint(v[4 * q + 2]), __float_as_uint(v[4 * q + 3])};
      if constexpr (NT) __builtin_nontemporal_store(w, p + q);
      else p[q] = w;
    }
  } else {
    static_assert(N == 4 || N % 8 == 0, "16-bit output stores 8 or 16n bytes");
    if constexpr (N == 4) {
      u32x2* p = reinterpret_cast<u32x2*>(static_cast<uint16_t*>(base) + elem);
      u32x2 w = {pack2<TO>(v[0], v[1]), pack2<TO>(v[2], v[3])};
      if constexpr (NT) __builtin_nontemporal_store(w, p);
      else *p = w;
    } else {
      u32x4* p = reinterpret_cast<u32x4*>(static_cast<uint16_t*>(base) + elem);
#pragma unroll
      for (int q = 0; q < N / 8; ++q) {
        u32x4 w = {pack2<TO>(v[8 * q], v[8 * q + 1]), pack2<TO>(v[8 * q + 2], v[8 * q + 3]),
                   pack2<TO>(v[8 * q + 4], v[8 * q + 5]), pack2<TO>(v[8 * q + 6], v[8 * q + 7])};
        if constexpr (NT) __builtin_nontemporal_store(w, p + q);
        else p[q] = w;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Online log-sum-exp state in base-2 units: m = max(x) * log2(e),
// s = sum 2^(x*log2(e) - m). s == 0 means "no element yet" (m is then -inf).
// fmaxf ignores NaN, so NaN inputs never reach m; they reach s (2^NaN = NaN),
// and every step below keeps a NaN s as NaN (NaN * 0 = NaN), so a NaN logit
// always ends in a non-finite log-sum-exp. merge() is commutative bit-for-bit,
// so an xor-butterfly leaves every lane of a wave with the same value, and a
// fixed cross-wave order makes the result identical on every thread and run.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void ms_merge(float& m, float& s, float m2, float s2) {
  const float M = fmaxf(m, m2);
  const float a = (s == 0.f) ? 0.f : s * hw_exp2(m - M);
  const float b = (s2 == 0.f) ? 0.f : s2 * hw_exp2(m2 - M);
  m = M;
  s = a + b;
}

// Reference point for 2^(x*log2e - ref): the running max, or 0 while it is -inf
// (all elements so far -inf or NaN), so -inf terms give 0 and NaN terms NaN.
__device__ __forceinline__ float ms_ref(float m) { return (m == kNegInf) ? 0.f : m; }

// Rescale a running sum from reference m to reference nm (nm >= m).
__device__ __forceinline__ float ms_rescale(float s, float m, float nm) {
  return (s == 0.f) ? 0.f : s * hw_exp2(m - ms_ref(nm));
}

// log-sum-exp (natural units) of a merged state, to a few 1e-8: m and the exponent of s
// add up exactly in f64, and log2f of s's mantissa is within an ulp of 1. In f32 the sum
// m + log2f(s) and its product round at the size of the log-sum-exp (16 at V = 151,936:
// 1e-6 of every log-prob, ratio and KL term).
__device__ __forceinline__ double ms_lse(float m, float s) {
  const int k = __builtin_amdgcn_frexp_expf(s);
  const float f = log2f(__builtin_amdgcn_frexp_mantf(s));
  return (static_cast<double>(m) + static_cast<double>(k) + static_cast<double>(f)) * 0.69314718055994530942;
}

// v of the lane that DPP control CTRL names, `id` where there is none (or ROWS masks this
// lane's 16-lane row off).
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ float dpp(float id, float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, id), __builtin_bit_cast(int, v),
                                                               CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ float read_lane(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Reduction of the first N lanes (a power of two up to 64), the result on every lane (a
// scalar): row_shr 1, 2, 4, 8 leave each 16-lane row's result in its last lane, row_bcast
// 15 and 31 carry it on. The order is fixed, so the result is deterministic.
template <int N, typename F>
__device__ __forceinline__ float lanes_reduce(float v, float id, F f) {
  if constexpr (N > 1) v = f(v, dpp<0x111>(id, v));
  if constexpr (N > 2) v = f(v, dpp<0x112>(id, v));
  if constexpr (N > 4) v = f(v, dpp<0x114>(id, v));
  if constexpr (N > 8) v = f(v, dpp<0x118>(id, v));
  if constexpr (N > 16) v = f(v, dpp<0x142, 0xa>(id, v));
  if constexpr (N > 32) v = f(v, dpp<0x143, 0xc>(id, v));
  return read_lane(v, N - 1);
}
template <int N>
__device__ __forceinline__ float lanes_max(float v) {
  return lanes_reduce<N>(v, kNegInf, [](float a, float b) { return fmaxf(a, b); });
}
template <int N>
__device__ __forceinline__ float lanes_sum(float v) {
  return lanes_reduce<N>(v, 0.f, [](float a, float b) { return a + b; });
}

// The merge of the first N lanes' (m, s) pairs: the largest m, then every s rescaled to it
// once and added. NaN and -inf behave as in ms_merge.
template <int N>
__device__ __forceinline__ void lanes_merge(float& m, float& s) {
  const float M = lanes_max<N>(m);
  s = lanes_sum<N>((s == 0.f) ? 0.f : s * hw_exp2(m - M));
  m = M;
}

// Reduce two (m, s) pairs over the workgroup. `lds` holds 4 floats per wave, 16-byte
// aligned. Returns the same values on every thread. The rows' merge is a serial chain
// during which the workgroup has no load in flight: six butterfly steps through
// ds_bpermute with two exponentials each, then a chain of 15 wave results, took 1720 live
// rows of 50,257 from 151 to 168 us, 288 f32 rows of 151,936 from 135 to 138 us and 36 bf16
// ones from 54 to 57 us. (Loading the token's advantage, scale and old log-prob ahead of
// the row, so that no load follows the merge, changed none of them by more than 0.5%.)
template <int BLOCK>
__device__ __forceinline__ void block_merge2(float& m1, float& s1, float& m2, float& s2,
                                             float* lds) {
  lanes_merge<64>(m1, s1);
  lanes_merge<64>(m2, s2);
  constexpr int NW = BLOCK / 64;
  if constexpr (NW > 1) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    float4* w4 = reinterpret_cast<float4*>(lds);
    if (lane == 0) w4[wid] = make_float4(m1, s1, m2, s2);
    __syncthreads();
    const float4 w = w4[lane & (NW - 1)];
    m1 = w.x;
    s1 = w.y;
    m2 = w.z;
    s2 = w.w;
    lanes_merge<NW>(m1, s1);
    lanes_merge<NW>(m2, s2);
  }
}

// ---------------------------------------------------------------------------
// Kernel argument block (passed by value) and per-row metadata.
// ---------------------------------------------------------------------------
// Handing values from one workgroup to another in the same launch (the last of a
// group of workgroups, chosen by an atomic ticket, reads what the others wrote). A
// device-scope release fence writes back the whole L2 of the XCD (buffer_wbl2), which
// cost microseconds per workgroup here. Instead each value is stored through to the
// device-coherent level (an agent-scope atomic store), the storing wave waits for its
// stores to complete before the ticket, and the reader, after the ticket, invalidates
// its caches' copies once (an agent-scope acquire fence: buffer_inv, no write-back) and
// loads as usual, so its loads go out together. (Agent-scope atomic loads would each
// wait for the one before.)
template <typename T>
__device__ __forceinline__ void store_coherent(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// This wave's stores complete (at the level they were issued to) before what follows.
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// Before reading what other workgroups stored with store_coherent (after the ticket).
__device__ __forceinline__ void acquire_coherent() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent"); }

struct RowArgs {
  const void* logits;
  const void* ref_logits;  // nullptr => no reference pass
  const void* ids;
  const void* mask;        // nullptr => all ones
  const float* old_logp;   // nullptr => on-policy
  const float* adv;        // [n_seq]
  const float* seq_scale;  // [n_seq]: 1 / (loss_norm * max(sum mask, 1))
  void* dlogits;           // nullptr => forward only
  float* logp;
  float* ref_logp;
  float* token_loss;
  int* err;                // the context's error slots (raise_error)
  int* next_row;           // persistent row kernel: rows handed out past the first grid
  // Without zero-fill: the live rows' indices and their count, filled by
  // live_rows_kernel before the persistent row kernel, which then visits only those
  // rows. nullptr: every row in order.
  int* row_list;
  int* row_count;
  float4* part;            // RowPlan::kParts: [nrows, parts] (policy m, s, reference m, s), then
                           // [nrows] (the target's policy and reference logits, its old log-prob)
  int32_t turn;            // resident rows dealt in grid strides: where the next stride starts
  int64_t nrows;           // logits rows of the launch
  int64_t vocab;
  int64_t rows;
  int64_t logit_stride;
  int64_t tok_stride;
  int64_t tok_offset;
  int32_t ids_i64;
  int32_t mask_u8;
  int32_t loss_mode;
  int32_t zero_fill;
  int32_t counters_zeroed;  // next_row / row_count were zeroed earlier on the stream (step_prep_kernel)
  float clip_eps;
  float kl_beta;
};

struct RowMeta {
  int64_t row;   // logits row index
  int64_t tix;   // token index into ids/mask/per-token outputs (valid when tok)
  int64_t id;    // target token
  float w;       // mask weight
  int32_t seq;
  bool tok;      // row carries a token (t < rows)
  bool live;     // tok && w != 0 && id != ignore && id in range
};

__device__ __forceinline__ RowMeta row_meta(const RowArgs& a, int64_t row) {
  RowMeta r;
  r.row = row;
  // Rows number below 2^31 (checked on the host): a 32-bit division.
  const int64_t s = static_cast<uint32_t>(row) / static_cast<uint32_t>(a.logit_stride);
  const int64_t t = row - s * a.logit_stride;
  r.seq = static_cast<int32_t>(s);
  r.tok = t < a.rows;
  r.tix = s * a.tok_stride + a.tok_offset + t;
  r.id = 0;
  r.w = 0.f;
  r.live = false;
  if (r.tok) {
    r.id = a.ids_i64 ? static_cast<const int64_t*>(a.ids)[r.tix]
                     : static_cast<int64_t>(static_cast<const int32_t*>(a.ids)[r.tix]);
    if (a.mask == nullptr) r.w = 1.f;
    else if (a.mask_u8) r.w = static_cast<const uint8_t*>(a.mask)[r.tix] ? 1.f : 0.f;
    else r.w = static_cast<const float*>(a.mask)[r.tix];
    const bool ignored = (r.id == PCP_IGNORE_INDEX);
    const bool in_range = (r.id >= 0) && (r.id < a.vocab);
    if (r.w != 0.f && !ignored && !in_range) {
      if (threadIdx.x == 0) raise_error(a.err, kErrTokenRange);
    }
    r.live = (r.w != 0.f) && in_range;
  }
  return r;
}

// k3 KL estimator exp(d) - d - 1 without cancellation: for |d| < 0.5 the series
// d^2 * sum_k d^k / (k+2)! (truncated after d^7: relative error < 1e-9), else
// expm1(d) - d (cancellation below a factor of 4 there).
__device__ __forceinline__ float kl_k3(float d) {
  if (fabsf(d) < 0.5f) {
    float p = 1.f / 362880.f;
    p = fmaf(p, d, 1.f / 40320.f);
    p = fmaf(p, d, 1.f / 5040.f);
    p = fmaf(p, d, 1.f / 720.f);
    p = fmaf(p, d, 1.f / 120.f);
    p = fmaf(p, d, 1.f / 24.f);
    p = fmaf(p, d, 1.f / 6.f);
    p = fmaf(p, d, 0.5f);
    return d * d * p;
  }
  return expm1f(d) - d;
}

// Per-token loss term and d loss / d logp.
struct TokenTerms {
  float loss;  // m * l'
  float coef;  // c = d loss / d logp (already includes m / (loss_norm * L_s))
};

// lp, lr: log-probs in f64, so that the differences below lose nothing of them. old():
// the token's behaviour-policy log-prob, called only where the loss has one.
template <typename Old>
__device__ __forceinline__ TokenTerms token_terms(const RowArgs& a, const RowMeta& r, double lp, double lr, Old old) {
  TokenTerms o;
  if (a.adv == nullptr) {  // forward-only request: no loss terms
    o.loss = 0.f;
    o.coef = 0.f;
    return o;
  }
  const float A = a.adv[r.seq];
  const float scale = a.seq_scale[r.seq] * r.w;
  if (a.loss_mode == PCP_LOSS_REINFORCE) {
    // token_losses = -logp * mask; seq_nll * adv; mean  (export_qwen_forward.py:156-163)
    o.loss = r.w * static_cast<float>(-lp);
    o.coef = -A * scale;
  } else {
    // On-policy: 1, but NaN for a target of probability 0 (lp = -inf), as lp - lp is.
    const float rho = expf(static_cast<float>(lp - (a.old_logp ? static_cast<double>(old()) : lp)));
    const float lo = 1.f - a.clip_eps, hi = 1.f + a.clip_eps;
    const float rc = fminf(fmaxf(rho, lo), hi);
    const float surr = fminf(rho * A, rc * A);
    const float dlr = static_cast<float>(lr - lp);
    o.loss = r.w * (-surr + a.kl_beta * kl_k3(dlr));
    // The min picks the unclipped branch (gradient -A*rho) unless the ratio left the
    // trust region on the side the advantage's sign rewards.
    const bool unclipped = (A >= 0.f) ? (rho <= hi) : (rho >= lo);
    const float dsurr = unclipped ? -A * rho : 0.f;
    // d k3 / d logp = 1 - exp(ref - logp) = -expm1(ref - logp)
    o.coef = scale * (dsurr - a.kl_beta * expm1f(dlr));
  }
  return o;
}

__device__ __forceinline__ TokenTerms token_terms(const RowArgs& a, const RowMeta& r, double lp, double lr) {
  return token_terms(a, r, lp, lr, [&] { return a.old_logp[r.tix]; });
}

// Write per-token outputs of a token row (thread 0 only).
__device__ __forceinline__ void write_token_outputs(const RowArgs& a, const RowMeta& r, float lp,
                                                    float lr, float tl) {
  if (threadIdx.x != 0 || !r.tok) return;
  if (a.logp) a.logp[r.tix] = lp;
  if (a.ref_logp) a.ref_logp[r.tix] = lr;
  if (a.token_loss) a.token_loss[r.tix] = tl;
}

}  // namespace pcp
