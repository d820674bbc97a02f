// Pipelined MFMA main loop for the ragged per-band GEMMs.
//
// A block computes C[BR x BC] += A[BR x K] * B[BC x K]^T with both operands
// staged in LDS as [rows][pitch] (K contiguous) in chunks of 32.  Two LDS
// buffers and one or two register copies keep the global loads of the next one
// or two chunks in flight during the MFMAs of chunk k; one barrier per chunk.
//
// LDS layout (16-bit types): row r, element k of a chunk lives at
//   r * pitch + 8 * ((k / 8) ^ ((r / 16) % 4)) + k % 8,
// i.e. the four 16-byte k-units of a row are XOR-swizzled by the row's 16-row
// group.  MFMA fragment reads (16 consecutive rows, one unit) stay 16-byte
// aligned and conflict-free, and the transposed stores of MNLoader (8 bytes to
// rows 4q..4q+3) spread over all banks.
//
// fp32 tiles use a plain odd pitch and the fp32 MFMAs, whose sum of a result is the chain of fused
// multiply-adds over k, bit for bit.  Large fp32 products (split_macs) take SPLIT instead: each value is
// split on its way into LDS into three bf16 numbers, x = x1 + x2 + x3 (each the rest's round-to-nearest
// bf16), and a product is the six bf16 MFMAs a1 b1, a1 b2, a2 b1, a2 b2, a1 b3, a3 b1 with fp32
// accumulation; the three left out come to at most 2^-24 of it, 2^-27.5 in the mean square.  The sum is
// exact (8 + 8 + 8 significant bits) from 2^-110 on; below, x3's last bits fall under bf16's smallest
// number, 2^-133.  bf16 products are exact in fp32, so the result's error stays that of the fp32 sums
// (measured against 64 bits: no larger than with the fp32 MFMAs), at 6 x 16 matrix-core cycles per 16 x 16
// x 32 instead of 8 x 32, and 3 LDS reads of 16 bytes per fragment instead of 8 of 4.  A tile holds three
// planes, of 64-byte rows (swz_k) or, from an MNLoader, of 32 K-rows as they are stored (swz_mn_p; read
// transposed).  A block that has met a number other than 0 below 2^-110, or has a non-finite accumulator
// (an infinity or a NaN among the inputs, or one above bf16's largest, whose split is not finite; or an
// overflow), goes through the sum again on the fp32 MFMAs, which give such inputs their usual results.
//
// Waves are laid out WR x WC over the tile; wave (wr, wc) owns rows
// [wr * BR/WR, ...) and columns [wc * BC/WC, ...) as TR x TC 16x16 tiles.
// Result layout (mfma.h): lane l of tile (i, j) holds
//   C[row0 + 16 i + 4 (l / 16) + r][col0 + 16 j + (l % 16)],  r = 0..3.
//
// Loaders move one 32-wide K chunk:  fetch(k0, regs) global -> registers,
// commit(regs, lds) registers -> LDS (fetch_edge / commit_edge for a partial chunk);
// prepare() runs once before the first chunk.
#pragma once

#include <type_traits>

#include "mfma.h"

namespace pmsst {

constexpr int kGemmThreads = 256;

// ---------------------------------------------------------------- LDS swizzles and fragment reads
// ds_read_b128 serves 16 lanes a cycle: lanes 0-3, 12-15, 20-27, then 4-11, 16-19, 28-31, and the
// same of the upper half.  In a fragment read those are rows 0-3 and 12-15 of one unit and rows 4-11
// of the next (or the reverse), and rows 4 apart share a bank quarter at the 64-byte pitch, so the
// swizzles s(q) of the row quads q must make s(0), s(3), 1 ^ s(1), 1 ^ s(2) distinct: s = 0, 3, 2, 1.
// (s = 0, 1, 2, 3 and (r / 2) ^ (r / 8) collide two by two.)  GEMM1 of the one-pass MLP reads rows
// 8 (r / 4) + r % 4 (+ 4), which s = 0, 3, 2, 1 spreads too.
__device__ __forceinline__ int swz_k(int r) { return -(r >> 2) & 3; }
// A transpose read takes 8 bytes of each of 32 lanes a cycle: K-rows k, k + 1, k + 2, k + 3 and the
// same + 8, 32 bytes of each, which must fill the 256 bytes of the 64 banks.  At a pitch of whole
// 256 bytes every row starts on bank 0, so the 8 rows take 8 different unit pairs; at an odd multiple
// of 128 bytes odd rows start half way round, and the 4 rows of a parity take the 4 pairs of a half.
// Rows k and k + 4 keep the same swizzle, as the second read of a fragment needs.  The swizzle stays
// inside aligned groups of 16 (or 8) units, which the pitch holds whole.
template <int PITCH>
__device__ __forceinline__ int swz_mn_p(int k) {
  static_assert(PITCH % 128 == 0, "rows of whole 128 bytes");
  if constexpr (PITCH % 256 == 0) return 2 * ((k & 3) | (((k >> 3) & 1) << 2));
  else return 2 * (((k >> 1) & 1) | (((k >> 3) & 1) << 1));
}

// First of the two transpose reads of an MN-contiguous fragment (columns c0 .. c0 + 15,
// c0 % 16 == 0, row pitch PITCH bytes); the second is at + 4 * PITCH.
template <int PITCH>
__device__ __forceinline__ uint32_t frag_mn_addr_p(uint32_t region, int c0, int lane) {
  const int j = lane & 15, g = lane >> 4;
  const int k = 8 * g + (j >> 2);                // K-row of this lane's 4 elements
  const int col = c0 + 4 * (j & 3);
  const int unit = col >> 3;
  return region + static_cast<uint32_t>(k * PITCH + 16 * (unit ^ swz_mn_p<PITCH>(k)) + 2 * (col & 7));
}

typedef short s16x4_t __attribute__((ext_vector_type(4)));

// Transposed fragment (two ds_read_b64_tr_b16 through the compiler's builtin, which it waits for)
__device__ __forceinline__ u32x4_t tr_frag(const char* p, int step) {
  typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
  const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
  const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + step));
  const uint2 a = __builtin_bit_cast(uint2, lo), b = __builtin_bit_cast(uint2, hi);
  return u32x4_t{a.x, a.y, b.x, b.y};
}

template <typename T>
__device__ __forceinline__ int lds_index(int r, int k) {
  constexpr int P = LdsPitch<T>::value;
  if constexpr (sizeof(T) == 2) {
    return r * P + ((((k >> 3) ^ ((r >> 4) & 3)) << 3) | (k & 7));
  } else {
    return r * P + k;
  }
}

// acc += A rows (ra..) x B rows (rb..) over one 32-wide chunk; `ra` / `rb` are the
// lane's row indices inside the A / B tiles.
template <typename T>
__device__ __forceinline__ f32x4_t mfma_tile(const T* __restrict__ a, int ra, const T* __restrict__ b, int rb,
                                             f32x4_t acc, int lane) {
  if constexpr (sizeof(T) == 2) {
    const int k = (lane >> 4) * 8;
    return mfma_chunk<T>(a + lds_index<T>(ra, k) - k, b + lds_index<T>(rb, k) - k, acc, lane);
  } else {
    return mfma_chunk<T>(a + ra * LdsPitch<T>::value, b + rb * LdsPitch<T>::value, acc, lane);
  }
}

// ---------------------------------------------------------------- loads
// K is walked in chunks of 32 that END at K: chunk c covers k in [kbeg + 32 c, kbeg + 32 c + 32)
// with kbeg = K - 32 ceil(K / 32) <= 0, so only chunk 0 can be partial (k < 0 masked).
// Loaders therefore have two paths:
//  * interior chunks (fetch / commit): rows / columns outside the tile's valid range are
//    CLAMPED to a valid one when the loader is prepared (their products only reach outputs
//    the epilogue discards), every k is in range, and each load is a uniform chunk base plus a
//    per-lane 32-bit byte offset computed once -- no per-chunk address arithmetic or masking;
//  * the partial chunk 0 (fetch_edge / commit_edge): loads never branch on bounds (an
//    out-of-range lane reads a valid element and records a bit) and commit_edge zeroes them.
// With V4 false (widths or strides not multiples of 4 elements) every chunk takes the
// element-wise guarded path.

template <typename T>
using raw_t = typename std::conditional<sizeof(T) == 2, uint16_t, uint32_t>::type;
// 4 consecutive elements as raw bits: 8 bytes for 16-bit types, 16 for fp32.
template <typename T>
using quad_t = typename std::conditional<sizeof(T) == 2, uint2, uint4>::type;

// LDS floats per tile row of a split tile: three bf16 planes of 64 bytes (the fp32 re-run's rows of
// LdsPitch<float> fit in them).
constexpr int kSplitRow = 48;
static_assert(kSplitRow >= LdsPitch<float>::value, "the fp32 re-run's tile fits");

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// Two fp32 values as three words of two bf16 each, high part first.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t (&w)[3]) {
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    w[p] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
    if (p < 2) {
      a -= __uint_as_float(w[p] << 16);
      b -= __uint_as_float(w[p] & 0xffff0000u);
    }
  }
}

// The least of 2 |x| - 1, as bits, over the numbers a thread has split (0 counts as the largest): below
// kSplitLeast some number other than 0 is under 2^-110.
constexpr uint32_t kSplitLeast = 2u * (17u << 23) - 1u;
__device__ __forceinline__ void note_least(const float (&v)[4], uint32_t& least) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t b = 2u * __float_as_uint(v[j]) - 1u;
    least = b < least ? b : least;
  }
}

// Byte offset of element (r, k) inside plane 0 of a split tile; plane p is p * ROWS * 64 bytes on.
__device__ __forceinline__ int split_offset(int r, int k) {
  return r * 64 + 16 * ((k >> 3) ^ swz_k(r & 15)) + 2 * (k & 7);
}

// 4 consecutive k (k % 4 == 0) of row r into the three planes.
template <int ROWS>
__device__ __forceinline__ void put_split(float* lds, int r, int k, const float (&v)[4], uint32_t& least) {
  note_least(v, least);
  char* dst = reinterpret_cast<char*>(lds) + split_offset(r, k);
  uint32_t lo[3], hi[3];
  split_pair(v[0], v[1], lo);
  split_pair(v[2], v[3], hi);
#pragma unroll
  for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2*>(dst + p * ROWS * 64) = make_uint2(lo[p], hi[p]);
}

// 4 consecutive rows mn (mn % 4 == 0) of K-row k into the three planes of a tile that keeps K-rows.
template <int ROWS>
__device__ __forceinline__ void put_split_mn(float* lds, int mn, int k, const float (&v)[4], uint32_t& least) {
  note_least(v, least);
  char* dst = reinterpret_cast<char*>(lds) + k * 2 * ROWS + 16 * ((mn >> 3) ^ swz_mn_p<2 * ROWS>(k)) + 2 * (mn & 7);
  uint32_t lo[3], hi[3];
  split_pair(v[0], v[1], lo);
  split_pair(v[2], v[3], hi);
#pragma unroll
  for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2*>(dst + p * ROWS * 64) = make_uint2(lo[p], hi[p]);
}

template <typename T>
__device__ __forceinline__ quad_t<T> raw_quad(const T* p) {
  return *reinterpret_cast<const quad_t<T>*>(p);
}

// Quad at a uniform base plus a per-lane byte offset (global_load with an SGPR base).
template <typename T>
__device__ __forceinline__ quad_t<T> quad_at(const T* base, uint32_t byte_off) {
  return *reinterpret_cast<const quad_t<T>*>(reinterpret_cast<const char*>(base) + byte_off);
}

template <typename T>
__device__ __forceinline__ quad_t<T> mask_quad(quad_t<T> q, bool ok) {
  q.x = ok ? q.x : 0u;
  q.y = ok ? q.y : 0u;
  if constexpr (sizeof(T) == 4) {
    q.z = ok ? q.z : 0u;
    q.w = ok ? q.w : 0u;
  }
  return q;
}

// Element-wise guarded quad: element j is loaded when `ok` and lo <= j < hi, else zero.
template <typename T>
__device__ __forceinline__ quad_t<T> load_quad_scalar(const T* p, const T* safe, bool ok, int lo, int hi) {
  uint32_t e[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const bool in = ok && j >= lo && j < hi;
    const raw_t<T> v = *reinterpret_cast<const raw_t<T>*>(in ? p + j : safe);
    e[j] = in ? static_cast<uint32_t>(v) : 0u;
  }
  quad_t<T> q;
  if constexpr (sizeof(T) == 2) {
    q.x = e[0] | (e[1] << 16);
    q.y = e[2] | (e[3] << 16);
  } else {
    q.x = e[0];
    q.y = e[1];
    q.z = e[2];
    q.w = e[3];
  }
  return q;
}

// Edge-path quad of elements k .. k+3 of a row (valid range [0, k_valid)): with V4 the quad is
// wholly in or out (raw load recording a validity bit, masked at commit); otherwise element-wise.
template <typename T, bool V4>
__device__ __forceinline__ quad_t<T> fetch_quad_k(const T* p, const T* safe, bool row_ok, int k, int k_valid,
                                                  uint32_t& okbits, int bit) {
  if constexpr (V4) {
    const bool ok = row_ok && k >= 0 && k < k_valid;
    okbits |= static_cast<uint32_t>(ok) << bit;
    return raw_quad<T>(ok ? p : safe);
  } else {
    okbits |= 1u << bit;
    return load_quad_scalar<T>(p, safe, row_ok, -k, k_valid - k);
  }
}

template <typename T>
__device__ __forceinline__ void quad_to_f32(const quad_t<T>& q, float (&o)[4]) {
  if constexpr (sizeof(T) == 2) {
    const Pack<T, 4> pk = __builtin_bit_cast(Pack<T, 4>, q);
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = to_f32(pk.v[j]);
  } else {
    o[0] = __uint_as_float(q.x);
    o[1] = __uint_as_float(q.y);
    o[2] = __uint_as_float(q.z);
    o[3] = __uint_as_float(q.w);
  }
}

// Stores a quad of consecutive k (kq % 4 == 0) of LDS row r (SPLIT: fp32 as three bf16 planes; `least` as
// note_least keeps it).
template <typename T, int ROWS, bool SPLIT>
__device__ __forceinline__ void commit_quad(T* lds, int r, int kq, const quad_t<T>& q,
                                            [[maybe_unused]] uint32_t& least) {
  if constexpr (SPLIT) {
    const float v[4] = {__uint_as_float(q.x), __uint_as_float(q.y), __uint_as_float(q.z), __uint_as_float(q.w)};
    put_split<ROWS>(lds, r, kq, v, least);
  } else if constexpr (sizeof(T) == 2) {
    *reinterpret_cast<uint2*>(lds + lds_index<T>(r, kq)) = q;
  } else {
    uint32_t* row = reinterpret_cast<uint32_t*>(lds);
    row[lds_index<T>(r, kq + 0)] = q.x;
    row[lds_index<T>(r, kq + 1)] = q.y;
    row[lds_index<T>(r, kq + 2)] = q.z;
    row[lds_index<T>(r, kq + 3)] = q.w;
  }
}

// K-contiguous rows: element (r, k) = base[row(r) * stride + k].  Thread t moves the quad
// (r, k) = (t / 8 + 32 i, 4 (t % 8)) of every chunk, i < ROWS / 32.  By default row(r) = r for
// r < rows_valid; prepare_rows() lets a kernel map tile rows to other source rows.
template <typename T, int ROWS, bool V4>
struct KRowLoader {
  static constexpr bool kTransposed = false;  // the split tile's layout: rows
  static constexpr int kQuads = ROWS * (kChunkK / 4) / kGemmThreads;
  static_assert(kQuads >= 1 && ROWS * (kChunkK / 4) % kGemmThreads == 0, "tile too small");
  struct Regs {
    quad_t<T> q[kQuads];
    uint32_t ok;
  };
  const T* base;
  int64_t stride;
  int rows_valid;
  int k_valid;
  int64_t src_row[kQuads] = {};  // source row of each of the thread's tile rows (clamped)
  uint32_t off[kQuads] = {};     // byte offset of (src_row, k = 4 (t % 8)) from base
  uint32_t rowok = 0;            // bit i: tile row i of this thread is a real row
  mutable uint32_t least = ~0u;  // see note_least

  // For a second run of the K loop: what it derives from its rows is derived again, not kept in registers
  // through the first run.
  __device__ __forceinline__ void forget() { asm volatile("" : "+v"(rows_valid)); }
  static __device__ __forceinline__ int tile_row(int i) {
    return (static_cast<int>(threadIdx.x) + i * kGemmThreads) / (kChunkK / 4);
  }
  static __device__ __forceinline__ int lane_k() { return (threadIdx.x % (kChunkK / 4)) * 4; }

  __device__ __forceinline__ void prepare() {
    rowok = 0;
#pragma unroll
    for (int i = 0; i < kQuads; ++i) {
      const int r = tile_row(i);
      src_row[i] = r < rows_valid ? r : rows_valid - 1;
      rowok |= static_cast<uint32_t>(r < rows_valid) << i;
    }
    finish_prepare();
  }
  // Call after filling src_row and rowok (custom row maps).
  __device__ __forceinline__ void finish_prepare() {
#pragma unroll
    for (int i = 0; i < kQuads; ++i)
      off[i] = static_cast<uint32_t>((src_row[i] * stride + lane_k()) * static_cast<int64_t>(sizeof(T)));
  }
  __device__ __forceinline__ bool row_ok(int i) const { return (rowok >> i) & 1; }

  __device__ __forceinline__ void fetch_edge(int k0, Regs& g) const {
    const int k = k0 + lane_k();
    g.ok = 0;
#pragma unroll
    for (int i = 0; i < kQuads; ++i)
      g.q[i] = fetch_quad_k<T, V4>(base + src_row[i] * stride + k, base, row_ok(i), k, k_valid, g.ok, i);
  }
  template <bool SPLIT>
  __device__ __forceinline__ void commit_edge(const Regs& g, T* lds) const {
#pragma unroll
    for (int i = 0; i < kQuads; ++i)
      commit_quad<T, ROWS, SPLIT>(lds, tile_row(i), lane_k(), mask_quad<T>(g.q[i], (g.ok >> i) & 1), least);
  }
  __device__ __forceinline__ void fetch(int k0, Regs& g) const {
    if constexpr (V4) {
#pragma unroll
      for (int i = 0; i < kQuads; ++i) g.q[i] = quad_at<T>(base + k0, off[i]);
    } else {
      fetch_edge(k0, g);
    }
  }
  template <bool SPLIT>
  __device__ __forceinline__ void commit(const Regs& g, T* lds) const {
    if constexpr (V4) {
#pragma unroll
      for (int i = 0; i < kQuads; ++i) commit_quad<T, ROWS, SPLIT>(lds, tile_row(i), lane_k(), g.q[i], least);
    } else {
      commit_edge<SPLIT>(g, lds);
    }
  }
};

// MN-contiguous source: element (k, mn) = base[k * kstride + mn], staged transposed into
// lds[mn][k].  A thread owns a block of KB consecutive k rows x 4 consecutive mn
// (consecutive threads take consecutive mn quads, so each global load is coalesced along mn),
// transposes it in registers and stores KB consecutive k values per mn row.  KB = ROWS / 32 so
// one block per thread covers the chunk.  Optional scales: per-mn `cs[mn]`, per-k
// `rs[k * rs_stride] * rs_mul`; `colsum` also sums the unscaled values of the thread's mn quad
// over its k rows (e.g. a bias gradient, see reduce_colsum).  Unscaled 16-bit interior chunks
// are transposed as raw bits (byte permutes, no conversions).
template <typename T, int ROWS, bool V4>
struct MNLoader {
  static constexpr bool kTransposed = true;  // the split tile's layout: K-rows
  static constexpr int kQuadsPerK = ROWS / 4;
  static constexpr int KB = ROWS / 32;
  static_assert(KB >= 1 && KB * kQuadsPerK * (kChunkK / KB) == ROWS * kChunkK / 4, "tile shape");
  static_assert(kQuadsPerK * (kChunkK / KB) == kGemmThreads, "one block per thread");
  struct Regs {
    quad_t<T> q[KB];
    float s[KB];
    uint32_t ok;
  };
  const T* base;
  int64_t kstride;
  int mn_valid;
  int k_valid;
  const T* cs = nullptr;        // per-mn scale, or null
  const float* rs = nullptr;    // per-k scale, or null
  int64_t rs_stride = 1;
  float rs_mul = 1.f;
  bool colsum = false;
  float c[4] = {1.f, 1.f, 1.f, 1.f};       // per-mn scale of this thread's quad
  mutable float csum[4] = {0.f, 0.f, 0.f, 0.f};
  int mn_src = 0;                          // this thread's (clamped) mn quad start
  uint32_t off[KB] = {};                   // byte offset of (kb + t, mn_src) from a chunk base
  mutable uint32_t least = ~0u;            // see note_least

  __device__ __forceinline__ void forget() { asm volatile("" : "+v"(mn_valid)); }
  static __device__ __forceinline__ int lane_mn() { return (threadIdx.x % kQuadsPerK) * 4; }
  static __device__ __forceinline__ int lane_kb() { return (threadIdx.x / kQuadsPerK) * KB; }

  __device__ __forceinline__ void prepare() {
    const int mn = lane_mn();
    mn_src = (V4 && mn >= mn_valid) ? mn_valid - 4 : mn;
#pragma unroll
    for (int t = 0; t < KB; ++t)
      off[t] = static_cast<uint32_t>(((lane_kb() + t) * kstride + mn_src) * static_cast<int64_t>(sizeof(T)));
    if (cs != nullptr) quad_to_f32<T>(load_quad_scalar<T>(cs + mn, cs, true, 0, mn_valid - mn), c);
  }

  __device__ __forceinline__ void fetch_edge(int k0, Regs& g) const {
    const int mn = lane_mn();
    g.ok = 0;
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      const int k = k0 + lane_kb() + t;
      const bool kok = k >= 0 && k < k_valid;
      const int kc = kok ? k : 0;
      if constexpr (V4) {
        g.ok |= static_cast<uint32_t>(kok) << t;
        g.q[t] = raw_quad<T>(kok ? base + static_cast<int64_t>(k) * kstride + mn_src : base);
      } else {
        g.ok |= 1u << t;
        g.q[t] = load_quad_scalar<T>(base + static_cast<int64_t>(kc) * kstride + mn, base, kok, 0, mn_valid - mn);
      }
      g.s[t] = rs != nullptr ? rs[static_cast<int64_t>(kc) * rs_stride] : 1.f;
    }
  }
  __device__ __forceinline__ void fetch(int k0, Regs& g) const {
    if constexpr (V4) {
      const T* kb = base + static_cast<int64_t>(k0) * kstride;
#pragma unroll
      for (int t = 0; t < KB; ++t) {
        g.q[t] = quad_at<T>(kb, off[t]);
        g.s[t] = rs != nullptr ? rs[static_cast<int64_t>(k0 + lane_kb() + t) * rs_stride] : 1.f;
      }
    } else {
      fetch_edge(k0, g);
    }
  }

  // Float path: optional masking of k rows (edge), column sums, scales.
  template <bool SPLIT>
  __device__ __forceinline__ void commit_f32(const Regs& g, T* lds, bool masked) const {
    const int mn = lane_mn();
    const int kb = lane_kb();
    float v[KB][4];
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      quad_to_f32<T>(masked ? mask_quad<T>(g.q[t], (g.ok >> t) & 1) : g.q[t], v[t]);
      if (colsum) {
#pragma unroll
        for (int j = 0; j < 4; ++j) csum[j] += v[t][j];
      }
      const float st = rs != nullptr ? g.s[t] * rs_mul : 1.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[t][j] *= st * c[j];
    }
    if constexpr (SPLIT) {
#pragma unroll
      for (int t = 0; t < KB; ++t) put_split_mn<ROWS>(lds, mn, kb + t, v[t], least);
      return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (sizeof(T) == 2) {
        float col[KB];
#pragma unroll
        for (int t = 0; t < KB; ++t) col[t] = v[t][j];
        store_pack<T, KB>(lds + lds_index<T>(mn + j, kb), col);
      } else {
#pragma unroll
        for (int t = 0; t < KB; ++t) lds[lds_index<T>(mn + j, kb + t)] = v[t][j];
      }
    }
  }
  // Raw transpose of 16-bit values: element j of quad t is the 16-bit half (j & 1) of word
  // (j >> 1); pairs of k rows are merged into one 32-bit word per mn with a byte permute.
  __device__ __forceinline__ void commit_raw16(const Regs& g, T* lds) const {
    const int mn = lane_mn();
    const int kb = lane_kb();
    constexpr uint32_t kLo = 0x05040100u, kHi = 0x07060302u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t w[(KB + 1) / 2];
#pragma unroll
      for (int t = 0; t + 1 < KB; t += 2) {
        const uint32_t a = (j >> 1) ? g.q[t].y : g.q[t].x;
        const uint32_t b = (j >> 1) ? g.q[t + 1].y : g.q[t + 1].x;
        w[t / 2] = __builtin_amdgcn_perm(b, a, (j & 1) ? kHi : kLo);
      }
      if constexpr (KB == 1) {
        const uint32_t a = (j >> 1) ? g.q[0].y : g.q[0].x;
        *reinterpret_cast<uint16_t*>(lds + lds_index<T>(mn + j, kb)) = static_cast<uint16_t>((j & 1) ? a >> 16 : a);
      } else if constexpr (KB == 2) {
        *reinterpret_cast<uint32_t*>(lds + lds_index<T>(mn + j, kb)) = w[0];
      } else {
        static_assert(KB == 4, "KB in {1, 2, 4}");
        *reinterpret_cast<uint2*>(lds + lds_index<T>(mn + j, kb)) = make_uint2(w[0], w[1]);
      }
    }
  }
  template <bool SPLIT>
  __device__ __forceinline__ void commit_edge(const Regs& g, T* lds) const { commit_f32<SPLIT>(g, lds, true); }
  template <bool SPLIT>
  __device__ __forceinline__ void commit(const Regs& g, T* lds) const {
    if constexpr (!V4) {
      commit_f32<SPLIT>(g, lds, true);
    } else if constexpr (sizeof(T) == 2) {
      if (cs == nullptr && rs == nullptr && !colsum) {
        commit_raw16(g, lds);
      } else {
        commit_f32<false>(g, lds, false);
      }
    } else {
      commit_f32<SPLIT>(g, lds, false);
    }
  }
};

// Column sums gathered by a `colsum` MNLoader: the 256 threads hold partial sums of
// 4 consecutive mn each (thread t: mn = 4 (t % ROWS/4)); they are combined in a fixed
// order through LDS and written as dst[mn] for mn < mn_valid.  Call after the main loop
// (which ends with a barrier), with every thread of the block.
template <typename T, int ROWS, bool V4>
__device__ __forceinline__ void reduce_colsum(const MNLoader<T, ROWS, V4>& ld, T* lds, T* __restrict__ dst) {
  constexpr int kQ = ROWS / 4;                  // mn quads
  constexpr int kGroups = kGemmThreads / kQ;    // threads per quad
  float* red = reinterpret_cast<float*>(lds);   // [kGroups][ROWS]
  const int q = threadIdx.x % kQ, grp = threadIdx.x / kQ;
#pragma unroll
  for (int j = 0; j < 4; ++j) red[grp * ROWS + 4 * q + j] = ld.csum[j];
  __syncthreads();
  if (threadIdx.x < ROWS && static_cast<int>(threadIdx.x) < ld.mn_valid) {
    float s = 0.f;
#pragma unroll 4
    for (int g2 = 0; g2 < kGroups; ++g2) s += red[g2 * ROWS + threadIdx.x];
    dst[threadIdx.x] = from_f32<T>(s);
  }
}

// Host check: loaders address a tile as a uniform base plus 32-bit per-lane byte offsets that
// span at most 256 rows of `stride` elements.
inline bool gemm_stride_ok(int64_t stride, size_t esz) {
  return stride >= 0 && (stride + 1) * 256 * static_cast<int64_t>(esz) < (int64_t{1} << 31);
}

// ---------------------------------------------------------------- XCD-aware block order
// MI355X has 8 XCDs (32 CUs and one L2 each); the hardware dispatches 1-D block b to
// XCD b % 8.  Kernels whose blocks fall into groups that read the same operand tile
// (e.g. the m-tiles of one band's weight chunk) number their blocks so that all
// `members` blocks of a group land on one XCD and are dispatched close together:
//   block b -> group (b / 8 / members) * 8 + b % 8, member (b / 8) % members.
// The grid is padded to whole groups of 8; padding blocks exit at once.
constexpr uint32_t kXcds = 8;

struct XcdGrid {
  uint32_t groups;
  uint32_t members;
  uint32_t blocks() const { return ((groups + kXcds - 1) / kXcds) * kXcds * members; }
};

__device__ __forceinline__ bool xcd_block(const XcdGrid& xg, uint32_t& group, uint32_t& member) {
  const uint32_t b = blockIdx.x;
  const uint32_t r = b / kXcds;
  member = r % xg.members;
  group = (r / xg.members) * kXcds + b % kXcds;
  return group < xg.groups;
}

template <int BR, int BC, int WR, int WC>
struct TileShape {
  static constexpr int kTR = BR / WR / 16;
  static constexpr int kTC = BC / WC / 16;
  static_assert(WR * WC == kGemmThreads / kWave, "4 waves per block");
  static_assert(kTR >= 1 && kTC >= 1 && BR % (WR * 16) == 0 && BC % (WC * 16) == 0, "bad tile");
};

// LDS elements the main loop needs for a BR x BC tile (two buffers; SPLIT: one split tile).
template <typename T, int BR, int BC, bool SPLIT = false>
constexpr int gemm_lds_elems() {
  return SPLIT ? (BR + BC) * kSplitRow : 2 * (BR + BC) * LdsPitch<T>::value;
}

// Register budget of the split kernels with 8 or fewer 16 x 16 tiles a wave, in waves per SIMD: their K
// steps wait on loads and barriers, which three blocks a CU cover better than two (224 against 228-324
// us for the mask backward's input gradient).
constexpr int kSplitWaves = 3;

// Multiply-adds of a launch from which an fp32 product takes the split.  Below them the fp32 MFMAs need
// less than 4 us for the products themselves; launches, loads and barriers are the time, and the split
// gains little or loses: the tiny model's mask MLP (130 rows, 64 -> 256, 0.27 G at most a launch) 148
// against 138 us, its band split 45.5 against 44.6, 32 bands of odd widths 128 against 131 and 64.2
// against 64.9.  What it would cost there is the sums' exact bits: a loss that takes absolute values (an
// L1 on spectra) turns the sign of one element of half a million, and so all gradients by 2e-3, when the
// estimate moves by 1e-7 of its size.  At 0.3 to 0.6 G (62 bands, 192 -> 768, 64 rows) 226 against 197 us.
constexpr int64_t kSplitMacs = 300'000'000;
inline bool split_macs(int64_t rows, int64_t in_features, int64_t out_features) {
  return rows * in_features >= (kSplitMacs + out_features - 1) / out_features;
}

// The K loop of a SPLIT kernel: one LDS tile, the next chunk's loads in registers while this one is
// multiplied (the blocks of a CU, two to six of them, cover each other's splits and barriers).  SPLIT:
// three bf16 planes and six products; else the fp32 MFMAs.
template <int BR, int BC, int WR, int WC, bool SPLIT, class LA, class LB>
__device__ __forceinline__ void gemm_f32_loop(LA& la, LB& lb, int K, float* lds,
                                              f32x4_t (&acc)[TileShape<BR, BC, WR, WC>::kTR]
                                                            [TileShape<BR, BC, WR, WC>::kTC]) {
  using S = TileShape<BR, BC, WR, WC>;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int r0 = (wave / WC) * (BR / WR);
  const int c0 = (wave % WC) * (BC / WC);
  const int nk = (K + kChunkK - 1) / kChunkK;
  const int kbeg = K - nk * kChunkK;  // chunk 0 may be partial
  float* lds_b = lds + BR * kSplitRow;
  la.prepare();
  lb.prepare();
  typename LA::Regs ra;
  typename LB::Regs rb;
  if (kbeg < 0) {
    la.fetch_edge(kbeg, ra);
    lb.fetch_edge(kbeg, rb);
    la.template commit_edge<SPLIT>(ra, lds);
    lb.template commit_edge<SPLIT>(rb, lds_b);
  } else {
    la.fetch(kbeg, ra);
    lb.fetch(kbeg, rb);
    la.template commit<SPLIT>(ra, lds);
    lb.template commit<SPLIT>(rb, lds_b);
  }
  // The matrix cores cut what a product adds below the accumulator's last place off one-sidedly, towards
  // minus infinity.  The products of the high parts, 16 bits long, hardly reach below it; those of the low
  // parts, 2^-8 and less of them, added to the same accumulator leave a mean error of -1.1e-8 of the
  // result's RMS at K = 192 and -1.0e-7 at K = 2048, where the fp32 MFMAs' is within 1e-9.  So the low
  // parts' products are summed apart: with 8 or fewer tiles a wave in accumulators of their own, added at
  // the end, and with more, for want of registers, from zero in each chunk, added by a rounded addition:
  // 7e-10 and 4e-10, and the error in the mean square from 1.9e-7 to 0.9e-7 and from 7.0e-7 to 3.1e-7, for
  // 4 % of the forward's time (62 groups of 192 -> 768, 1032 rows: 212 -> 221 us).
  constexpr bool kLow = SPLIT && S::kTR * S::kTC <= 8;
  f32x4_t low[kLow ? S::kTR : 1][kLow ? S::kTC : 1];
#pragma unroll
  for (int i = 0; i < (kLow ? S::kTR : 1); ++i)
#pragma unroll
    for (int j = 0; j < (kLow ? S::kTC : 1); ++j) low[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto mma = [&]() {
    if constexpr (SPLIT) {
      constexpr int kP[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};  // small parts first
      auto term = [&](int i, int j, int q, const bf16x8_t (&a)[3], const bf16x8_t (&b)[3], f32x4_t& chunk) {
        f32x4_t& d = q == 5 ? acc[i][j] : kLow ? low[kLow ? i : 0][kLow ? j : 0] : chunk;
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kP[q][0]], b[kP[q][1]], d, 0, 0, 0);
      };
      auto add_chunk = [&](int i, int j, const f32x4_t& chunk) {
        if constexpr (!kLow) {
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][r] += chunk[r];
        }
      };
      auto frag = [&](auto tr, const float* tile, auto rows, int r, int t, bf16x8_t (&f)[3]) {
        constexpr int ROWS = decltype(rows)::value;
        const char* base = reinterpret_cast<const char*>(tile);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          if constexpr (decltype(tr)::value)
            f[p] = __builtin_bit_cast(
                bf16x8_t, tr_frag(base + p * ROWS * 64 + frag_mn_addr_p<2 * ROWS>(0, r + 16 * t, lane), 4 * 2 * ROWS));
          else
            f[p] = *reinterpret_cast<const bf16x8_t*>(base + p * ROWS * 64 +
                                                      split_offset(r + 16 * t + (lane & 15), 8 * (lane >> 4)));
        }
      };
      using RowsA = std::integral_constant<int, BR>;
      using RowsB = std::integral_constant<int, BC>;
      using TrA = std::integral_constant<bool, LA::kTransposed>;
      using TrB = std::integral_constant<bool, LB::kTransposed>;
      // The operand with fewer tiles stays in registers, the other's tiles pass by, with 4 x 4 tiles twice, once
      // for each half of the first: all of its parts beside the chunk sums spill, and so do the sums of
      // several passing tiles, which the scheduling barrier keeps apart.
      if constexpr (S::kTR <= S::kTC) {
        constexpr int kHold = !kLow && S::kTR == 4 ? 2 : S::kTR;
#pragma unroll
        for (int h = 0; h < S::kTR; h += kHold) {
          bf16x8_t a[kHold][3];
#pragma unroll
          for (int i = 0; i < kHold; ++i) frag(TrA{}, lds, RowsA{}, r0, h + i, a[i]);
#pragma unroll
          for (int j = 0; j < S::kTC; ++j) {
            bf16x8_t b[3];
            frag(TrB{}, lds_b, RowsB{}, c0, j, b);
            f32x4_t chunk[kHold] = {};
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
              for (int i = 0; i < kHold; ++i) term(h + i, j, q, a[i], b, chunk[i]);
#pragma unroll
            for (int i = 0; i < kHold; ++i) add_chunk(h + i, j, chunk[i]);
            if constexpr (!kLow) __builtin_amdgcn_sched_barrier(0);
          }
        }
      } else {
        bf16x8_t b[S::kTC][3];
#pragma unroll
        for (int j = 0; j < S::kTC; ++j) frag(TrB{}, lds_b, RowsB{}, c0, j, b[j]);
#pragma unroll
        for (int i = 0; i < S::kTR; ++i) {
          bf16x8_t a[3];
          frag(TrA{}, lds, RowsA{}, r0, i, a);
          f32x4_t chunk[S::kTC] = {};
#pragma unroll
          for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int j = 0; j < S::kTC; ++j) term(i, j, q, a, b[j], chunk[j]);
#pragma unroll
          for (int j = 0; j < S::kTC; ++j) add_chunk(i, j, chunk[j]);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < S::kTR; ++i)
#pragma unroll
        for (int j = 0; j < S::kTC; ++j)
          acc[i][j] = mfma_tile<float>(lds, r0 + i * 16 + (lane & 15), lds_b, c0 + j * 16 + (lane & 15), acc[i][j],
                                       lane);
    }
  };
  for (int kc = 0;;) {
    __syncthreads();
    const bool more = ++kc < nk;
    if (more) {
      la.fetch(kbeg + kc * kChunkK, ra);
      lb.fetch(kbeg + kc * kChunkK, rb);
    }
    mma();
    __syncthreads();
    if (!more) break;
    la.template commit<SPLIT>(ra, lds);
    lb.template commit<SPLIT>(rb, lds_b);
  }
  if constexpr (kLow) {
#pragma unroll
    for (int i = 0; i < S::kTR; ++i)
#pragma unroll
      for (int j = 0; j < S::kTC; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] += low[i][j][r];
  }
}

// Runs the K loop; `acc` is accumulated (callers zero it).
//
// DEPTH = 1: chunk c + 1 is fetched into registers while chunk c is multiplied and
// committed to the other LDS buffer afterwards.  DEPTH = 2: chunk c is fetched into
// register set R[c % 2] two iterations ahead, so two chunks of global loads are in
// flight during the MFMAs of a third, at the cost of a second register set (the
// loop is unrolled by two so the sets stay fixed registers).  Buffer offsets are
// computed from the __shared__ base (no pointer tables), so every LDS access stays
// a ds_* instruction and waits only on the LDS counter.
//
// SPLIT (fp32): gemm_f32_loop on the three bf16 planes, and again on the fp32 MFMAs if a sum is not finite
// or a number too small for an exact split was among the operands.
template <typename T, int BR, int BC, int WR, int WC, int DEPTH = 1, bool SPLIT = false, class LA, class LB>
__device__ __forceinline__ void gemm_mainloop(LA& la, LB& lb, int K, T* lds,
                                              f32x4_t (&acc)[TileShape<BR, BC, WR, WC>::kTR]
                                                            [TileShape<BR, BC, WR, WC>::kTC]) {
  static_assert(DEPTH == 1 || DEPTH == 2, "prefetch depth 1 or 2");
  static_assert(!SPLIT || sizeof(T) == 4, "fp32 only");
  using S = TileShape<BR, BC, WR, WC>;
  if constexpr (SPLIT) {
    if (K <= 0) return;
    const LA la0 = la;  // the loaders' row and column sums start again with a re-run
    const LB lb0 = lb;
    gemm_f32_loop<BR, BC, WR, WC, true>(la, lb, K, lds, acc);
    bool good = (la.least < lb.least ? la.least : lb.least) >= kSplitLeast;
#pragma unroll
    for (int i = 0; i < S::kTR; ++i)
#pragma unroll
      for (int j = 0; j < S::kTC; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) good = good && fabsf(acc[i][j][r]) <= 3.402823466e38f;
    if (__syncthreads_or(!good)) {
      la = la0;
      lb = lb0;
      la.forget();
      lb.forget();
#pragma unroll
      for (int i = 0; i < S::kTR; ++i)
#pragma unroll
        for (int j = 0; j < S::kTC; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      gemm_f32_loop<BR, BC, WR, WC, false>(la, lb, K, lds, acc);
    }
    return;
  } else {
  constexpr int P = LdsPitch<T>::value;
  constexpr int kBuf = (BR + BC) * P;  // elements of one (A, B) buffer pair
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int r0 = (wave / WC) * (BR / WR);
  const int c0 = (wave % WC) * (BC / WC);
  const int nk = (K + kChunkK - 1) / kChunkK;
  if (nk == 0) return;

  // The scheduler would otherwise hoist the LDS commit of the next chunk (independent
  // addresses) above the MFMAs, making them wait for the in-flight loads it commits.
  auto mma = [&](int cur) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < S::kTR; ++i) {
#pragma unroll
      for (int j = 0; j < S::kTC; ++j) {
        acc[i][j] = mfma_tile<T>(lds + cur, r0 + i * 16 + (lane & 15), lds + cur + BR * P, c0 + j * 16 + (lane & 15),
                                 acc[i][j], lane);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // chunk c covers k in [kbeg + 32 c, kbeg + 32 c + 32); only chunk 0 can be partial
  const int kbeg = K - nk * kChunkK;
  const bool edge0 = kbeg < 0;
  la.prepare();
  lb.prepare();
  typename LA::Regs ra0;
  typename LB::Regs rb0;
  if (edge0) {
    la.fetch_edge(kbeg, ra0);
    lb.fetch_edge(kbeg, rb0);
  } else {
    la.fetch(kbeg, ra0);
    lb.fetch(kbeg, rb0);
  }
  auto commit0 = [&]() {
    if (edge0) {
      la.template commit_edge<false>(ra0, lds);
      lb.template commit_edge<false>(rb0, lds + BR * P);
    } else {
      la.template commit<false>(ra0, lds);
      lb.template commit<false>(rb0, lds + BR * P);
    }
  };
  // The steady-state loops below fetch unconditionally: with every trip issuing the
  // same loads into the same registers, the wait-count analysis can see that a
  // register set's previous loads retired before it is refilled, and no conditional
  // path splits the accumulators' live ranges.
  if constexpr (DEPTH == 1) {
    commit0();
    __syncthreads();
    int kc = 0;
    for (; kc + 1 < nk; ++kc) {
      const int cur = (kc & 1) * kBuf;
      la.fetch(kbeg + (kc + 1) * kChunkK, ra0);
      lb.fetch(kbeg + (kc + 1) * kChunkK, rb0);
      mma(cur);
      la.template commit<false>(ra0, lds + kBuf - cur);
      lb.template commit<false>(rb0, lds + kBuf - cur + BR * P);
      __syncthreads();
    }
    mma((kc & 1) * kBuf);
    __syncthreads();
  } else {
    typename LA::Regs ra1;
    typename LB::Regs rb1;
    if (nk > 1) {
      la.fetch(kbeg + kChunkK, ra1);
      lb.fetch(kbeg + kChunkK, rb1);
    }
    commit0();
    __syncthreads();
    // Entering each trip: chunk kc is in LDS buffer (kc & 1) and its registers (set 0)
    // are free; chunk kc + 1 is in flight into set 1.
    int kc = 0;
    for (; kc + 3 < nk; kc += 2) {
      const int cur = (kc & 1) * kBuf;
      la.fetch(kbeg + (kc + 2) * kChunkK, ra0);
      lb.fetch(kbeg + (kc + 2) * kChunkK, rb0);
      mma(cur);
      la.template commit<false>(ra1, lds + kBuf - cur);
      lb.template commit<false>(rb1, lds + kBuf - cur + BR * P);
      __syncthreads();
      la.fetch(kbeg + (kc + 3) * kChunkK, ra1);
      lb.fetch(kbeg + (kc + 3) * kChunkK, rb1);
      mma(kBuf - cur);
      la.template commit<false>(ra0, lds + cur);
      lb.template commit<false>(rb0, lds + cur + BR * P);
      __syncthreads();
    }
    // 1 to 3 chunks left: kc (in LDS), kc + 1 (set 1, in flight), kc + 2 (not fetched)
    const int cur = (kc & 1) * kBuf;
    if (kc + 2 < nk) {
      la.fetch(kbeg + (kc + 2) * kChunkK, ra0);
      lb.fetch(kbeg + (kc + 2) * kChunkK, rb0);
      mma(cur);
      la.template commit<false>(ra1, lds + kBuf - cur);
      lb.template commit<false>(rb1, lds + kBuf - cur + BR * P);
      __syncthreads();
      mma(kBuf - cur);
      la.template commit<false>(ra0, lds + cur);
      lb.template commit<false>(rb0, lds + cur + BR * P);
      __syncthreads();
      mma(cur);
    } else if (kc + 1 < nk) {
      mma(cur);
      la.template commit<false>(ra1, lds + kBuf - cur);
      lb.template commit<false>(rb1, lds + kBuf - cur + BR * P);
      __syncthreads();
      mma(kBuf - cur);
    } else {
      mma(cur);
    }
    __syncthreads();
  }
  }
}

}  // namespace pmsst
