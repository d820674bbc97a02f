// The grouped linear's products at wide layers, 16-bit storage, fp32 accumulation:
//   h[m, g, :]   = tanh(x[m, g, :] W_g^T + bias_g)   (K = in_features; rounded before the tanh)
//   dx[m, g, :]  = dy[m, g, :] W_g            (K = out_features)
//   dW[g][o][i]  = sum_m dy[m, g, o] x[m, g, i], db[g][o] = sum_m dy[m, g, o]   (K = rows)
// dy[M, G, O], x and dx[M, G, I], W and dW[G, O, I] row-major.
//
// Backward block = 8 waves on a tile of AR x BR results: A rows run along the result's contiguous axis (a
// lane's 4 accumulators are 4 neighbours of it), B rows along its rows.  Wave (wa, wb) owns
// 16 TA x 16 TB of it.  32-wide K chunks of both operands move by global -> LDS DMA into a ring of
// kGgStages stages; K-contiguous operands (dy in dx) as 64-byte rows, the others (W in dx, both in
// dW) as K-rows of the tile's width, read transposed (ds_read_b64_tr_b16).  Forward block = 4 waves on a
// tile half as high with a ring of 3 stages, two blocks per CU: its K loop is short (2 to 16 chunks) and
// one block's loads and tanh epilogue run beside the other's products.
//
// What bounds it: the matrix cores want 32 MFMAs of 16 cycles per wave and chunk on a 256 x 256 tile,
// two waves to a SIMD, i.e. 1024 cycles a chunk, in which the block's fragment reads take 768 LDS
// cycles and its DMAs 32 KB of L2.  So the tile is as large as the registers allow (128 accumulators
// a lane), and a chunk's fragments are read while the previous chunk's are multiplied (two register
// sets), which keeps LDS and matrix cores busy together.  62 groups of 512 -> 2048 at 1896 rows: dx
// 262 us, 930 TFLOP/s (the register-staged kernel 731 us), dW 276 us, 890 TFLOP/s (me_bwd_dw_dma_kernel,
// 64 x 128 tiles, 396 us); a library bf16 product of 8192^3 reaches 1290 on the same card.
#include "common.h"
#include "dma_gemm.h"
#include "grouped_dx.h"
#include "ring.h"

namespace pmsst {
namespace {

enum GgOp { kGgDx, kGgDw, kGgFwd };

struct GgArgs {
  const void* a;   // dx, fwd: W; dw: x
  const void* b;   // dx, dw: dy; fwd: x
  void* d;         // dx, dW or h
  void* db;        // dw: bias gradient or null; fwd: bias
  int64_t M;
  int G, O, I;
};

// One 16-byte-per-lane global -> LDS DMA from a uniform base plus a 32-bit byte offset per lane (see
// dma16_m0 for what the compiler sees of it).
__device__ __forceinline__ void dma16_base(const char* base, uint32_t off, uint32_t lds) {
  uint32_t save;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(save)
      : "v"(off), "s"(base), "s"(lds)
      : "memory");
}

constexpr int gg_waves(GgOp op) { return op == kGgFwd ? 4 : 8; }

template <typename T, GgOp OP, int TA, int WA>
__global__ __launch_bounds__(gg_waves(OP) * 64) __attribute__((amdgpu_waves_per_eu(2))) void gg_kernel(GgArgs a,
                                                                                                      BandSched sc) {
  constexpr int NW = gg_waves(OP), S = NW == 8 ? 4 : 3;
  constexpr int WB = NW / WA, TB = 4;
  constexpr int AR = 16 * TA * WA, BR = 16 * TB * WB;
  constexpr bool A_KC = OP == kGgFwd, B_KC = OP != kGgDw;  // K-contiguous operands
  constexpr int kABytes = AR * 64, kStage = kABytes + BR * 64;
  constexpr int kPA = kABytes / 1024, kPT = kStage / 1024;  // 1 KB DMA pieces: A's, then B's
  constexpr int PW = (kPT + NW - 1) / NW;            // per wave; a wave with fewer repeats its first
  constexpr int kOP = AR + 8;                        // row pitch (elements) of the staged result
  constexpr int kLds = S * kStage > BR * kOP * 2 ? S * kStage : BR * kOP * 2;
  static_assert(AR % 64 == 0 && kLds <= 160 * 1024, "tile");
  __shared__ __attribute__((aligned(1024))) char lds[kLds];

  int g;
  uint32_t tb, ta, per;  // B tile, A tile
  if (!sched_block(sc, g, tb, ta, per)) return;
  const int lane = threadIdx.x & 63, gq = lane >> 4, rr = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int wa = wave % WA, wb = wave / WA;
  const int64_t dyrow = static_cast<int64_t>(a.G) * a.O, xrow = static_cast<int64_t>(a.G) * a.I;
  const int K = OP == kGgDx ? a.O : OP == kGgDw ? static_cast<int>(a.M) : a.I;
  const int nk = (K + 31) / 32;
  const int kbeg = K - 32 * nk;  // dw: chunks end at M, so only chunk 0 has K rows to leave out
  const int a0 = static_cast<int>(ta) * AR;
  const int64_t b0 = static_cast<int64_t>(tb) * BR;
  const int aleft = (OP == kGgFwd ? a.O : a.I) - a0;
  const int avalid = aleft < AR ? aleft : AR;
  const int64_t bleft = (OP == kGgDw ? a.O : a.M) - b0;
  const int bvalid = bleft < BR ? static_cast<int>(bleft) : BR;

  // ---- DMA plan: piece k of a stage (k = wave + NW q).  MN operand: flattened 16-byte units
  // 64 k + lane of its 32 K-rows; K-contiguous: rows 16 k + lane / 4.  Columns and rows past the tile's
  // valid part repeat its last (their products are not stored).
  const int64_t astride = OP == kGgDw ? xrow : a.I;     // elements between A's K-rows (fwd: rows)
  const int64_t bstride = OP == kGgFwd ? xrow : dyrow;  // elements between B's rows (dw: K-rows)
  const int64_t wg = static_cast<int64_t>(g) * a.O * a.I;
  const char* abase = static_cast<const char*>(a.a) + 2 * (OP == kGgDx   ? wg + a0
                                                           : OP == kGgDw ? static_cast<int64_t>(g) * a.I + a0
                                                                         : wg + static_cast<int64_t>(a0) * a.I);
  const char* bbase = static_cast<const char*>(a.b) + 2 * (static_cast<int64_t>(g) * (OP == kGgFwd ? a.I : a.O) +
                                                           (OP == kGgDw ? b0 : b0 * bstride));
  if (OP == kGgDw) {
    abase += 2 * kbeg * astride;
    bbase += 2 * kbeg * bstride;
  }
  const int64_t astep = A_KC ? 64 : 64 * astride, bstep = B_KC ? 64 : 64 * bstride;  // bytes per chunk
  uint32_t off[PW], ldst[PW];
  bool isa[PW];
  [[maybe_unused]] int krow[PW];  // K-row of this lane's unit
#pragma unroll
  for (int q = 0; q < PW; ++q) {
    int k = wave + NW * q;
    k = k < kPT ? k : wave;
    isa[q] = k < kPA;
    ldst[q] = static_cast<uint32_t>(k * 1024);
    const int64_t stride = isa[q] ? astride : bstride;
    const int valid = isa[q] ? avalid : bvalid;
    if (!(isa[q] ? A_KC : B_KC)) {
      const int units = isa[q] ? AR / 8 : BR / 8;
      const int U = 64 * (isa[q] ? k : k - kPA) + lane;
      const int kr = U / units;
      const int u = (U % units) ^ (isa[q] ? swz_mn_p<2 * AR>(kr) : swz_mn_p<2 * BR>(kr));
      const int col = 8 * u < valid ? 8 * u : valid - 8;
      krow[q] = kr;
      off[q] = static_cast<uint32_t>((kr * stride + col) * 2);
    } else {
      const int r = 16 * (isa[q] ? k : k - kPA) + (lane >> 2);
      const int rc = r < valid ? r : valid - 1;
      krow[q] = 0;
      off[q] = static_cast<uint32_t>((rc * stride + 8 * ((lane & 3) ^ swz_k(lane >> 2))) * 2);
    }
  }
  const uint32_t lds0 = lds_addr(lds);
  auto dma = [&](int c) {
    const uint32_t st = lds0 + static_cast<uint32_t>((c % S) * kStage);
    const char* ab = abase + c * astep;
    const char* bb = bbase + c * bstep;
#pragma unroll
    for (int q = 0; q < PW; ++q)
      dma16_base(isa[q] ? ab : bb, off[q], __builtin_amdgcn_readfirstlane(st + ldst[q]));
  };
  // chunk 0: K rows before row 0 are read from row 0
  {
#pragma unroll
    for (int q = 0; q < PW; ++q) {
      uint32_t o = off[q];
      if (OP == kGgDw && kbeg + krow[q] < 0)
        o += static_cast<uint32_t>(-(kbeg + krow[q])) * static_cast<uint32_t>((isa[q] ? astride : bstride) * 2);
      dma16_base(isa[q] ? abase : bbase, o, __builtin_amdgcn_readfirstlane(lds0 + ldst[q]));
    }
  }
#pragma unroll
  for (int c = 1; c < S - 1; ++c)
    if (c < nk) dma(c);

  f32x4_t acc[TA][TB];
#pragma unroll
  for (int i = 0; i < TA; ++i)
#pragma unroll
    for (int j = 0; j < TB; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if constexpr (OP == kGgFwd) {  // the sums start at the bias, as the one-pass MLP's do
    const T* bias = static_cast<const T*>(a.db) + static_cast<int64_t>(g) * a.O + a0;
#pragma unroll
    for (int i = 0; i < TA; ++i) {
      const int o = 16 * (TA * wa + i) + 4 * gq;
      float v[4];
      load_pack<T, 4>(bias + (o < avalid ? o : avalid - 4), v);
#pragma unroll
      for (int j = 0; j < TB; ++j) acc[i][j] = f32x4_t{v[0], v[1], v[2], v[3]};
    }
  }
  // column sums of B (db): lane's 8 K values of column 16 j + rr, summed per chunk
  const bool do_bias = OP == kGgDw && a.db != nullptr && ta == 0 && wa == 0;
  [[maybe_unused]] float csum[TB];
#pragma unroll
  for (int j = 0; j < TB; ++j) csum[j] = 0.f;

  // ---- fragment offsets inside a stage
  uint32_t aoff[TA], boff[TB];
#pragma unroll
  for (int i = 0; i < TA; ++i)
    aoff[i] = A_KC ? frag_k_addr(0, 16 * (TA * wa + i), lane) : frag_mn_addr_p<2 * AR>(0, 16 * (TA * wa + i), lane);
#pragma unroll
  for (int j = 0; j < TB; ++j)
    boff[j] = B_KC ? frag_k_addr(kABytes, 16 * (TB * wb + j), lane)
                   : frag_mn_addr_p<2 * BR>(kABytes, 16 * (TB * wb + j), lane);
  auto read = [&](int c, u32x4_t (&fa)[TA], u32x4_t (&fb)[TB]) {
    const char* st = lds + (c % S) * kStage;
#pragma unroll
    for (int j = 0; j < TB; ++j) {
      if constexpr (B_KC) fb[j] = *reinterpret_cast<const u32x4_t*>(st + boff[j]);
      else fb[j] = tr_frag(st + boff[j], 4 * 2 * BR);
    }
#pragma unroll
    for (int i = 0; i < TA; ++i) {
      if constexpr (A_KC) fa[i] = *reinterpret_cast<const u32x4_t*>(st + aoff[i]);
      else fa[i] = tr_frag(st + aoff[i], 4 * 2 * AR);
    }
  };
  auto mma = [&](const u32x4_t (&fa)[TA], const u32x4_t (&fb)[TB]) {
#pragma unroll
    for (int i = 0; i < TA; ++i)
#pragma unroll
      for (int j = 0; j < TB; ++j) acc[i][j] = mfma_raw<T>(fa[i], fb[j], acc[i][j]);
    if constexpr (OP == kGgDw) {
      if (do_bias) {
        typedef T v8 __attribute__((ext_vector_type(8)));
#pragma unroll
        for (int j = 0; j < TB; ++j) {
          const v8 e = __builtin_bit_cast(v8, fb[j]);
          float s[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) s[r] = to_f32(e[2 * r]) + to_f32(e[2 * r + 1]);
          csum[j] += (s[0] + s[1]) + (s[2] + s[3]);
        }
      }
    }
  };
  // The turn between chunk c and c + 1: chunk c + 1 has landed for every wave and every wave's reads of
  // chunk c are done, so its stage takes chunk c + S; `after` chunks issued behind c + 1 may still be
  // in flight.  The LDS wait is the builtin, so that the compiler knows chunk c's fragments are in
  // their registers and puts no wait of its own (which would cover the reads of chunk c + 1, issued
  // first) before their MFMAs.
  auto lds_done_barrier = [&]() {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto wait_chunks = [&](int after) {
    if (S == 4 && after >= 2) vm_wait<2 * PW>();
    else if (after >= 1) vm_wait<PW>();
    else vm_wait<0>();
  };
  static_assert(S == 3 || S == 4, "wait_chunks");
  // a chunk's fragment reads spread between the MFMAs of the chunk before it
  constexpr int kReads = (A_KC ? 1 : 2) * TA + (B_KC ? 1 : 2) * TB, kMma = TA * TB;
  auto interleave = [&]() {
    constexpr int kPer = kMma / (kReads / 2);
#pragma unroll
    for (int i = 0; i < kReads / 2; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, kPer, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kMma - kPer * (kReads / 2), 0);
  };

  u32x4_t fa0[TA], fb0[TB], fa1[TA], fb1[TB];
  wait_chunks(nk - 1 < S - 2 ? nk - 1 : S - 2);
  if (OP == kGgDw && kbeg < 0) {  // chunk 0: this wave's own units of K rows before row 0
#pragma unroll
    for (int q = 0; q < PW; ++q)
      if (kbeg + krow[q] < 0) *reinterpret_cast<u32x4_t*>(lds + ldst[q] + lane * 16) = u32x4_t{0u, 0u, 0u, 0u};
  }
  lds_done_barrier();
  if (S - 1 < nk) dma(S - 1);
  read(0, fa0, fb0);
  int c = 0;
  for (; c + 1 + S < nk; c += 2) {  // both turns have their chunk to move: no branch inside
    vm_wait<(S - 2) * PW>();
    lds_done_barrier();
    dma(c + S);
    read(c + 1, fa1, fb1);
    mma(fa0, fb0);
    interleave();
    vm_wait<(S - 2) * PW>();
    lds_done_barrier();
    dma(c + 1 + S);
    read(c + 2, fa0, fb0);
    mma(fa1, fb1);
    interleave();
  }
  auto turn = [&](int k) {
    wait_chunks(nk - 2 - k < S - 2 ? nk - 2 - k : S - 2);
    lds_done_barrier();
    if (k + S < nk) dma(k + S);
  };
  for (; c < nk; c += 2) {
    if (c + 1 < nk) {
      turn(c);
      read(c + 1, fa1, fb1);
    }
    mma(fa0, fb0);
    if (c + 1 < nk) {
      if (c + 2 < nk) {
        turn(c + 1);
        read(c + 2, fa0, fb0);
      }
      mma(fa1, fb1);
    }
  }

  if (OP == kGgDw && do_bias) {
    T* db = static_cast<T*>(a.db) + static_cast<int64_t>(g) * a.O + b0;
#pragma unroll
    for (int j = 0; j < TB; ++j) {
      float v = csum[j];
      v += __shfl_xor(v, 16, kWave);
      v += __shfl_xor(v, 32, kWave);
      const int o = 16 * (TB * wb + j) + rr;
      if (lane < 16 && o < bvalid) db[o] = from_f32<T>(v);
    }
  }

  // ---- epilogue through LDS: [BR rows][AR], written out as whole rows
  __syncthreads();  // every wave is done with the ring (its last wait was vmcnt(0))
  T* ot = reinterpret_cast<T*>(lds);
#pragma unroll
  for (int j = 0; j < TB; ++j) {
    const int r = 16 * (TB * wb + j) + rr;
#pragma unroll
    for (int i = 0; i < TA; ++i) {
      float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
      if constexpr (OP == kGgFwd) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = tanh16<T>(to_f32(from_f32<T>(v[e])));
      }
      store_pack<T, 4>(ot + r * kOP + 16 * (TA * wa + i) + 4 * gq, v);
    }
  }
  __syncthreads();
  constexpr int kUnits = AR / 8;
  const int64_t drow = OP == kGgDx ? xrow : OP == kGgDw ? a.I : dyrow;
  const int64_t d0 = OP == kGgDx   ? static_cast<int64_t>(g) * a.I
                     : OP == kGgDw ? static_cast<int64_t>(g) * a.O * a.I
                                   : static_cast<int64_t>(g) * a.O;
  T* d = static_cast<T*>(a.d) + d0 + b0 * drow + a0;
  const int nu = avalid / 8;  // whole units
#pragma unroll
  for (int p = 0; p < BR * kUnits / (64 * NW); ++p) {
    const int q = static_cast<int>(threadIdx.x) + 64 * NW * p;
    const int r = q / kUnits, u = q % kUnits;
    if (r < bvalid && u < nu)
      *reinterpret_cast<u32x4_t*>(d + r * drow + 8 * u) = *reinterpret_cast<const u32x4_t*>(ot + r * kOP + 8 * u);
  }
}

template <typename T, GgOp OP, int TA, int WA>
int launch(const GgArgs& a, hipStream_t stream) {
  BandSched sc;
  uint32_t per_xcd = 0;
  constexpr int AR = 16 * TA * WA;
  constexpr int BR = 16 * 4 * gg_waves(OP) / WA;
  const int64_t a_tiles = ((OP == kGgFwd ? a.O : a.I) + AR - 1) / AR;  // tiles of AR along the A rows
  const int64_t b_rows = OP == kGgDw ? a.O : a.M;
  if (!build_even_sched(a.G, (b_rows + BR - 1) / BR, [&](int) { return a_tiles; }, &sc, &per_xcd))
    return fail(PMSST_EINVAL, "grouped linear: too many groups or rows for the block schedule");
  hipLaunchKernelGGL((gg_kernel<T, OP, TA, WA>), dim3(per_xcd * kXcds), dim3(64 * gg_waves(OP)), 0, stream, a, sc);
  return check_launch("gg_kernel");
}

template <typename T, GgOp OP>
int launch_op(const GgArgs& a, hipStream_t stream) {
  if ((OP == kGgFwd ? a.O : a.I) % 256 == 0) return launch<T, OP, 8, 2>(a, stream);
  return launch<T, OP, 6, 2>(a, stream);
}

bool shape_ok(int64_t groups, int64_t in_features, int64_t out_features, int64_t rows, size_t elem) {
  // 32-bit byte offsets: 256 rows of dy, 32 K-rows of x
  return elem == 2 && rows > 0 && groups <= kSchedMaxBands && in_features % 8 == 0 && out_features % 8 == 0 &&
         256 * groups * out_features * 2 < (int64_t{1} << 31) && 256 * groups * in_features * 2 < (int64_t{1} << 31) &&
         groups * in_features < (int64_t{1} << 31) && groups * out_features < (int64_t{1} << 31);
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

bool wide_dx_supported(int64_t groups, int64_t in_features, int64_t out_features, int64_t rows, size_t elem,
                       const void* dy, const void* w, const void* dx) {
  if (!shape_ok(groups, in_features, out_features, rows, elem) || out_features % 32 != 0 || !aligned16(dy) ||
      !aligned16(w) || !aligned16(dx))
    return false;
  // Above 256, where glin_dx_kernel ends, the register-staged kernel with its 64 x 64 results a block is the
  // alternative: it wins while it has fewer than 2.75 blocks' worth of results a CU, with few groups 4 (its
  // blocks then walk a long K side by side where this kernel's tiles leave CUs idle).  62 groups of 512 ->
  // 1024: 64 rows (1.9) 23.5 us against 26.4, 96 rows (2.9) 29 against 27, 130 rows 39 against 26; 384 ->
  // 768: 80 rows (1.8) 18.9 against 19.3, 128 rows (2.9) 21.6 against 19.6; 30 groups of 512 -> 2048: 130
  // rows (1.9) 38 against 43, 200 rows (2.9) 46 against 44; 16 of 768 -> 1536: 320 rows (3.75) 35.7 against
  // 36.5, 600 rows (7) 69 against 39; 8 of 512 -> 2048: 600 rows (2.3) 38 against 45, 1032 rows (4) 58 against
  // 47; one of 2048 -> 2048: 1500 rows (2.9) 40 against 45, 2760 rows (5.4) 68 against 47.
  if (in_features > 256) {
    const int64_t quarters = groups >= 24 ? 11 : 16;
    return groups * rows * in_features >= quarters * 1024 * num_cus();
  }
  // At 192 and 256 glin_dx_kernel's smaller blocks (two per CU) win unless whole rounds of one 256-row
  // block per CU are at least 80 % full: M = 1032, 62 groups of 192 -> 768: 310 blocks, 61 % of two
  // rounds, 53 us against 43; M = 2760, 60 groups: 660 blocks, 86 % of three, 89 us against 96.
  const int64_t blocks = groups * ((rows + 255) / 256), cus = num_cus(), rounds = (blocks + cus - 1) / cus;
  return (in_features == 192 || in_features == 256) && 5 * blocks >= 4 * rounds * cus;
}

template <typename T>
int launch_wide_dx(const void* dy, const void* w, void* dx, int64_t groups, int64_t in_features, int64_t out_features,
                   int64_t rows, hipStream_t stream) {
  return launch_op<T, kGgDx>(GgArgs{w, dy, dx, nullptr, rows, static_cast<int>(groups), static_cast<int>(out_features),
                                    static_cast<int>(in_features)}, stream);
}

bool wide_dw_supported(int64_t groups, int64_t in_features, int64_t out_features, int64_t rows, size_t elem,
                       const void* dy, const void* x, const void* dw) {
  if (!shape_ok(groups, in_features, out_features, rows, elem) || in_features < 192 || rows < 32 || !aligned16(dy) ||
      !aligned16(x) || !aligned16(dw))
    return false;  // below 192 inputs columns of the tile stay empty
  // Against the kernel that would run otherwise: how many rounds of its blocks, on the CUs it can use, stand
  // against a round of this kernel's (one block per CU).  me_bwd_dw_dma_kernel (in_features in whole 64s; 64
  // x 128 tiles) runs a group's blocks on one XCD; a round takes 18 us at 2760 rows, one of these tiles 92
  // (256 inputs wide) or 73 (192).  Rounds against one, and the two times in us:
  //   192 wide: 4.5 (62 groups of 192 -> 768): 320 rows 15.3, 15.9; 1032 rows 33.7, 32.7; 1400 rows 45.2, 41.8;
  //     2760 rows 92, 77.  4.5 (62 of 384 -> 768): 1032 rows 60.8, 63.7; 1400 rows 80, 81; 1896 rows 109, 106.
  //     6 (62 of 384 -> 1536): 128 rows 27.3, 29.5; 200 rows 36.8, 35.1; 1032 rows 120, 102.
  //     3.1 (62 of 320 -> 640): 2760 rows 126, 144.
  //   256 wide: 6 (62 of 256 -> 768): 64 rows 11.4, 10.7; 1032 rows 49, 38.  8 (62 of 512 -> 2048): 64 rows
  //     38.7, 38.8; 1032 rows 225, 159.  4 (62 of 256 -> 512): 1032 rows 30.5, 37.2; 2760 rows 83, 84.  4.5
  //     (16 of 768 -> 1536): 2760 rows 141, 145.  16 (one of 2048 -> 2048): 64 rows 18, 9.
  const int64_t a_cols = in_features % 256 == 0 ? 256 : 192, cus = num_cus();
  const auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int64_t rounds = cdiv(groups * cdiv(out_features, 256) * cdiv(in_features, a_cols), cus);
  if (in_features % 64 == 0) {
    const int64_t other = cdiv(groups, kXcds) * (in_features / 64) * cdiv(out_features, 128) * kXcds;  // blocks
    if (a_cols == 256) return other >= 6 * rounds * cus && rows >= 64;
    return (other >= 6 * rounds * cus && rows > 128) || (2 * other >= 9 * rounds * cus && rows >= 1400);
  }
  // Else the register-staged kernel, 64 x 64 tiles spread evenly: 6.8 (62 groups of 200 -> 400): 130 rows 12.6,
  // 12.3, 320 rows 18.9, 15.4; 6.3 (62 of 200 -> 800): 200 rows 21.4, 22.8, 320 rows 28, 27; 5.5 (62 of 264 ->
  // 528): 320 rows 24.6, 26.7, 600 rows 41.6, 39.4; 9.3 (62 of 520 -> 1040): 130 rows 38.7, 35.8; 1.6 (8 of
  // 200 -> 800): 2760 rows 51, 64.
  const int64_t other = groups * cdiv(in_features, 64) * cdiv(out_features, 64);
  return other >= 5 * rounds * cus && rows * other >= 2000 * rounds * cus;
}

template <typename T>
int launch_wide_dw(const void* dy, const void* x, void* dw, void* db, int64_t groups, int64_t in_features,
                   int64_t out_features, int64_t rows, hipStream_t stream) {
  return launch_op<T, kGgDw>(GgArgs{x, dy, dw, db, rows, static_cast<int>(groups), static_cast<int>(out_features),
                                    static_cast<int>(in_features)}, stream);
}

bool wide_tanh_supported(int64_t groups, int64_t in_features, int64_t out_features, int64_t rows, size_t elem,
                         const void* x, const void* w, const void* bias, const void* out) {
  // From 128 outputs: the tile is 192 or 256 wide.  64 outputs leave two thirds of it empty (62 groups of
  // 192 -> 64: 31 rows 6.4 us against 9.2, 1896 rows 20 against 24; 64 -> 64: 15 against 19); at 128 the
  // register-staged kernel takes 7.8 us at 31 rows and 28 at 1896 (62 groups of 64 -> 128), this one 7.7 and
  // 20, and it stays ahead from one row and one group on (one group of 512 -> 2048, one row: 20 and 13 us;
  // 62 groups of 192 -> 768, 31 rows: 15.5 and 11.0).
  return out_features >= 128 && shape_ok(groups, in_features, out_features, rows, elem) &&
         in_features % 32 == 0 && groups > 0 &&
         x != nullptr && w != nullptr && out != nullptr && in_features > 0 && out_features > 0 &&
         256 * in_features * 2 < (int64_t{1} << 31) && aligned16(x) && aligned16(w) && aligned16(out) &&
         bias != nullptr && reinterpret_cast<uintptr_t>(bias) % 8 == 0;
}

template <typename T>
int launch_wide_tanh(const void* x, const void* w, const void* bias, void* out, int64_t groups, int64_t in_features,
                     int64_t out_features, int64_t rows, hipStream_t stream) {
  return launch_op<T, kGgFwd>(GgArgs{w, x, out, const_cast<void*>(bias), rows, static_cast<int>(groups),
                                     static_cast<int>(out_features), static_cast<int>(in_features)}, stream);
}

#define PMSST_GG(T)                                                                                                  \
  template int launch_wide_tanh<T>(const void*, const void*, const void*, void*, int64_t, int64_t, int64_t, int64_t, \
                                   hipStream_t);                                                                    \
  template int launch_wide_dx<T>(const void*, const void*, void*, int64_t, int64_t, int64_t, int64_t, hipStream_t); \
  template int launch_wide_dw<T>(const void*, const void*, void*, void*, int64_t, int64_t, int64_t, int64_t,        \
                                 hipStream_t);
PMSST_GG(bf16)
PMSST_GG(f16)
#undef PMSST_GG

}  // namespace pmsst
