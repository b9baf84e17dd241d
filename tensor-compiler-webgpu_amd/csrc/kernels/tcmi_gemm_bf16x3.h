// fp32 matmul on CDNA4's bf16 matrix cores, with a fused epilogue.
//
// The bf16 matrix cores run 16 times as many flops as the fp32 ones, and a float32
// is, but for the range, the exact sum of three bf16 numbers: x = x0 + x1 + x2, x0 = bf16(x), x1 =
// bf16(x - x0), x2 = x - x0 - x1 (8 + 8 + 8 significant bits; both differences are
// exact). So a·b = Σ a_i·b_j, each a_i·b_j exact in float32, and this kernel sums the
// six products with i + j <= 2 into fp32 accumulators. The three left out are at
// most 2^-24·|a·b| together, one rounding of a float32 product (a = b = 1 + 2^-8 - 2^-17; over
// normal values 2^-27.4 in the root mean square). Six MFMAs take 6/16 of the fp32 instructions' time.
//
// Error against float64 is no larger than the fp32 kernel's (tcmi_gemm.h): it rounds an
// accumulator 6 times in 32 k, the fp32 kernel 8 times or more. Measured without a bias, fp32
// against this: 4096^3 1.1e-6 / 1.0e-6, K 256 2.9e-7 / 2.3e-7, K 64 1.4e-7 / 0.9e-7.
//
// bf16's range ends at 2^-133 and float32's at 2^-149, so operands are split times 2^24: the parts of
// every finite float32 below 2^103, subnormal ones too, then hold all its bits, and the sums are
// multiplied by 2^-48 at the end. (Exact, and 1 % faster than to look for operands whose parts
// lose bits: 4096^3 640 us against 645, 8192 x 1024 x 4096 with its gradients 1054 / 1069; a look at each
// operand's magnitude as it is split 652, 1107.) Where that overflows, the fp32 kernel decides: a
// tile with a sum that is not finite (an infinity or NaN among the operands, one that the scale or
// bf16's rounding makes infinite, a sum of 2^80 or more) is computed again by gemm_f32_sum, in the
// same workgroup.
//
// Operands are tcmi_gemm.h's views. The thread that loads an operand element splits it, so
// LDS holds three bf16 tiles per operand and every wavefront reads its fragments as they
// enter the MFMA, 8 consecutive k of one row (or column) per lane in one ds_read_b128:
//   tile[part][q][line] of 16 bytes: k = 8q .. 8q+7 of `line` (A's row, B's column),
// which neither the reads (16 lines of each of the 4 q) nor the writes (the same, or 64 lines of one
// q) find in conflict (SQ_LDS_BANK_CONFLICT 0; with the planes 64 bytes further apart
// half of the LDS cycles were conflicts).
//
// A unit is one (line, q): 8 elements one thread loads, splits and stores. Where k is the
// contiguous index (KC) its loads are two of 128 bits (4-byte aligned: any row length),
// elsewhere eight of 32 bits, consecutive lanes on consecutive lines. They are buffer
// loads: an element outside the operand is given an offset past the buffer's end and
// reads as 0, with no branch, so the count of loads in flight is static and the wait
// before a split is for that unit's loads alone.
//
// Pipeline: while slice s (32 of K) feeds the matrix cores from one LDS buffer, the units
// of slice s + 1 are split and stored to the other, a share beside each column of tiles,
// their vector instructions between its MFMAs, and each unit's registers take slice
// s + 2's loads as soon as they are free, so a load has a whole slice to arrive. The one
// barrier of a slice stands before its last column, which multiplies while the next
// slice's first fragments are read.
//
// What bounds it: power, where tiles are many. 4096^3 takes 610 - 640 us (220 TFLOP/s; the fp32 kernel
// 1040 us, 132) in 1.33 M cycles, the matrix cores busy for 59 % of them and LDS for 26 %, at 2.07 GHz; on
// zeros the same cycles run at 2.39 GHz, 543 us. With one tile a CU (8192 x 1024 x 256, 39 us at 2.4 GHz)
// the matrix cores are busy for 26 % and LDS for 23 %: the chain of a slice from its loads to its
// products stands open. Tried: 128 x 256 tiles
// by 4 wavefronts of 64 x 128 (less LDS traffic, one wavefront per SIMD) 707 us; two or four
// slices of loads in flight, and K groups inside a workgroup, no faster.

#pragma once

#include "tcmi_gemm.h"

namespace tcmi {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

// Offset given to an element outside its operand: past every buffer this kernel takes
// (the lowering keeps operands under 2^31 bytes).
constexpr uint32_t BEYOND = 0x80000000u;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two floats rounded to bf16 (nearest even), the first in the low half.
__device__ __forceinline__ bf16x2 bf16_pair(float a, float b) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  return __builtin_convertvector((f2{a, b}), bf16x2);
}
// x less the pair's low (high) half: one dot product with (-1, 0) ((0, -1)), exact where the
// half is x rounded to bf16. The weights come from registers: as an inline constant the
// instruction would read a float's -1 as a pair.
struct Minus {
  uint32_t lo = 0x0000bf80u, hi = 0xbf800000u;
  __device__ __forceinline__ Minus() { asm("" : "+s"(lo), "+s"(hi)); }
  __device__ __forceinline__ float less_lo(float x, bf16x2 p) const { return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, lo), p, x, false); }
  __device__ __forceinline__ float less_hi(float x, bf16x2 p) const { return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, hi), p, x, false); }
};
// What operands are multiplied by before they are split, so that a float32's lowest bit, 2^-149,
// is above bf16's least normal value.
constexpr float SPLIT_SCALE = 0x1p24f;

// The operand's line index (A: row, B: column) and its k index as element offsets.
template <class V, bool B>
struct Axis {
  static constexpr bool MAPPED = mapped_view<V>(0);
  static __device__ __forceinline__ uint32_t line(uint32_t x) { return static_cast<uint32_t>(B ? vcol<V>(x) : vrow<V>(x)); }
  static __device__ __forceinline__ uint32_t k(uint32_t x) { return static_cast<uint32_t>(B ? vrow<V>(x) : vcol<V>(x)); }
};

// One operand's tile of L lines x 32 k, staged by THREADS threads. KC: k contiguous (groups
// of 4 where the view is mapped); KT: the K range may end inside a slice.
template <class V, bool B, int L, int THREADS, bool KC, bool KT>
struct Bf16x3Stage {
  using X = Axis<V, B>;
  static constexpr int PLANE = L * 16;
  static constexpr int PART = 4 * PLANE;
  static constexpr int BYTES = 3 * PART;
  static constexpr int ALL = 4 * L;
  static constexpr int UNITS = (ALL + THREADS - 1) / THREADS;   // per thread; past ALL, loads of 0 and no store

  __amdgpu_buffer_rsrc_t buf;
  uint32_t at[UNITS];    // byte offset of the unit's line (and, unmapped, of its first k in a slice)
  float x[UNITS][8];     // the slice in flight
  Minus minus;

  static __device__ __forceinline__ int unit_line(int u) { return KC ? u / 64 * 16 + u % 16 : u % L; }
  static __device__ __forceinline__ int unit_q(int u) { return KC ? u / 16 % 4 : u / L; }

  __device__ __forceinline__ void begin(const float* p, uint32_t bytes, uint32_t line0, uint32_t lines, int tid) {
    buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, static_cast<int>(bytes), 0x00020000);
#pragma unroll
    for (int v = 0; v < UNITS; ++v) {
      const int u = tid + v * THREADS;
      const uint32_t line = line0 + unit_line(u);
      at[v] = line < lines && u < ALL ? 4 * (X::line(line) + (X::MAPPED ? 0u : X::k(8 * unit_q(u)))) : BEYOND;
    }
  }

  // The loads of unit v of the slice at k0, of a K range ending at kend.
  __device__ __forceinline__ void load(int v, uint32_t k0, uint32_t kend, int tid) {
    const uint32_t kq = 8 * unit_q(tid + v * THREADS);
    if constexpr (KC) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t k = k0 + kq + 4 * h;
        uint32_t off = at[v];
        if constexpr (X::MAPPED) {
          if (off != BEYOND) off += 4 * X::k(!KT || k < kend ? k : 0u);
        } else {
          off += 16 * h;
          // A group of 4 that crosses kend is loaded 1-3 elements early (inside its
          // line: the range holds at least 4) and moved into place by split.
          if (KT && off < BEYOND) off += 4 * (k + 4 > kend ? k0 - (k + 4 - kend) : k0);
        }
        if (KT && k >= kend) off = BEYOND;
        constexpr bool FIXED = !X::MAPPED && !KT;   // the slice's k in the scalar part of the offset
        const u4 r = __builtin_amdgcn_raw_buffer_load_b128(buf, static_cast<int>(off), FIXED ? static_cast<int>(4 * k0) : 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[v][4 * h + e] = __uint_as_float(r[e]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t k = k0 + kq + e;
        uint32_t off = at[v];
        if constexpr (X::MAPPED) {
          if (off != BEYOND) off += 4 * X::k(!KT || k < kend ? k : 0u);
        }
        if (KT && k >= kend) off = BEYOND;
        // The scalar part of the offset stays inside the operand where every lane's k is past the end.
        const uint32_t ke = !KT || k0 + e < kend ? k0 + e : 0u;
        const uint32_t r = __builtin_amdgcn_raw_buffer_load_b32(buf, static_cast<int>(off), X::MAPPED ? 0 : static_cast<int>(4 * X::k(ke)), 0);
        x[v][e] = __uint_as_float(r);
      }
    }
  }

  // Unit v (of the slice at k0) split into its three parts, stored to `tile`.
  __device__ __forceinline__ void split(int v, char* tile, uint32_t k0, uint32_t kend, int tid) {
    const int u = tid + v * THREADS;
    float* e = x[v];
    if constexpr (KC && KT && !X::MAPPED) {
      if (k0 + 32 > kend) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t k = k0 + 8 * unit_q(u) + 4 * h;
          const uint32_t over = k < kend && k + 4 > kend ? k + 4 - kend : 0u;
#pragma unroll
          for (uint32_t s = 1; s < 4; ++s) {
            if (over == s) {
#pragma unroll
              for (uint32_t i = 0; i < 4; ++i) e[4 * h + i] = i + s < 4 ? e[4 * h + i + s] : 0.f;
            }
          }
        }
      }
    }
    u4 p0, p1, p2;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = vop<V>(e[2 * i]) * SPLIT_SCALE, b = vop<V>(e[2 * i + 1]) * SPLIT_SCALE;
      const bf16x2 q0 = bf16_pair(a, b);
      const float a1 = minus.less_lo(a, q0), b1 = minus.less_hi(b, q0);
      const bf16x2 q1 = bf16_pair(a1, b1);
      p0[i] = __builtin_bit_cast(uint32_t, q0);
      p1[i] = __builtin_bit_cast(uint32_t, q1);
      p2[i] = __builtin_bit_cast(uint32_t, bf16_pair(minus.less_lo(a1, q1), minus.less_hi(b1, q1)));
    }
    if (ALL % THREADS != 0 && u >= ALL) return;
    char* t = tile + unit_q(u) * PLANE + unit_line(u) * 16;
    *reinterpret_cast<u4*>(t) = p0;
    *reinterpret_cast<u4*>(t + PART) = p1;
    *reinterpret_cast<u4*>(t + 2 * PART) = p2;
  }
};

// C tile of BM x BN = (WM·TM·16) x (WN·TN·16) by WM x WN wavefronts, as gemm_f32's (the same
// arguments, accumulator layout, epilogue and K split); a_bytes and b_bytes are the operand
// buffers' sizes. FM, FN, FW: gemm_f32_sum's tiles for a recomputed tile (same BM, BN, threads).
template <int WM, int WN, int TM, int TN, bool AKC, bool BKC, bool KT, int AMODE, int BMODE, bool SPLIT, class AV, class BV, class Epi,
          class Args = TcmiArgs>
__device__ __forceinline__ void gemm_bf16x3(const Args& A, const float* __restrict__ a_ptr, const float* __restrict__ b_ptr,
                                            const uint32_t a_bytes, const uint32_t b_bytes, const uint32_t batch, const uint32_t M,
                                            const uint32_t K, const uint32_t N, const uint32_t chunks, const uint32_t chunkK,
                                            const uint32_t zid, const uint32_t tx, const uint32_t ty) {
  static_assert(WM == 2, "gemm_f32_sum's wavefront rows");
  static_assert(TN > 1, "a slice's splits stand beside every column of tiles but the last");
  constexpr int THREADS = 64 * WM * WN;
  constexpr int BM = WM * TM * 16, BN = WN * TN * 16;
  using SA = Bf16x3Stage<AV, false, BM, THREADS, AKC, KT>;
  using SB = Bf16x3Stage<BV, true, BN, THREADS, BKC, KT>;
  constexpr int BUF = SA::BYTES + SB::BYTES;
  using Tiles = GemmTiles<BM, BN, 16, AMODE, BMODE, AV, BV>;
  constexpr int FP32 = 4 * 2 * (Tiles::A + Tiles::B);
  constexpr int POOL = 2 * BUF > FP32 ? 2 * BUF : FP32;
  float* const pool = lds_pool<POOL / 4>();
  char* const lds = reinterpret_cast<char*>(pool);

  const uint32_t kz = SPLIT ? zid % chunks : 0u;
  const uint32_t bz = SPLIT ? zid / chunks : zid;
  const uint32_t kbeg = SPLIT ? kz * chunkK : 0u;
  const uint32_t kend = SPLIT ? min(K, kbeg + chunkK) : K;
  const uint32_t m0 = ty * BM, n0 = tx * BN;

  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int t16 = lane & 15, q = lane >> 4;

  f4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};

  SA sa;
  SB sb;
  const uint32_t a_off = static_cast<uint32_t>(AV::batch(bz)), b_off = static_cast<uint32_t>(BV::batch(bz));
  sa.begin(a_ptr + a_off, a_bytes - 4 * a_off, m0, M, tid);
  sb.begin(b_ptr + b_off, b_bytes - 4 * b_off, n0, N, tid);

  // Fragment addresses of this lane in a buffer.
  const int fa = q * SA::PLANE + (wm * TM * 16 + t16) * 16;
  const int fb = SA::BYTES + q * SB::PLANE + (wn * TN * 16 + t16) * 16;
  auto frag = [&](const char* p) { return *reinterpret_cast<const bf16x8*>(p); };

  const uint32_t slices = (kend - kbeg + 31) / 32;
#pragma unroll
  for (int v = 0; v < SA::UNITS; ++v) sa.load(v, kbeg, kend, tid);
#pragma unroll
  for (int v = 0; v < SB::UNITS; ++v) sb.load(v, kbeg, kend, tid);
#pragma unroll
  for (int v = 0; v < SA::UNITS; ++v) {
    sa.split(v, lds, kbeg, kend, tid);
    if (slices > 1) sa.load(v, kbeg + 32, kend, tid);
  }
#pragma unroll
  for (int v = 0; v < SB::UNITS; ++v) {
    sb.split(v, lds + SA::BYTES, kbeg, kend, tid);
    if (slices > 1) sb.load(v, kbeg + 32, kend, tid);
  }
  __syncthreads();

  bf16x8 a[TM][3], b[3];
  auto a_frags = [&](const char* from, int p) {
#pragma unroll
    for (int i = 0; i < TM; ++i) a[i][p] = frag(from + fa + p * SA::PART + i * 256);
  };
  auto b_frags = [&](const char* from, int j, bf16x8 (&f)[3]) {
#pragma unroll
    for (int p = 0; p < 3; ++p) f[p] = frag(from + fb + p * SB::PART + j * 256);
  };
  b_frags(lds, 0, b);
#pragma unroll
  for (int p = 2; p >= 0; --p) a_frags(lds, p);

  // One slice from buffer `cur`; `next`: the k of the slice whose units are split into the
  // other buffer, `then`: of the slice loaded after it (`more`, `again`: whether they exist).
  auto slice = [&](const int cur, const uint32_t next, const bool more, const uint32_t then, const bool again) {
    const char* from = lds + cur * BUF;
    char* to = lds + (cur ^ 1) * BUF;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      bf16x8 bn[3];
      if (j + 1 < TN) {
        b_frags(from, j + 1, bn);
      } else if (more) {
        // Every read of this buffer and every store to the other is done: after the barrier
        // the next slice's fragments are read while the last column multiplies, A's parts
        // each as soon as their last product here has taken them.
        __syncthreads();
        b_frags(to, 0, bn);
      }
      // A column's six products are added to the sums in turn, the largest last: an accumulator
      // rounds 6 times in 32 k. B first, A second: lane (t16, q) holds row t16,
      // columns 4q .. 4q+3.
      constexpr int PA[6] = {2, 1, 1, 0, 0, 0}, PB[6] = {0, 1, 0, 2, 1, 0};
#pragma unroll
      for (int s = 0; s < 6; ++s) {
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[PB[s]], a[i][PA[s]], acc[i][j], 0, 0, 0);
        if (j + 1 == TN && more && (s == 5 || PA[s + 1] != PA[s])) {
          __builtin_amdgcn_sched_barrier(0);
          a_frags(to, PA[s]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // This column's share of the next slice's units: A's, then B's.
      if (j + 1 < TN && more) {
        constexpr int ALL = SA::UNITS + SB::UNITS;
#pragma unroll
        for (int u = j * ALL / (TN - 1); u < (j + 1) * ALL / (TN - 1); ++u) {
          if (u < SA::UNITS) {
            sa.split(u, to, next, kend, tid);
            if (again) sa.load(u, then, kend, tid);
          } else {
            sb.split(u - SA::UNITS, to + SA::BYTES, next, kend, tid);
            if (again) sb.load(u - SA::UNITS, then, kend, tid);
          }
        }
      }
      if (j + 1 < TN && more) {
        // One MFMA, then vector work of the split, in turn: a wavefront's matrix core and
        // vector ALU run side by side.
        constexpr int VALU = (40 * (SA::UNITS + SB::UNITS) / (TN - 1) + 6 * TM - 1) / (6 * TM);
        __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
        for (int n = 0; n < 6 * TM; ++n) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 0; p < 3; ++p) b[p] = bn[p];
    }
  };
  // Slice t is computed from LDS buffer t & 1; the first loop has no condition on any load.
  uint32_t s = 0;
  for (; s + 3 < slices; s += 2) {
    const uint32_t k0 = kbeg + s * 32;
    slice(0, k0 + 32, true, k0 + 64, true);
    slice(1, k0 + 64, true, k0 + 96, true);
  }
  for (; s < slices; ++s) {
    const uint32_t k0 = kbeg + s * 32;
    slice(s & 1, k0 + 32, s + 1 < slices, k0 + 64, s + 2 < slices);
  }
  __syncthreads();

  // The scale taken out; a tile that holds a sum that is not finite is summed again in fp32.
  uint32_t* const seen = reinterpret_cast<uint32_t*>(pool);
  if (tid == 0) *seen = 0u;
  __syncthreads();
  float zero = 0.f;   // NaN after a sum that is not finite
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        zero = fmaf(acc[i][j][r], 0.f, zero);
        acc[i][j][r] *= 1.f / (SPLIT_SCALE * SPLIT_SCALE);
      }
  if (!(zero == 0.f)) *seen = 1u;
  __syncthreads();
  const bool redo = __builtin_amdgcn_readfirstlane(*seen) != 0u;
  if (redo) {
    __syncthreads();
    gemm_f32_sum<TM, TN, 16, 1, AMODE, BMODE, AV, BV, WN, false>(pool, pool + 2 * Tiles::A, a_ptr + AV::batch(bz), b_ptr + BV::batch(bz), M,
                                                                  N, kbeg, kend, (kend - kbeg + 15) / 16, m0, n0, tid, acc);
  }
  gemm_store<TM, TN, SPLIT, Epi>(A, acc, batch, M, N, kz, bz, m0 + wm * TM * 16 + t16, n0 + wn * TN * 16 + 4 * q);
}

}  // namespace tcmi
