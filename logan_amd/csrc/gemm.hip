// Prefill / large-batch product with MLX-affine weights on MFMA (gfx950):
//   y[m][n] = sum_k x[m][k] * bf16(code[n][k] * scale[n][k/gs] + bias[n][k/gs])
// the semantics of logan-metal's QMM (backend_metal.mm:1480-1560: each
// dequantised weight rounded to bf16 in threadgroup memory, bf16 x bf16
// products accumulated in f32, bf16 output).
//
// affine_qmm_tile_kernel serves all but the smallest products and, of those
// whose operands are off the alignment of its wider copies (packed rows off 16
// bytes, scales or biases off 4), the ones of up to 64 rows: those take
// affine_qmm_kernel (64 x 64 tiles, 4 waves, dword loads).
// Operand layout of v_mfma_f32_32x32x16_bf16 (checked on the device): lane l
// holds row (col) l % 32 and 8 consecutive k at offset 8 * (l / 32) of each
// 16-wide k slice; the result's element i of lane l is row
// 8 * (i / 4) + 4 * (l / 32) + i % 4, column l % 32.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "affine_dev.hpp"
#include "lh_internal.hpp"
#include "mfma_dev.hpp"

namespace lh {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct GemmParams {
  const uint8_t *w;
  const uint16_t *sc;
  const uint16_t *bi;
  const uint16_t *x;
  void *y;
  long long row_bytes;
  int M, N, K, ng, gs, fp16, x_stride, y_stride, y_bf16;
};

constexpr int kTile = 64;        // block tile (m and n) and k step
constexpr int kLdsStride = 72;   // bf16 per LDS row: 64 + 8 pad (no bank conflicts)

// Codes per dequantising thread: 16 (4 per row of 64) for widths whose
// 16-code runs start on a dword boundary; 5-bit runs of 32 codes (2 per row).
template <int BITS>
struct DeqGeom {
  static constexpr int CPT = BITS == 5 ? 32 : 16;
  static constexpr int THREADS = kTile * (kTile / CPT);  // 256 or 128
  static constexpr int DW = CPT * BITS / 32;             // dwords of codes
};

template <int BITS>
__device__ __forceinline__ uint32_t code_of(const uint32_t (&w)[DeqGeom<BITS>::DW], int j) {
  const int bit = j * BITS, i = bit >> 5, sh = bit & 31;
  uint32_t c = w[i] >> sh;
  if (sh + BITS > 32) c |= w[i + 1] << (32 - sh);
  return c & ((1u << BITS) - 1u);
}

// Split-K: the blocks of one tile that share a k range write f32 partial
// sums part[z][m][n] into one of kQSlots module-scope slots (a SlotRing
// lease: calls on any streams that would overlap on a slot are ordered on
// the device); qmm_reduce_kernel adds them in z order and writes y.
// slot < 0: one k range, y written directly.
constexpr int kQSlots = 2;
constexpr size_t kQSlotFloats = size_t(1) << 23;  // 32 MB per slot
static __device__ __align__(256) float g_qmm_part[kQSlots * kQSlotFloats];

__device__ __forceinline__ void qmm_store(const GemmParams &p, int slot, int z, int m, int n,
                                          float v) {
  if (slot >= 0)
    g_qmm_part[(size_t)slot * kQSlotFloats + ((size_t)z * p.M + m) * p.N + n] = v;
  else if (p.y_bf16)
    reinterpret_cast<__bf16 *>(p.y)[(size_t)m * p.y_stride + n] = (__bf16)v;
  else
    reinterpret_cast<float *>(p.y)[(size_t)m * p.y_stride + n] = v;
}

// all KS loads of a thread issued before the first add; V = 4 when rows are
// a multiple of 4 columns (16-byte partial loads), the y store then one 8- or
// 16-byte store when y rows are 16-byte aligned (yvec)
template <int KS, int V>
__global__ __launch_bounds__(256) void qmm_reduce_kernel(GemmParams p, int slot, int yvec) {
  typedef float fv __attribute__((ext_vector_type(V)));
  const float *part = g_qmm_part + (size_t)slot * kQSlotFloats;
  const size_t MN = (size_t)p.M * p.N, nv = MN / V;
  for (size_t v = (size_t)blockIdx.x * 256 + threadIdx.x; v < nv; v += (size_t)gridDim.x * 256) {
    const size_t i = v * V;
    fv t[KS];
#pragma unroll
    for (int z = 0; z < KS; ++z) t[z] = __builtin_nontemporal_load(reinterpret_cast<const fv *>(part + z * MN + i));
    fv s = t[0];
#pragma unroll
    for (int z = 1; z < KS; ++z) s += t[z];  // in k order
    const size_t o = (i / p.N) * p.y_stride + i % p.N;
    if (p.y_bf16) {
      __bf16 *y = reinterpret_cast<__bf16 *>(p.y) + o;
      if constexpr (V == 4) {
        if (yvec) {
          typedef __bf16 b4 __attribute__((ext_vector_type(4)));
          *reinterpret_cast<b4 *>(y) = b4{(__bf16)s[0], (__bf16)s[1], (__bf16)s[2], (__bf16)s[3]};
          continue;
        }
      }
#pragma unroll
      for (int e = 0; e < V; ++e) y[e] = (__bf16)s[e];
    } else {
      float *y = reinterpret_cast<float *>(p.y) + o;
      if constexpr (V == 4) {
        if (yvec) {
          *reinterpret_cast<fv *>(y) = s;
          continue;
        }
      }
#pragma unroll
      for (int e = 0; e < V; ++e) y[e] = s[e];
    }
  }
}

template <int V>
static void launch_qmm_reduce(const GemmParams &p, int slot, int KS, hipStream_t st) {
  const size_t nv = (size_t)p.M * p.N / V;
  const dim3 grid((unsigned)std::min<size_t>((nv + 255) / 256, 4096));
  const int es = p.y_bf16 ? 2 : 4;
  const int yvec = (reinterpret_cast<uintptr_t>(p.y) & 15) == 0 && ((long long)p.y_stride * es) % 16 == 0;
  switch (KS) {
#define LH_QRED(k) \
  case k: hipLaunchKernelGGL((qmm_reduce_kernel<k, V>), grid, dim3(256), 0, st, p, slot, yvec); break;
    LH_QRED(2) LH_QRED(3) LH_QRED(4) LH_QRED(5) LH_QRED(6) LH_QRED(7) LH_QRED(8) LH_QRED(9)
    LH_QRED(10) LH_QRED(11) LH_QRED(12) LH_QRED(13) LH_QRED(14) LH_QRED(15) LH_QRED(16)
#undef LH_QRED
    default: break;
  }
}

template <int BITS>
__global__ __launch_bounds__(256) void affine_qmm_kernel(GemmParams p, int ksteps, int slot) {
  using G = DeqGeom<BITS>;
  __shared__ __align__(16) __bf16 sW[kTile * kLdsStride];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bm0 = blockIdx.x * kTile, bn0 = blockIdx.y * kTile;
  const int wm = wave >> 1, wn = wave & 1;
  const int half = lane >> 5, l32 = lane & 31;

  // dequantising role: row n = tid / (64 / CPT), codes [kq, kq + CPT)
  const int dn = tid / (kTile / G::CPT);
  const int kq = (tid % (kTile / G::CPT)) * G::CPT;
  const bool deq = tid < G::THREADS;
  const int nrow = min(bn0 + dn, p.N - 1);
  const uint8_t *wrow = p.w + (size_t)nrow * p.row_bytes;
  const uint16_t *srow = p.sc + (size_t)nrow * p.ng;
  const uint16_t *brow = p.bi + (size_t)nrow * p.ng;

  // x operand row of this lane (clamped; rows past M are never stored)
  const int xm = min(bm0 + wm * 32 + l32, p.M - 1);
  const uint16_t *xrow = p.x + (size_t)xm * p.x_stride;

  // software pipeline: the loads of step k0 + 64 are issued before step k0 is
  // dequantised and multiplied
  // (two register buffers with compile-time indices: the loop body is
  // unrolled by two steps)
  uint32_t wv0[G::DW], wv1[G::DW];
  uint32_t sr0 = 0, br0 = 0, sr1 = 0, br1 = 0;
  uint4 xa0[4], xa1[4];
  auto issue = [&](int k0, uint32_t (&wv)[G::DW], uint32_t &sraw, uint32_t &braw, uint4 (&xa)[4]) {
    if (deq) {
      const uint32_t *src = reinterpret_cast<const uint32_t *>(wrow + (size_t)(k0 + kq) * BITS / 8);
#pragma unroll
      for (int i = 0; i < G::DW; ++i) wv[i] = src[i];
      const int gidx = (k0 + kq) / p.gs;
      sraw = srow[gidx];
      braw = brow[gidx];
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      xa[ks] = *reinterpret_cast<const uint4 *>(xrow + k0 + 16 * ks + 8 * half);
  };
  f32x16 acc = {};
  auto step = [&](const uint32_t (&wv)[G::DW], uint32_t sraw, uint32_t braw, const uint4 (&xa)[4]) {
    if (deq) {
      const float s = aux_to_f32_sel(sraw, p.fp16), b = aux_to_f32_sel(braw, p.fp16);
      uint32_t packed[G::CPT / 2];
#pragma unroll
      for (int j = 0; j < G::CPT; j += 2) {
        bf16x2 v;
        v[0] = (__bf16)fmaf((float)code_of<BITS>(wv, j), s, b);
        v[1] = (__bf16)fmaf((float)code_of<BITS>(wv, j + 1), s, b);
        packed[j / 2] = __builtin_bit_cast(uint32_t, v);
      }
      uint4 *dst = reinterpret_cast<uint4 *>(sW + dn * kLdsStride + kq);
#pragma unroll
      for (int v = 0; v < G::CPT / 8; ++v)
        dst[v] = make_uint4(packed[4 * v], packed[4 * v + 1], packed[4 * v + 2], packed[4 * v + 3]);
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const bf16x8 a = __builtin_bit_cast(bf16x8, xa[ks]);
      const bf16x8 b = *reinterpret_cast<const bf16x8 *>(sW + (wn * 32 + l32) * kLdsStride + 16 * ks +
                                                        8 * half);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    }
    __syncthreads();
  };
  const int z = blockIdx.z;
  const int kb = z * ksteps * kTile, ke = min(p.K, kb + ksteps * kTile);
  issue(kb, wv0, sr0, br0, xa0);
  for (int k0 = kb; k0 < ke; k0 += 2 * kTile) {
    if (k0 + kTile < ke) issue(k0 + kTile, wv1, sr1, br1, xa1);
    __builtin_amdgcn_sched_barrier(0);
    step(wv0, sr0, br0, xa0);
    if (k0 + kTile < ke) {
      if (k0 + 2 * kTile < ke) issue(k0 + 2 * kTile, wv0, sr0, br0, xa0);
      __builtin_amdgcn_sched_barrier(0);
      step(wv1, sr1, br1, xa1);
    }
  }
  // store: element i of this lane is (row 8*(i/4) + 4*half + i%4, col l32)
  const int n = bn0 + wn * 32 + l32;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int m = bm0 + wm * 32 + 8 * (i / 4) + 4 * half + (i % 4);
    if (m < p.M && n < p.N) qmm_store(p, slot, z, m, n, acc[i]);
  }
}

constexpr int kQTargetBlocks = 512;  // about two blocks per CU
static SlotRing g_qmm_slots(kQSlots);

// ---------------------------------------------------------------------------
// Products of up to kQMultiMax matrices that read the same x (q/k/v, qkvz/ba,
// gate/up) in one grid, BM x 128 output tiles, one 8-wave block per CU (two of
// 32-row tiles).
//
// What bounds it: 256-row tiles the matrix and vector pipes, which hardly
// overlap (8-bit, 2 x 14336 columns, K 4096, M 2048: of 2,040 cycles per 64-k
// step a SIMD's matrix pipe is busy 1,024 and its vector pipe 690, most of it
// the forming of the bf16 weights, at the 1.8-1.9 GHz the card holds under this
// load); tiles of at most 128 rows a step's chain of LDS reads, forming, MFMAs
// and barrier with two waves a SIMD (M 100: 1,760 cycles for 512 and 590), the
// codes arriving at 2.7 TB/s. Hence:
//   * every copy from memory goes straight into LDS (global_load_lds, issued
//     through inline assembly and waited for by count) NST - 1 steps ahead: x
//     rows, packed codes, and the scale / bias words a chunk of steps at a
//     time. No VGPR holds a load in flight, and every line is read whole;
//   * the weights never go back to LDS: a lane reads its run of codes, forms
//     bf16(code * scale + bias) in the MFMA operand's layout and feeds it to
//     all MI = BM / 32 row tiles. The 8 waves are 4 (32 columns each) x 2 (k
//     halves of each step), so every weight is formed once per block; the two
//     waves of a tile add their sums through LDS after the last step;
//   * the copies of a step are issued between its MFMAs, at the places the
//     scheduling barriers fix: issued together at its start they hold the
//     waves at the CU's one address path before their first MFMA (measured while
//     it was written, 28672 x 4096, 8-bit, M 2048: 600 us so, 551 us spread).
// Measured, us, a product repeated on the same operands (before: 256 x 128 tiles
// with the weights staged in LDS as bf16, 128 x 128 below 256 rows):
//   8-bit, 28672 x 4096: M 100  66.0 -> 39.3, M 2048  522 -> 467 (1030 TFLOP/s)
//   8-bit, 4096 x 14336: M 100  40.0 -> 31.6, M 2048  251 -> 220
//   4-bit, 12352 x 2048: M 512  36.8 -> 32.9;  2048 x 4096: 30.1 -> 26.2
// Within a step, wave k-group kg and lane half h own the run of 16 codes at
// k = 16 (2 kg + h), and MFMA slice j takes 8 of them: any order of k serves
// as long as both operands use it.
// LDS: x rows are 128 bytes, 16-byte granule q of row r at q ^ ((r >> 1) & 7)
// (16 rows of an operand read spread over all banks); 8-bit codes likewise at
// q ^ ((r >> 2) & 3) of their 64 bytes; the narrower rows are not swizzled.
// Conflict cycles counted per LDS instruction: none with 128-row 8-bit tiles, 0.66
// with 256 rows (5 % of the time), 0.4-0.5 at 4 bits.
constexpr int kTN = 128;   // tile columns
constexpr int kQMultiMax = 8;

struct QmmMat {
  const uint8_t *w;
  const uint16_t *sc;
  const uint16_t *bi;
  void *y;
  long long row_bytes;
  int N, ng, y_stride, col0;  // col0: first column of this matrix in split partial rows (a multiple of 4)
};
struct QmmMulti {
  QmmMat m[kQMultiMax];
  int tile_start[kQMultiMax + 1];  // first 128-column tile of matrix i
  const uint16_t *x;
  int n, M, K, gs, fp16, x_stride, y_bf16, part_N;
  int vec;  // y rows take 16-byte stores
};

__device__ __forceinline__ uint32_t q_lds_addr(const void *p) {
  return (uint32_t)(uintptr_t)((__attribute__((address_space(3))) const uint8_t *)p);
}
// lane l's 16 (4, 2) bytes at base + off land at lds + 16 l (4 l; the 2 as a
// zero-extended dword); lds and base are wave-uniform. Completion counts in vmcnt, unseen by the compiler.
__device__ __forceinline__ void q_copy16(const void *base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void q_copy4(const void *base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
               :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void q_copy2(const void *base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_ushort %0, %1"
               :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void q_wait() {
  static_assert(N >= 0 && N <= 63, "vmcnt is 6 bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// wait until all but the last N LDS operations of this wave are done (they
// return in order). A copy into LDS is unseen by the compiler, which places no
// wait between the reads of a stage and the copies that overwrite it.
template <int N>
__device__ __forceinline__ void q_wait_lds() {
  static_assert(N >= 0 && N <= 15, "lgkmcnt is 4 bits");
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}

// Geometry of one instantiation. ALN: packed rows start on 16 bytes (5 bits: on
// 4), scales and biases on 4. Without it the codes come by dwords and the
// sidecars may start on the second half of one.
template <int BITS, int MI, bool GS64, bool ALN>
struct QTile {
  static constexpr int BM = 32 * MI;               // tile rows
  static constexpr int RB = 8 * BITS;              // code bytes per row and step
  static constexpr int XB = BM * 128;              // x bytes per stage
  static constexpr int WB = kTN * RB;
  // LDS of a block: 32-row tiles leave room for a second one on the CU. With one,
  // products of few rows and more than 256 column tiles ran in full rounds (8 and
  // 6 bits with 8 stages, M 5, us, 64 x 64 kernel / so / with a second block:
  // 33000 x 1024 15 / 19 / 14, 100000 x 2304 68 / 75 / 54, 152064 x 4096 266 /
  // 166 / 154; 256 tiles or fewer the same: 28672 x 4096 47 / 31 / 31).
  static constexpr int LIM = BM == 32 ? 81920 : 163840;
  // steps of a chunk of scale / bias words, dwords per row of it: CS groups of
  // 64 that may start inside a dword; groups of 32 start on one (when ALN)
  static constexpr int ndw(int cs) { return GS64 ? cs / 2 + 1 : cs + !ALN; }
  static constexpr int ab(int cs) { return 2 * kTN * ndw(cs) * 4; }  // [scale, bias][128][ndw]
  // stages of x and of the codes (a step's codes are read a step ahead of its x)
  static constexpr int rings(int nst) { return nst * XB + (nst - 1) * WB; }
  static constexpr int fit(int nst) { return rings(nst) + 2 * ab(8) <= LIM ? nst : fit(nst - 1); }
  static constexpr int NST = BM >= 192 ? 4 : BM == 128 ? 5 : BM == 64 ? 8 : fit(8);
  static constexpr int NWS = NST - 1;
  static constexpr int AUX0 = rings(NST);
  static constexpr int CS = AUX0 + 2 * ab(8) <= LIM ? 8 : AUX0 + 2 * ab(6) <= LIM ? 6 : 4;
  static constexpr int NDW = ndw(CS);
  static constexpr int AB = ab(CS);
  static constexpr int XI = BM / 8;                // x copies (1 KB) of a stage
  static constexpr int LX = (XI + 7) / 8;          // per wave
  static constexpr bool W16 = ALN && BITS != 5;    // code copies of 1 KB, else of 256 bytes
  static constexpr int WI = W16 ? BITS : 4 * BITS;
  static constexpr int LW = (WI + 7) / 8;
  static constexpr int L = LX + LW;
  static constexpr int NA = (4 * NDW + 7) / 8;     // scale / bias copies per wave and chunk
  static constexpr int RINGS = AUX0 + 2 * AB;
  // sum exchange: a 32 x 32 tile per wave; stores: one of 33-float rows
  static constexpr int ROUND = 8 * 4096 + 8 * 32 * 33 * 4;
  static constexpr int BYTES = RINGS > ROUND ? RINGS : ROUND;
  static_assert(BYTES <= LIM && CS >= NST, "ring geometry");
  static_assert((NST - 2) * L + NA <= 63, "vmcnt is 6 bits");
};

// wait until all but the last n * L (n <= MAX, uniform) copies of this wave have landed
template <int L, int MAX>
__device__ __forceinline__ void q_wait_steps(int n) {
  if constexpr (MAX > 0) {
    if (n >= MAX) q_wait<MAX * L>();
    else q_wait_steps<L, MAX - 1>(n);
  } else {
    q_wait<0>();
  }
}

// the lane's run of 16 codes from its row's RB bytes in LDS
template <int BITS>
struct QRun {
  uint32_t w[BITS == 4 ? 2 : BITS == 8 ? 4 : 3];
  __device__ __forceinline__ void read(const uint8_t *row, int r, int run) {
    if constexpr (BITS == 8) {
      const uint4 v = *reinterpret_cast<const uint4 *>(row + ((run ^ ((r >> 2) & 3)) << 4));
      w[0] = v.x;
      w[1] = v.y;
      w[2] = v.z;
      w[3] = v.w;
    } else if constexpr (BITS == 4) {
      const uint2 v = *reinterpret_cast<const uint2 *>(row + 8 * run);
      w[0] = v.x;
      w[1] = v.y;
    } else {
      // the dword holding the first code on; 5-bit codes may start at its bit 16
      const uint32_t *p = reinterpret_cast<const uint32_t *>(row + ((2 * BITS * run) & ~3));
#pragma unroll
      for (int i = 0; i < 3; ++i) w[i] = p[i];
    }
  }
  // codes 8 j + 2 i, + 1 as f32 (from what split() left)
  __device__ __forceinline__ void split(int j, int sh, uint32_t (&t)[3]) const {
    if constexpr (BITS == 4) {
      // (asm: the compiler would undo the two masks into a shift and a mask per code)
      t[1] = w[j] >> 4;
      asm("v_and_b32 %0, 0xf0f0f0f, %1" : "=v"(t[0]) : "v"(w[j]));
      asm("v_and_b32 %0, 0xf0f0f0f, %0" : "+v"(t[1]));
    } else if constexpr (BITS == 8) {
      t[0] = w[2 * j];
      t[1] = w[2 * j + 1];
    } else if constexpr (BITS == 5) {
      // sh: bit of the run's first code in w[0] (0 or 16)
      t[0] = __builtin_amdgcn_alignbit(w[1], w[0], sh);
      t[1] = __builtin_amdgcn_alignbit(w[2], w[1], sh);
      t[2] = w[2] >> sh;
    } else {
#pragma unroll
      for (int i = 0; i < 3; ++i) t[i] = w[i];
    }
  }
  // bf16(code * s + b) of codes 8 j + 2 i, + 1, packed
  static __device__ __forceinline__ uint32_t pair(const uint32_t (&t)[3], int j, int i, float s, float b) {
    float f[2];
    if constexpr (BITS == 4) {
      f[0] = (float)((t[0] >> (8 * i)) & 255u);
      f[1] = (float)((t[1] >> (8 * i)) & 255u);
    } else if constexpr (BITS == 8) {
      f[0] = (float)((t[i >> 1] >> (16 * (i & 1))) & 255u);
      f[1] = (float)((t[i >> 1] >> (16 * (i & 1) + 8)) & 255u);
    } else {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int bit = (8 * j + 2 * i + e) * BITS, q = bit >> 5, o = bit & 31;
        uint32_t v = t[q] >> o;
        if (o + BITS > 32) v |= t[q + 1] << (32 - o);
        f[e] = (float)(v & ((1u << BITS) - 1u));
      }
    }
    bf16x2 v;
    v[0] = (__bf16)fmaf(f[0], s, b);
    v[1] = (__bf16)fmaf(f[1], s, b);
    return __builtin_bit_cast(uint32_t, v);
  }
};

// GS64: groups of 64 codes (a group per step); else any multiple of 32
// (FP16: of the aligned form; the other takes p.fp16)
template <int BITS, int MI, bool GS64, bool FP16, bool ALN>
__global__ __launch_bounds__(512, 2) void affine_qmm_tile_kernel(QmmMulti p, int mtiles, int ntiles,
                                                                 int ksteps, int slot) {
  using G = QTile<BITS, MI, GS64, ALN>;
  constexpr int BM = G::BM, NST = G::NST, CS = G::CS, NDW = G::NDW;
  __shared__ __align__(256) uint8_t smem[G::BYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 3, kg = wave >> 2;
  const int half = lane >> 5, l32 = lane & 31;
  // Block order: each XCD (block id mod 8) takes one run of the tiles, row tiles
  // fastest, so that the row tiles of one (column tile, k range) meet its
  // weights in one L2 and every XCD has as many blocks to within one
  const int total = mtiles * ntiles * ((p.K / 64 + ksteps - 1) / ksteps);
  const int lin = (int)(blockIdx.x & 7) * ((total + 7) / 8) + (int)(blockIdx.x >> 3);
  if (lin >= total) return;
  const int mt = lin % mtiles, col = lin / mtiles;
  const int nt = col % ntiles, z = col / ntiles;
  int mi = 0;
#pragma unroll
  for (int t = 1; t < kQMultiMax; ++t) mi = t < p.n && nt >= p.tile_start[t] ? t : mi;
  mi = __builtin_amdgcn_readfirstlane(mi);
  const QmmMat &mat = p.m[mi];
  const int bm0 = mt * BM, bn0 = (nt - p.tile_start[mi]) * kTN;
  const int kb = z * ksteps * 64;
  int nst = (min(p.K, kb + ksteps * 64) - kb) >> 6;
  // the arguments the loop uses, kept in registers (the copies' memory
  // clobbers would have them loaded again, and waited for, in every step)
  int N = mat.N, ng = mat.ng, gs = p.gs;
  const uint16_t *sc = mat.sc, *bi = mat.bi;
  asm volatile("" : "+s"(N), "+s"(ng), "+s"(gs), "+s"(sc), "+s"(bi), "+s"(nst));

  // ---- this wave's copies: of every stage, LX of x and LW of the codes ----
  uint32_t xoff[G::LX], woff[G::LW], wdst[G::LW];
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(q_lds_addr(smem));
  const uint32_t xdst = lds0 + 1024 * ((wave * G::LX) % G::XI);
#pragma unroll
  for (int i = 0; i < G::LX; ++i) {
    const int r = 8 * ((wave * G::LX + i) % G::XI) + (lane >> 3);  // copies past the tile repeat one
    const int g = (lane & 7) ^ ((r >> 1) & 7);
    xoff[i] = (uint32_t)(min(r, p.M - 1 - bm0) * p.x_stride + 8 * g) * 2u;
  }
#pragma unroll
  for (int i = 0; i < G::LW; ++i) {
    const int c = (wave * G::LW + i) % G::WI, u = 64 * c + lane;
    int r, b;
    if constexpr (!G::W16) {
      r = u / (G::RB / 4);
      const int q = u % (G::RB / 4);
      b = BITS == 8 ? 16 * ((q >> 2) ^ ((r >> 2) & 3)) + 4 * (q & 3) : 4 * q;
    } else {
      r = u / (G::RB / 16);
      const int q = u % (G::RB / 16);
      b = 16 * (BITS == 8 ? q ^ ((r >> 2) & 3) : q);
    }
    woff[i] = (uint32_t)(min(r, N - 1 - bn0) * (int)mat.row_bytes + b);
    wdst[i] = lds0 + NST * G::XB + (G::W16 ? 1024 : 256) * c;
  }
  const uint8_t *xsrc = reinterpret_cast<const uint8_t *>(p.x + (size_t)bm0 * p.x_stride + kb);
  const uint8_t *wsrc = mat.w + (size_t)bn0 * mat.row_bytes + (size_t)kb * BITS / 8;
  // the next step's copy k of L, into the stages at bytes xst, wst of the rings
  int xst = 0, wst = 0;
  auto copy = [&](int k) __attribute__((always_inline)) {
    if (k < G::LX) {
      const int i = k < G::LX ? k : 0;
      q_copy16(xsrc, xoff[i], xdst + xst + 1024 * i);
    } else {
      const int i = k < G::LX ? 0 : k - G::LX;
      if constexpr (G::W16) q_copy16(wsrc, woff[i], wdst[i] + wst);
      else q_copy4(wsrc, woff[i], wdst[i] + wst);
    }
  };
  auto next = [&]() __attribute__((always_inline)) {
    xsrc += 128;
    wsrc += G::RB;
    xst = xst == (NST - 1) * G::XB ? 0 : xst + G::XB;
    wst = wst == (G::NWS - 1) * G::WB ? 0 : wst + G::WB;
  };
  // Scale / bias words: chunks of CS steps, the ndw dwords of each row that
  // hold the chunk's groups (from the dword with the first one on: rows of an
  // odd number of groups start inside a dword), in two buffers. 64
  // consecutive dwords of a chunk's [scale, bias][128][ndw] are one copy.
  // Sidecars that start on the second half of a dword are copied from that
  // dword on (aligned, so never past what holds their first word) and counted
  // from there: lead[] is 1 then.
  uint32_t lead[2] = {0, 0};
  if constexpr (!ALN) {
    lead[0] = (uint32_t)(reinterpret_cast<uintptr_t>(sc) >> 1) & 1u;
    lead[1] = (uint32_t)(reinterpret_cast<uintptr_t>(bi) >> 1) & 1u;
    sc -= lead[0];
    bi -= lead[1];
  }
  const bool g32 = !GS64 && gs == 32;
  const int ndw = GS64 || g32 ? NDW : CS / 2 + 1;
  const uint32_t ldsa = lds0 + G::AUX0;
  // the last dword wholly inside the matrix; when the total is odd, the word
  // after it is copied alone (zero-extended)
  const uint32_t atot = (uint32_t)N * ng * 2u;
  const bool odd = (ALN ? (atot & 2u) != 0 : ((atot ^ 2 * lead[0]) & 2u) != 0 || ((atot ^ 2 * lead[1]) & 2u) != 0) &&
                   bn0 + kTN >= N;
  auto aux_chunk = [&](int c) __attribute__((always_inline)) {
    const int k = kb + 64 * CS * c;
    const uint32_t g0 = GS64 ? (uint32_t)k >> 6 : (uint32_t)k / (uint32_t)gs;
    const int per = 2 * ndw;  // copies of the scales (128 ndw / 64), then the biases'
#pragma unroll
    for (int i = 0; i < G::NA; ++i) {
      int s = wave * G::NA + i;  // copies past the chunk repeat one
      s = s >= 2 * per ? s - 2 * per : s;
      const bool bias = s >= per;
      const uint32_t d = 64 * (bias ? s - per : s) + lane;
      const uint32_t r = GS64 ? d / NDW : g32 ? d / NDW : d / (CS / 2 + 1);
      const uint32_t ld = bias ? lead[1] : lead[0], at = atot + 2 * ld, amax = (at & ~3u) - 4u;
      const uint32_t u16i = ((uint32_t)min(bn0 + (int)r, N - 1) * ng + g0 + ld) & ~1u;
      const uint32_t o = 2 * u16i + 4 * (d - r * ndw);
      const uint16_t *src = bias ? bi : sc;
      const uint32_t dst = __builtin_amdgcn_readfirstlane(ldsa + (c & 1) * G::AB + 256 * s);
      if (!odd) {
        q_copy4(src, min(o, amax), dst);
      } else {
        // (waited for at once: its copies would not be the NA counted)
        if (o == at - 2) q_copy2(src, o, dst);
        else q_copy4(src, min(o, amax), dst);
        q_wait<0>();
      }
    }
  };

  // ---- operands ----
  const int run = 2 * kg + half;
  const int nrow = wn * 32 + l32;
  const uint8_t *xrd[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) xrd[j] = smem + l32 * 128 + (((2 * run + j) ^ ((l32 >> 1) & 7)) << 4);
  const uint8_t *wrd = smem + NST * G::XB + nrow * G::RB;
  const uint8_t *ard = smem + G::AUX0 + nrow * (4 * ndw);
  // word of a row's first group within its dword
  const int pars = ((bn0 + nrow) * ng + (int)lead[0]) & 1;
  const int parb = ALN ? pars : ((bn0 + nrow) * ng + (int)lead[1]) & 1;
  const int sh = BITS == 5 ? 16 * (run & 1) : 0;

  f32x16 acc[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) acc[i] = f32x16{};

  struct Raw {
    QRun<BITS> c;
    uint32_t s, b;
  };
  const int fp16 = p.fp16;
  auto aux = [&](uint32_t v) __attribute__((always_inline)) {
    if constexpr (ALN) return FP16 ? f16_to_f32(v) : bf16_to_f32(v);
    else return aux_to_f32_sel(v, fp16);
  };
  // The next step's scale / bias words: GS64: two bytes on per step, and at a
  // chunk's first step to the other buffer and the word its first group
  // starts at. Other sizes (32-code groups: two per step; the rest at most
  // one): where the group of the runs' half of the step is, counted from the
  // chunk's first.
  const int gse = GS64 || g32 ? 64 : gs, ginc = g32 ? 2 : 1;
  const int ablk = GS64 ? 0 : 32 * kg;
  int rt = 0;  // the next step
  int cgr = GS64 ? kb >> 6 : kb / gs;         // first group of the next step
  int rgr = GS64 ? cgr : (kb + ablk) / gs;    // and of its runs
  int crem = GS64 || g32 ? 0 : kb % gs, rrem = GS64 || g32 ? 0 : (kb + ablk) % gs;
  int cg0 = cgr;
  auto read_raw = [&](int wo, Raw &r) __attribute__((always_inline)) {
    const int c = rt / CS;
    if (rt == c * CS) cg0 = cgr;
    const uint8_t *ap = ard + ((c & 1) * G::AB + 2 * (rgr - cg0));
    const uint8_t *as = ap + 2 * ((pars + cg0) & 1), *ab = ALN ? as : ap + 2 * ((parb + cg0) & 1);
    r.c.read(wrd + wo, l32, run);
    r.s = *reinterpret_cast<const uint16_t *>(as);
    r.b = *reinterpret_cast<const uint16_t *>(ab + kTN * 4 * ndw);
    ++rt;
    if constexpr (GS64) {
      ++cgr;
      ++rgr;
    } else {
      crem += 64;
      rrem += 64;
      const bool n0 = crem >= gse, n1 = rrem >= gse;
      cgr += n0 ? ginc : 0;
      rgr += n1 ? ginc : 0;
      crem -= n0 ? gse : 0;
      rrem -= n1 ? gse : 0;
    }
  };
  // Pipeline. Step t's iteration waits for its own copies of step t + 1 (those
  // of the NST - 3 steps after it may be in flight) and for its LDS reads but
  // the MI of the next x operands, meets the barrier (step
  // t + 1 is then readable, and nobody reads x of step t - 1 or codes of step t
  // any more) and, between its MFMAs, issues the copies of step t + NST - 1; a
  // chunk's first step also copies the next chunk's scale / bias words. While
  // the MFMAs of one k slice run, the next slice's weights are formed and each
  // x operand is read again, for the next slice, as soon as its MFMA has taken
  // it: across the step's end too. The order is fixed by scheduling barriers:
  // copies issued together at the step's start hold the waves at the CU's
  // one address path (40 KB take about 640 cycles) before their first MFMA.
  aux_chunk(0);
  for (int t = 0; t < NST - 1 && t < nst; ++t) {
#pragma unroll
    for (int k = 0; k < G::L; ++k) copy(k);
    next();
  }
  q_wait_steps<G::L, NST - 2>(min(NST - 2, nst - 1));
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  Raw raw;
  bf16x8 xa[MI];
  uint32_t wf[2][4];
  read_raw(0, raw);
  __builtin_amdgcn_sched_barrier(0);  // ahead of x's reads: the wait below counts those alone
#pragma unroll
  for (int i = 0; i < MI; ++i) xa[i] = *reinterpret_cast<const bf16x8 *>(xrd[0] + 4096 * i);
  {
    uint32_t tw[3];
    raw.c.split(0, sh, tw);
#pragma unroll
    for (int i = 0; i < 4; ++i) wf[0][i] = QRun<BITS>::pair(tw, 0, i, aux(raw.s), aux(raw.b));
  }
  int so = 0, wo = 0, cs = 0;  // stages of step t; t % CS
  auto step = [&](auto copies, int t) __attribute__((always_inline)) {
    constexpr bool COPY = decltype(copies)::value;
    cs = cs == CS - 1 ? 0 : cs + 1;
    const int sn = so == (NST - 1) * G::XB ? 0 : so + G::XB;
    wo = wo == (G::NWS - 1) * G::WB ? 0 : wo + G::WB;
    __builtin_amdgcn_sched_barrier(0);
    // (past the last step: a stage of older data, read and not used)
    Raw nraw;
    read_raw(wo, nraw);
    int k = 0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (COPY && j == 1 && cs == 1) aux_chunk(t / CS + 1);
      const Raw &r = j == 0 ? raw : nraw;
      const uint8_t *xp = j == 0 ? xrd[1] + so : xrd[0] + sn;
      const bf16x8 wv = __builtin_bit_cast(bf16x8, make_uint4(wf[j][0], wf[j][1], wf[j][2], wf[j][3]));
      uint32_t tw[3];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, xa[i], acc[i], 0, 0, 0);
        xa[i] = *reinterpret_cast<const bf16x8 *>(xp + 4096 * i);
        // the last slice's codes come from LDS at the step's start: not first thing
        constexpr int P0 = MI > 4 ? MI - 4 : 0;
        if (i == P0) r.c.split(j ^ 1, sh, tw);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (i == min(P0 + q, MI - 1)) wf[j ^ 1][q] = QRun<BITS>::pair(tw, j ^ 1, q, aux(r.s), aux(r.b));
        if constexpr (COPY) {
#pragma unroll
          for (int c = 0; c < G::L; ++c)
            if (c >= k && c < ((j * MI + i + 1) * G::L) / (2 * MI)) copy(c);
          k = ((j * MI + i + 1) * G::L) / (2 * MI);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (COPY) next();
    raw = nraw;
    so = sn;
  };
  int t = 0;
  for (; t + NST - 1 < nst; ++t) {
    __builtin_amdgcn_sched_barrier(0);
    if ((unsigned)(cs - 1) < (unsigned)(NST - 3)) q_wait<(NST - 3) * G::L + G::NA>();
    else q_wait<(NST - 3) * G::L>();
    q_wait_lds<MI>();
    __builtin_amdgcn_s_barrier();
    step(std::true_type{}, t);
  }
  for (; t < nst; ++t) {
    __builtin_amdgcn_sched_barrier(0);
    q_wait<0>();
    q_wait_lds<MI>();
    __builtin_amdgcn_s_barrier();
    step(std::false_type{}, t);
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- sums of the two waves of a tile, added in k order, and stores ----
  // Element e of a 32 x 32 tile in lane l: column (m) l % 32, row (n)
  // 8 (e / 4) + 4 (l / 32) + e % 4. A wave turns its tile through LDS, so that a
  // store instruction writes whole runs of 64 (bf16) or 128 bytes of y's rows;
  // straight from the sums it writes 16 or 32 bytes in each of 32 rows. Nothing
  // overlaps a block's stores (16384 columns, M 2048, 8-bit, us, without sums and
  // stores / straight / turned: K 512 38.8 / 64.1 / 56.6, K 2048 131.8 / 155.0 /
  // 147.9; f32 partial sums the same either way).
  // Row tile i is summed and stored by k-group i % 2.
  const bool split = slot >= 0;
  float *part = split ? g_qmm_part + (size_t)slot * kQSlotFloats + (size_t)z * p.M * p.part_N + mat.col0
                      : nullptr;
  float *const flat = reinterpret_cast<float *>(smem + 32768 + wave * (32 * 33 * 4));
  auto turned = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  };
  auto store = [&](int i, const f32x16 &v) {
    const int nw = bn0 + wn * 32;
    if (split || (p.vec && !p.y_bf16)) {
      // 16-byte granule c of row r at c ^ (r & 7) of its 128 bytes
      float4 *const t = reinterpret_cast<float4 *>(flat);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        t[8 * l32 + ((2 * q + half) ^ (l32 & 7))] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
      turned();
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = 8 * q + (lane >> 3), c = lane & 7;
        const int m = bm0 + 32 * i + r, n = nw + 4 * c;
        const float4 f = t[8 * r + (c ^ (r & 7))];
        if (m >= p.M) continue;
        float *dst = split ? part + (size_t)m * p.part_N + n
                           : reinterpret_cast<float *>(mat.y) + (size_t)m * mat.y_stride + n;
        if (n + 4 <= (split ? (N + 3) & ~3 : N)) {
          *reinterpret_cast<float4 *>(dst) = f;
        } else {
          const float fe[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < N) dst[e] = fe[e];
        }
      }
    } else if (p.vec) {
      // 16-byte granule c of row r at c ^ ((r >> 2) & 3) of its 64 bytes
      typedef __bf16 b4 __attribute__((ext_vector_type(4)));
      typedef __bf16 b8 __attribute__((ext_vector_type(8)));
#pragma unroll
      for (int q = 0; q < 4; ++q)
        reinterpret_cast<b4 *>(flat)[8 * l32 + 2 * (q ^ ((l32 >> 2) & 3)) + half] =
            b4{(__bf16)v[4 * q], (__bf16)v[4 * q + 1], (__bf16)v[4 * q + 2], (__bf16)v[4 * q + 3]};
      turned();
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int r = 16 * q + (lane >> 2), c = lane & 3;
        const int m = bm0 + 32 * i + r, n = nw + 8 * c;
        const b8 f = reinterpret_cast<const b8 *>(flat)[4 * r + (c ^ ((r >> 2) & 3))];
        if (m >= p.M) continue;
        __bf16 *dst = reinterpret_cast<__bf16 *>(mat.y) + (size_t)m * mat.y_stride + n;
        if (n + 8 <= N) {
          *reinterpret_cast<b8 *>(dst) = f;
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (n + e < N) dst[e] = f[e];
        }
      }
    } else {
      // rows off 16 bytes: element stores of 32 consecutive columns
#pragma unroll
      for (int e = 0; e < 16; ++e) flat[l32 * 33 + 8 * (e / 4) + 4 * half + e % 4] = v[e];
      turned();
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = 2 * e + half, mm = bm0 + 32 * i + row, n = nw + l32;
        const float f = flat[row * 33 + l32];
        if (mm < p.M && n < N) {
          if (p.y_bf16) reinterpret_cast<__bf16 *>(mat.y)[(size_t)mm * mat.y_stride + n] = (__bf16)f;
          else reinterpret_cast<float *>(mat.y)[(size_t)mm * mat.y_stride + n] = f;
        }
      }
    }
  };
  // a round: the tiles 2 r and 2 r + 1; each wave hands over the one it does not own
  float4 *const mine = reinterpret_cast<float4 *>(smem + wave * 4096) + lane;
  const float4 *const other = reinterpret_cast<const float4 *>(smem + (wave ^ 4) * 4096) + lane;
#pragma unroll
  for (int r = 0; r < (MI + 1) / 2; ++r) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();  // the stages (or the last round's sums) are read
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (2 * r + q < MI && kg != q) {
        const f32x16 &v = acc[2 * r + q < MI ? 2 * r + q : 0];
#pragma unroll
        for (int c = 0; c < 4; ++c) mine[64 * c] = make_float4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (2 * r + q < MI && kg == q) {
        f32x16 v = acc[2 * r + q < MI ? 2 * r + q : 0];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float4 f = other[64 * c];
          v[4 * c] += f.x;
          v[4 * c + 1] += f.y;
          v[4 * c + 2] += f.z;
          v[4 * c + 3] += f.w;
        }
        store(2 * r + q, v);
      }
    }
  }
}

// sums the KS partial slices of a split product in k order (z = 0, 1, ...):
// all KS loads of a thread are issued before the first add. A thread takes 4
// consecutive columns of one row with 16-byte loads (every matrix's first
// column and the rows are multiples of 4 columns: the 4 never cross a matrix
// or a row, and only a matrix's last may lie past its end); the y store is
// then one 8- or 16-byte store when y rows are 16-byte aligned.
template <int KS>
__global__ __launch_bounds__(256) void qmm_reduce_multi_kernel(QmmMulti p, int slot) {
  typedef float fv __attribute__((ext_vector_type(4)));
  const float *part = g_qmm_part + (size_t)slot * kQSlotFloats;
  const size_t MN = (size_t)p.M * p.part_N, nv = MN / 4;
  for (size_t v = (size_t)blockIdx.x * 256 + threadIdx.x; v < nv; v += (size_t)gridDim.x * 256) {
    const size_t i = v * 4;
    fv t[KS];
#pragma unroll
    for (int z = 0; z < KS; ++z) t[z] = __builtin_nontemporal_load(reinterpret_cast<const fv *>(part + z * MN + i));
    fv s = t[0];
#pragma unroll
    for (int z = 1; z < KS; ++z) s += t[z];  // in k order
    const int m = (int)(i / p.part_N), c = (int)(i % p.part_N);
    int mi = 0;
#pragma unroll
    for (int u = 1; u < kQMultiMax; ++u) mi = u < p.n && c >= p.m[u].col0 ? u : mi;
    const QmmMat &q = p.m[mi];
    const int n = c - q.col0;
    const size_t o = (size_t)m * q.y_stride + n;
    const bool vec = p.vec && n + 4 <= q.N;
    if (p.y_bf16) {
      __bf16 *y = reinterpret_cast<__bf16 *>(q.y) + o;
      if (vec) {
        typedef __bf16 b4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<b4 *>(y) = b4{(__bf16)s[0], (__bf16)s[1], (__bf16)s[2], (__bf16)s[3]};
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < q.N) y[e] = (__bf16)s[e];
    } else {
      float *y = reinterpret_cast<float *>(q.y) + o;
      if (vec) {
        *reinterpret_cast<fv *>(y) = s;
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < q.N) y[e] = s[e];
    }
  }
}

static void launch_qmm_reduce_multi(const QmmMulti &p, int slot, int KS, hipStream_t st) {
  const size_t nv = (size_t)p.M * p.part_N / 4;
  const dim3 grid((unsigned)std::min<size_t>((nv + 255) / 256, 4096));
  switch (KS) {
#define LH_QRED(k) \
  case k: hipLaunchKernelGGL((qmm_reduce_multi_kernel<k>), grid, dim3(256), 0, st, p, slot); break;
    LH_QRED(2) LH_QRED(3) LH_QRED(4) LH_QRED(5) LH_QRED(6) LH_QRED(7) LH_QRED(8) LH_QRED(9)
    LH_QRED(10) LH_QRED(11) LH_QRED(12) LH_QRED(13) LH_QRED(14) LH_QRED(15) LH_QRED(16)
#undef LH_QRED
    default: break;
  }
}

bool affine_qmm_supported(const DevMat &m) {
  if (!(m.bits == 4 || m.bits == 5 || m.bits == 6 || m.bits == 8)) return false;
  if (m.I <= 0 || m.I % kTile != 0 || m.O <= 0) return false;
  if (m.gs <= 0 || m.gs % 32 != 0 || m.I % m.gs != 0) return false;
  if (m.row_bytes != (long long)m.I * m.bits / 8) return false;
  if ((m.row_bytes & 3) != 0 || (reinterpret_cast<uintptr_t>(m.w) & 3) != 0) return false;
  return true;
}

// Whether the tile kernel takes the product: every matrix supported, the same
// K / bits / group size / aux type and per-lane offsets within a tile that fit
// 32 bits; kQAligned: with 16-byte copies of the packed rows (5-bit rows: 4-byte
// ones) and sidecars on whole dwords, kQDword: by dwords.
enum { kQNone, kQAligned, kQDword };
static int qmm_tile_form(const DevMat *ms, int n, int x_stride) {
  if (n < 1 || n > kQMultiMax || x_stride > (1 << 22)) return kQNone;
  int form = kQAligned;
  for (int i = 0; i < n; ++i) {
    const DevMat &m = ms[i];
    if (!affine_qmm_supported(m)) return kQNone;
    if (m.I != ms[0].I || m.bits != ms[0].bits || m.gs != ms[0].gs || m.fp16 != ms[0].fp16) return kQNone;
    if (m.row_bytes > (1 << 23) || (long long)m.O * m.ng > 0x7fff0000LL / 2) return kQNone;
    if ((long long)m.O * m.ng < 2) return kQNone;
    const uintptr_t aux = reinterpret_cast<uintptr_t>(m.sc) | reinterpret_cast<uintptr_t>(m.bi);
    if ((aux & 1) != 0) return kQNone;
    if ((m.bits != 5 && (reinterpret_cast<uintptr_t>(m.w) & 15) != 0) || (aux & 3) != 0) form = kQDword;
  }
  return form;
}

// Tile rows and K split of a product: the least estimated time in us: a 64-k
// step of a block, whose weights are formed whatever its rows, or the time its
// codes take to arrive; a block's pipeline fill and sum exchange; and for a split
// its partial sums written and read back and one more launch; one block per CU
// (of 32-row tiles it holds two, which take about half again as long as one:
// nearer to one round than to the two counted). The fitted constants rank the
// choices rather than predict the time: over 3,382 measured choices of 273 shapes
// (24 to 2200 rows, 1000 to 28672 columns) the estimate is 11 % off on average
// and 7 % low, and the choice costs 0.3 % over the best one measured, 12 % at most.
struct QmmPlan {
  int bm, split;
};
static QmmPlan qmm_plan(int M, int tiles, int cols, int ksteps, int bits, int max_bm) {
  static const int kBm[5] = {32, 64, 128, 192, 256};
  QmmPlan best{256, 1};
  float tb = 1e30f;
  for (int c = 0; c < 5; ++c) {
    const int bm = kBm[c], mt = (M + bm - 1) / bm;
    if (bm > max_bm) break;
    const float step = std::max(0.39f + 0.32f * bm / 256, 0.33f * bits / 8);
    const float fixed = 1.8f + 5.0f * bm / 256;
    for (int sp = 1; sp <= 16; ++sp) {
      const int ks = (ksteps + sp - 1) / sp;
      if ((ksteps + ks - 1) / ks != sp) continue;
      if (sp > 1 && (ks < 3 || (size_t)sp * M * cols > kQSlotFloats)) continue;
      const int rounds = (int)(((long long)mt * tiles * sp + 255) / 256);
      float t = rounds * (ks * step + fixed);
      if (sp > 1) t += 4.4f + (float)sp * M * cols * 8 / 5.5e6f;
      if (t < tb) {
        tb = t;
        best = QmmPlan{bm, sp};
      }
    }
  }
  return best;
}

// the route of a product: kernel (kQNone: affine_qmm_kernel, one launch per
// matrix, whose K split launch_affine_qmm chooses), tile rows and k ranges
struct QmmRoute {
  int form, bm, split;
};
static QmmRoute qmm_route(const DevMat *ms, int n, int x_stride, int M) {
  // Products this small are launch and latency: the tile kernel's prologue (its
  // rings, three or more steps ahead) and sum exchange cost more than they
  // save. us, 64 x 64 kernel / tile kernel, 4-bit: 17 x 512 (M x N), K 2048:
  // 8.0 / 9.0; 17 x 4096, K 2048: 10.6 / 11.1; 64 x 1024, K 2048: 10.3 / 10.3;
  // 64 x 2048, K 2048: 13.6 / 11.9; 17 x 1024, K 9728: 13.2 / 13.7;
  // 17 x 2048, K 9728: 16.2 / 14.4.
  const bool small = n == 1 && (long long)M * ms[0].O <= (M <= 24 ? 81920 : 65536) &&
                     (long long)ms[0].O * ms[0].I <= (10 << 20);
  // By dwords above 64 rows only: up to there the 64 x 64 kernel forms every
  // weight once as well. 4096 x 4096, 8-bit, 64 x 64 kernel / tile kernel by
  // dwords, us: sidecars off 4 bytes, M 100: 29.5 / 20.8, 512: 81.9 / 38.7,
  // 2048: 286 / 74; 4-bit weights off 16 bytes: 30.2 / 22.5, 79.8 / 36.6, 281 / 73.
  const int form = small ? kQNone : qmm_tile_form(ms, n, x_stride);
  if (form == kQNone || (form == kQDword && M <= kTile)) return QmmRoute{kQNone, 0, 0};
  int tiles = 0, cols = 0;
  for (int i = 0; i < n; ++i) {
    tiles += (ms[i].O + kTN - 1) / kTN;
    cols += (ms[i].O + 3) & ~3;
  }
  // (256 rows of 8-bit dwords leave no room for chunks of 32-code groups that
  // start inside a dword)
  const int max_bm = form == kQDword && ms[0].bits == 8 && ms[0].gs != 64 ? 192 : 256;
  const QmmPlan plan = qmm_plan(M, tiles, cols, ms[0].I / 64, ms[0].bits, max_bm);
  return QmmRoute{form, plan.bm, plan.split};
}

bool affine_qmm_route(const DevMat *ms, int n, int x_stride, int M, int (&route)[3]) {
  for (int i = 0; i < n; ++i)
    if (!affine_qmm_supported(ms[i])) return false;
  const QmmRoute r = qmm_route(ms, n, x_stride, M);
  route[0] = r.form;
  route[1] = r.bm;
  route[2] = r.split;
  return true;
}

template <int BITS, bool GS64, bool FP16, bool ALN>
static hipError_t launch_qmm_tile_bits(const QmmMulti &p, int bm, int mt, int tiles, int split, int ksteps,
                                       int slot, hipStream_t st) {
  const dim3 grid((mt * tiles * split + 7) / 8 * 8), block(512);
  switch (bm) {
#define LH_QTILE(MI)                                                                                           \
  case 32 * MI: hipLaunchKernelGGL((affine_qmm_tile_kernel<BITS, MI, GS64, FP16, ALN>), grid, block, 0, st, p, \
                                   mt, tiles, ksteps, slot); break;
    LH_QTILE(1) LH_QTILE(2) LH_QTILE(4) LH_QTILE(6)
    case 256:
      if constexpr (ALN || GS64 || BITS != 8) {
        hipLaunchKernelGGL((affine_qmm_tile_kernel<BITS, 8, GS64, FP16, ALN>), grid, block, 0, st, p, mt, tiles,
                           ksteps, slot);
        break;
      }
      return hipErrorInvalidValue;
#undef LH_QTILE
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

static hipError_t launch_qmm_tile(const DevMat *ms, int n, const uint16_t *x, int x_stride, int M,
                                  void *const *ys, const int *y_strides, int y_bf16, const QmmRoute &route,
                                  hipStream_t st) {
  QmmMulti p;
  p.x = x;
  p.n = n;
  p.M = M;
  p.K = ms[0].I;
  p.gs = ms[0].gs;
  p.fp16 = ms[0].fp16;
  p.x_stride = x_stride;
  p.y_bf16 = y_bf16;
  int tiles = 0, cols = 0;
  for (int i = 0; i < kQMultiMax; ++i) {
    if (i < n) {
      p.m[i] = QmmMat{ms[i].w, ms[i].sc, ms[i].bi, ys[i], ms[i].row_bytes, ms[i].O, ms[i].ng,
                      y_strides[i], cols};
      p.tile_start[i] = tiles;
      tiles += (ms[i].O + kTN - 1) / kTN;
      cols += (ms[i].O + 3) & ~3;  // 16-byte partial stores
    } else {
      p.m[i] = p.m[0];
      p.tile_start[i] = tiles;
    }
  }
  p.tile_start[kQMultiMax] = tiles;
  p.part_N = cols;
  bool yv = true;
  for (int i = 0; i < n; ++i) {
    const int es = y_bf16 ? 2 : 4;
    yv = yv && (reinterpret_cast<uintptr_t>(ys[i]) & 15) == 0 && ((long long)y_strides[i] * es) % 16 == 0;
  }
  p.vec = yv ? 1 : 0;
  const int ksteps_all = p.K / 64;
  const int bm = route.bm, split = route.split, mt = (M + bm - 1) / bm;
  const int ksteps = (ksteps_all + split - 1) / split;
  SlotRing::Lease lease;
  if (split > 1) {
    const hipError_t le = g_qmm_slots.take(st, lease);
    if (le != hipSuccess) return le;
  }
  const int slot = split > 1 ? lease.slot() : -1;
  hipError_t e;
  switch (ms[0].bits) {
#define LH_QFORM(B, G64)                                                                                         \
  (route.form == kQDword ? launch_qmm_tile_bits<B, G64, false, false>(p, bm, mt, tiles, split, ksteps, slot, st) \
   : p.fp16              ? launch_qmm_tile_bits<B, G64, true, true>(p, bm, mt, tiles, split, ksteps, slot, st)   \
                         : launch_qmm_tile_bits<B, G64, false, true>(p, bm, mt, tiles, split, ksteps, slot, st))
#define LH_QBITS(B) \
  case B: e = p.gs == 64 ? LH_QFORM(B, true) : LH_QFORM(B, false); break;
    LH_QBITS(4) LH_QBITS(5) LH_QBITS(6) LH_QBITS(8)
#undef LH_QBITS
#undef LH_QFORM
    default: return hipErrorInvalidValue;
  }
  if (e != hipSuccess || split == 1) return e;
  launch_qmm_reduce_multi(p, slot, split, st);
  e = hipGetLastError();
  const hipError_t le = lease.done();
  return e != hipSuccess ? e : le;
}

hipError_t launch_affine_qmm_multi(const DevMat *ms, int n, const uint16_t *x, int x_stride, int M,
                                   void *const *ys, int y_bf16, hipStream_t st) {
  if (n < 1 || n > kQMultiMax || M <= 0) return hipErrorInvalidValue;
  if ((reinterpret_cast<uintptr_t>(x) & 15) != 0 || (x_stride & 7) != 0) return hipErrorInvalidValue;
  int strides[kQMultiMax];
  for (int i = 0; i < n; ++i) strides[i] = ms[i].O;
  if (n > 1) {
    const QmmRoute r = qmm_route(ms, n, x_stride, M);
    if (r.form != kQNone) return launch_qmm_tile(ms, n, x, x_stride, M, ys, strides, y_bf16, r, st);
  }
  for (int i = 0; i < n; ++i) {
    const hipError_t e = launch_affine_qmm(ms[i], x, x_stride, M, ys[i], ms[i].O, y_bf16, st);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_affine_qmm(const DevMat &m, const uint16_t *x, int x_stride, int M, void *y,
                             int y_stride, int y_bf16, hipStream_t st) {
  if (!affine_qmm_supported(m) || M <= 0) return hipErrorInvalidValue;
  if ((reinterpret_cast<uintptr_t>(x) & 15) != 0 || (x_stride & 7) != 0) return hipErrorInvalidValue;
  const QmmRoute r = qmm_route(&m, 1, x_stride, M);
  if (r.form != kQNone) {
    void *ys[1] = {y};
    const int strides[1] = {y_stride};
    return launch_qmm_tile(&m, 1, x, x_stride, M, ys, strides, y_bf16, r, st);
  }
  GemmParams p;
  p.w = m.w;
  p.sc = m.sc;
  p.bi = m.bi;
  p.x = x;
  p.y = y;
  p.row_bytes = m.row_bytes;
  p.M = M;
  p.N = m.O;
  p.K = m.I;
  p.ng = m.ng;
  p.gs = m.gs;
  p.fp16 = m.fp16;
  p.x_stride = x_stride;
  p.y_stride = y_stride;
  p.y_bf16 = y_bf16;
  // 64 x 64 tiles; grids short of about two blocks per CU split K as well (at
  // most 16 ways, partials within one slot)
  const int ksteps_all = m.I / 64;
  const int tiles = ((M + kTile - 1) / kTile) * ((m.O + kTile - 1) / kTile);
  int split = 1;
  while (split < 16 && tiles * split < kQTargetBlocks && 2 * split <= ksteps_all &&
         (size_t)(2 * split) * M * m.O <= kQSlotFloats)
    split *= 2;
  const int ksteps = (ksteps_all + split - 1) / split;
  split = (ksteps_all + ksteps - 1) / ksteps;
  SlotRing::Lease lease;
  if (split > 1) {
    const hipError_t le = g_qmm_slots.take(st, lease);
    if (le != hipSuccess) return le;
  }
  const int slot = split > 1 ? lease.slot() : -1;
  const dim3 grid((M + kTile - 1) / kTile, (m.O + kTile - 1) / kTile, split);
  switch (m.bits) {
    case 4: hipLaunchKernelGGL(affine_qmm_kernel<4>, grid, dim3(256), 0, st, p, ksteps, slot); break;
    case 5: hipLaunchKernelGGL(affine_qmm_kernel<5>, grid, dim3(256), 0, st, p, ksteps, slot); break;
    case 6: hipLaunchKernelGGL(affine_qmm_kernel<6>, grid, dim3(256), 0, st, p, ksteps, slot); break;
    case 8: hipLaunchKernelGGL(affine_qmm_kernel<8>, grid, dim3(256), 0, st, p, ksteps, slot); break;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || split == 1) return e;
  if ((m.O & 3) == 0)
    launch_qmm_reduce<4>(p, slot, split, st);
  else
    launch_qmm_reduce<1>(p, slot, split, st);
  e = hipGetLastError();
  const hipError_t le = lease.done();
  return e != hipSuccess ? e : le;
}

}  // namespace lh
