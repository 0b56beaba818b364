// bgemm_tile.h - device pieces shared by the BF16 GEMM kernels (bgemm.hip, bgemm_flex.hip): the
// LDS layout of an operand's k-tile, the workgroup order and the epilogues.
#pragma once

#include "hk_device.h"
#include "hk_host.h"

namespace hk {
namespace gemm {

constexpr int BK = 64;  // k-tile

typedef short bf16x8_t __attribute__((ext_vector_type(8)));
typedef short bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
#define HK_LDS __attribute__((address_space(3)))

// 16-byte global -> LDS copy of one lane (global_load_lds_dwordx4): the wave's 64 lanes write
// 1 KiB of LDS at m0 + 16 * lane. Written as inline asm on purpose: for the builtin, the
// compiler assumes every later LDS read may alias the copy and waits for ALL of them to land
// before any LDS read, which would serialise the load pipeline against the MFMA loop. Here the
// kernel waits for the copies itself (vmcnt) before the barrier that publishes a stage.
// Address = sbase (wave-uniform 64-bit, SGPRs) + voff (per-lane byte offset).
__device__ __forceinline__ void copy16_to_lds(const void* sbase, int voff, unsigned lds_addr) {
  // m0 (the LDS destination) is an input operand, so the compiler knows the asm sets it. Its
  // hazard checks do not see inside the asm, so the asm supplies the wait states itself: an
  // SALU write of m0 needs 1 before an LDS-DMA load, and an SGPR of sbase written by a VALU
  // (v_readlane, when the compiler reloads a spilled SGPR) needs 5 before a VMEM read of it.
  asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase),
               "{m0}"(lds_addr));
}

// One operand of a k-tile in LDS: 256 rows of M (or N) by BK = 64 k, bf16, 32 KiB.
//
// gfx950's LDS has 64 banks of 4 bytes: a ds_read_b128 is served 16 lanes (256 bytes) per
// cycle and a ds_read_b64(_tr) 32 lanes per cycle, so each such lane group must cover all 64
// banks once (a 2-way conflict halves the read rate; measured 134 against 222 B/clk/CU).
//
// K-major operands (element (row, k) at base[row * ld + k]) are stored [row][64 k]: 128-byte
// rows whose eight 16-byte chunks sit at chunk ^ ((row >> 1) & 7). A wave's copy instruction
// moves 8 rows (lane l: row l / 8, stored chunk l % 8, which is global chunk
// (l % 8) ^ ((row >> 1) & 7), so each row's 128 contiguous bytes are read by 8 lanes). The
// MFMA operand of a lane is 8 consecutive k of one row, one ds_read_b128; the 16 lanes of one
// read cycle take 16 consecutive rows at one logical chunk: the even rows fill one 128-byte
// bank half at 8 distinct chunk positions and the odd rows the other.
//
// M/N-major operands (element at base[k * ld + row]) are stored as in HBM, [64 k][256 rows]:
// 512-byte k-rows (256 bytes for a 128-wide B tile) whose 16-byte chunk c sits at
// c ^ (2 * (krow & 3)) ^ (8 * ((c >> 1) & 1)). Both row pitches are whole multiples of the 64
// banks, so a chunk's banks depend on its stored position mod 16 alone and the placement below
// holds for both. A copy instruction moves 2 k-rows (4 for 256-byte rows; 32 or 16 lanes read
// one contiguous row segment). The
// MFMA operand (8 consecutive k of one row/column) is gathered with two ds_read_b64_tr_b16:
// within each 16-lane group, lane j reads 4 bf16 of k-row kb + j / 4 at columns
// c0 + 4 (j % 4) and the hardware transposes the 16 x 4 block so lane i receives column
// c0 + i, k = kb .. kb + 3. One group covers 4 k-rows x 32 bytes, which the (krow & 3) term
// spreads over 32 banks; the two groups of a read cycle sit 16 columns (2 chunks) apart and
// the (c >> 1) term places them in opposite bank halves.
template <bool KMAJOR, int ROWS = 256>
struct TileOperand {
  // M/N-major: a copy instruction (1 KiB) covers kRowsPerCopy k-rows of ROWS * 2 bytes.
  static constexpr int kKRowBytes = ROWS * 2;
  static constexpr int kRowsPerCopy = 1024 / kKRowBytes;
  static constexpr int kLanesPerRow = 64 / kRowsPerCopy;
  // M/N-major: stored position of logical 16-byte chunk c of k-row krow, and its inverse.
  // 64-wide tiles have 128-byte k-rows, half the banks: the 4 k-rows and 4 chunks of one read
  // cycle cover the banks once when k-rows 2 apart use opposite 64-byte halves.
  __device__ static int stored_chunk(int c, int krow) {
    if (ROWS == 64) return c ^ (4 * ((krow >> 1) & 1));
    return c ^ (2 * (krow & 3)) ^ (8 * ((c >> 1) & 1));
  }
  __device__ static int logical_chunk(int p, int krow) {
    if (ROWS == 64) return p ^ (4 * ((krow >> 1) & 1));
    return p ^ (8 * (((p >> 1) ^ krow) & 1)) ^ (2 * (krow & 3));
  }
  // Byte offset of lane `lane`'s 16 bytes of copy instruction ii (0 .. 31) from the tile's
  // global base at k = 0, and the (row, k) of its first element.
  __device__ static void source(int ii, int lane, int& row, int& k) {
    if (KMAJOR) {
      row = ii * 8 + (lane >> 3);
      k = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
    } else {
      k = ii * kRowsPerCopy + lane / kLanesPerRow;
      row = logical_chunk(lane % kLanesPerRow, k) * 8;
    }
  }
  __device__ static int64_t byte_offset(int row, int k, int64_t ld) {
    return KMAJOR ? 2 * (static_cast<int64_t>(row) * ld + k)
                  : 2 * (static_cast<int64_t>(k) * ld + row);
  }
  // Global step of one k-tile (elements).
  __device__ static int64_t ktile_step(int64_t ld) { return KMAJOR ? BK : BK * ld; }
  // LDS byte offset of the MFMA operand of MFMA block b (32 rows at wave offset wo),
  // 16-deep k step s; `half` selects the second 4-k read of an M/N-major operand.
  __device__ static int frag(int wo, int b, int s, int half, int lane) {
    if (KMAJOR) {
      const int row = wo + b * 32 + (lane & 31);
      const int c = 2 * s + (lane >> 5);
      return row * 128 + ((c ^ ((row >> 1) & 7)) * 16);
    } else {
      const int g = lane >> 4, j = lane & 15;
      const int col = wo + b * 32 + 16 * (g & 1) + 4 * (j & 3);
      const int krow = 16 * s + 8 * (g >> 1) + (j >> 2) + 4 * half;
      return krow * kKRowBytes + stored_chunk(col >> 3, krow) * 16 + (col & 7) * 2;
    }
  }
  __device__ static bf16x8_t read(const unsigned char HK_LDS* st, int wo, int b, int s,
                                  int lane) {
    if (KMAJOR) {
      return *reinterpret_cast<const bf16x8_t HK_LDS*>(st + frag(wo, b, s, 0, lane));
    } else {
      const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (bf16x4_t HK_LDS*)(st + frag(wo, b, s, 0, lane)));
      const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (bf16x4_t HK_LDS*)(st + frag(wo, b, s, 1, lane)));
      return bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
  }
};

// A grid of several matrices (x: the tiles of one, z: matrices x k splits): workgroup (t, z) takes
// the item that gives each XCD a run of consecutive ones, so that the tiles of a small matrix meet in
// one L2 instead of each being read by every XCD (MI355X, TN: 520 x 168 x 2264 in 32 batches 77 -> 31 us,
// 88 x 336 x 3928 in 64 batches 130 -> 49). The hardware deals workgroups to the 8 XCDs round-robin in
// linear order. tiles x nz < 2^31.
__device__ __forceinline__ void matrix_order(int tiles, int nz, int& t, int& z) {
  const unsigned total = static_cast<unsigned>(tiles) * nz;
  const unsigned id = static_cast<unsigned>(z) * tiles + t, xcd = id & 7;
  const unsigned item = xcd * (total >> 3) + min(xcd, total & 7) + (id >> 3);
  z = static_cast<int>(item / tiles);
  t = static_cast<int>(item - static_cast<unsigned>(z) * tiles);
}

// Linear tile id t -> (tile_m, tile_n): consecutive ids to one XCD (unless the caller has ordered
// them), grouped 8 tile-rows. The hardware deals workgroups to the 8 XCDs round-robin, so t % 8 is
// the XCD when t is a workgroup id or one offset by a multiple of 8.
__device__ __forceinline__ void tile_coords(int t, int tiles_m, int tiles_n, int& tm, int& tn,
                                            bool ordered = false) {
  const int total = tiles_m * tiles_n;
  if (!ordered && (total & 7) == 0) t = (t & 7) * (total >> 3) + (t >> 3);
  constexpr int G = 8;
  const int per_group = G * tiles_n;
  const int group = t / per_group;
  const int first_m = group * G;
  const int gsz = min(tiles_m - first_m, G);
  const int in_group = t - group * per_group;
  tm = first_m + in_group % gsz;
  tn = in_group / gsz;
}

// Output transform: C = alpha * acc + beta * C, or, with a bias (bias != NULL),
// C = alpha * acc + beta * bias and C is written without being read. The bias element of
// output (row, col) is bias[row * brow + col * bcol]: (brow, bcol) = (0, 1) for a per-column
// bias (numel N), (1, 0) per row (numel M), (0, 0) scalar (numel 1), (N, 1) full (numel M*N,
// the same for every batch).
struct Epi {
  float alpha, beta;
  const uint16_t* bias;
  int64_t brow, bcol;
  bool ragged;  // rows of C that are no whole number of aligned 16-byte vectors
};

__device__ __forceinline__ float bias_at(const Epi& ep, int row, int col) {
  return hk::bf16_to_f32(ep.bias[row * ep.brow + col * ep.bcol]);
}

// Bias element of column col of batch b for an fp32 output (hk::F32Out).
__device__ __forceinline__ float f32out_bias(const hk::F32Out& fo, int M, int N, int b, int col) {
  if (fo.bias_stride == N) return fo.bias[col];
  if (fo.bias_stride == static_cast<int64_t>(M) * N)
    return fo.bias[static_cast<int64_t>(b % M) * N + col];
  if (fo.bias_stride == 1) return fo.bias[0];
  return 0.f;
}

// Scheduling hint: NR LDS reads spread over NM MFMAs (reads first in each pair), so the
// operands of the next k step are fetched while the current one multiplies.
template <int NM, int NR, int Q = 0>
__device__ __forceinline__ void interleave_reads() {
  if constexpr (Q < NM) {
    constexpr int per = (NR + NM - 1) / NM;
    constexpr int left = NR - Q * per;
    constexpr int n = left <= 0 ? 0 : (left < per ? left : per);
    if constexpr (n > 0) __builtin_amdgcn_sched_group_barrier(0x100, n, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    interleave_reads<NM, NR, Q + 1>();
  }
}

// Hands the accumulators of a wave to `out` through LDS, one 32-row MFMA block row at a time:
// the wave stores its block row into its own fp32 staging area (32 rows, pitch kWaveN * 4 + 16
// bytes, so the 16 lanes of one 16-byte write cycle start 4 banks apart) and reads it back as 8
// consecutive columns per lane: out(row, col, a, b) gets the wave-relative row and column of
// values a[0..3], b[0..3], and kWaveN / 8 consecutive lanes hold one row segment, so the
// outputs can be written 16 (bf16) or 32 (fp32) bytes per lane in whole lines. Stored straight
// from the MFMA layout instead, every store touched 32 rows and each 128-byte line of C was
// assembled from 8 stores (bf16): 23% of the BASELINE product. The area is the wave's own, so
// it needs no barrier beyond the one that ends the main loop.
template <int kWaveN, int kBlkM, typename Out>
__device__ __forceinline__ void staged_rows(const f32x16_t (&acc)[kBlkM][kWaveN / 32],
                                            unsigned char HK_LDS* area, int lane, Out&& out) {
  constexpr int kBlkN = kWaveN / 32;
  constexpr int P = kWaveN * 4 + 16;        // staging pitch (bytes)
  constexpr int LPR = kWaveN / 8;           // lanes per row
  constexpr int RPP = 64 / LPR;             // rows per pass
  const int r = lane & 31, h = lane >> 5;
  const int rr0 = lane / LPR, cc = (lane % LPR) * 8;
#pragma unroll
  for (int i = 0; i < kBlkM; ++i) {
#pragma unroll
    for (int j = 0; j < kBlkN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4_t HK_LDS*>(area + r * P + (32 * j + 8 * q + 4 * h) * 4) =
            f32x4_t{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                    acc[i][j][4 * q + 3]};
#pragma unroll
    for (int p = 0; p < 32 / RPP; ++p) {
      const int rr = p * RPP + rr0;
      const f32x4_t a = *reinterpret_cast<const f32x4_t HK_LDS*>(area + rr * P + cc * 4);
      const f32x4_t b = *reinterpret_cast<const f32x4_t HK_LDS*>(area + rr * P + cc * 4 + 16);
      out(32 * i + rr, cc, a, b);
    }
  }
}

// The bf16 epilogue on staged rows: C = alpha * acc + beta * C (or + beta * bias) in fp32,
// one rounding to bf16 (v_cvt_pk_bf16_f32, round to nearest even), 16-byte stores. RAGGED: rows
// of C at any 2-byte address and any N; eight columns inside N are still one (unaligned) 16-byte
// access, the columns that cross N are stored one by one.
template <bool BIAS, bool RAGGED = false>
struct Bf16RowOut {
  const Epi& ep;
  uint16_t* Cb;
  int64_t ldc;
  int M, N, wrow0, wcol0;
  __device__ void operator()(int rr, int cc, const f32x4_t& a, const f32x4_t& b) const {
    const int row = wrow0 + rr, col = wcol0 + cc;
    if (row >= M || col >= N) return;  // not RAGGED: N % 8 == 0, the 8 columns are all in or out
    f32x2_t v[4] = {f32x2_t{a[0], a[1]} * ep.alpha, f32x2_t{a[2], a[3]} * ep.alpha,
                    f32x2_t{b[0], b[1]} * ep.alpha, f32x2_t{b[2], b[3]} * ep.alpha};
    uint16_t* cp = Cb + static_cast<int64_t>(row) * ldc + col;
    const int n = RAGGED ? min(8, N - col) : 8;
    if (BIAS) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c0 = RAGGED ? min(col + 2 * e, N - 1) : col + 2 * e;
        const int c1 = RAGGED ? min(col + 2 * e + 1, N - 1) : col + 2 * e + 1;
        v[e] += ep.beta * f32x2_t{bias_at(ep, row, c0), bias_at(ep, row, c1)};
      }
    } else if (ep.beta != 0.0f) {
      uint32_t o[4];
      if (n == 8) {
        if (RAGGED) {
          __builtin_memcpy(o, cp, 16);
        } else {
          const uint4 old = *reinterpret_cast<const uint4*>(cp);
          o[0] = old.x, o[1] = old.y, o[2] = old.z, o[3] = old.w;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[e] = (2 * e < n ? cp[2 * e] : 0u) |
                 (2 * e + 1 < n ? static_cast<uint32_t>(cp[2 * e + 1]) << 16 : 0u);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] += ep.beta * f32x2_t{__uint_as_float(o[e] << 16), __uint_as_float(o[e] & 0xffff0000u)};
    }
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bf16x2_t bv = __builtin_convertvector(v[e], bf16x2_t);
      __builtin_memcpy(&w[e], &bv, 4);
    }
    if (RAGGED) {
      if (n == 8) {
        __builtin_memcpy(cp, w, 16);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (e < n) cp[e] = static_cast<uint16_t>(e & 1 ? w[e >> 1] >> 16 : w[e >> 1]);
      }
      return;
    }
    // non-temporal: C is not read again by this product, and keeping it out of the caches
    // leaves them to the operands (8192^3 NN: 742 -> 714 us on MI355X). The fp32 split-K
    // partials below are read back by the finalize kernel and keep ordinary stores (with
    // non-temporal ones the 8192 x 1280 x 5120 dA product went from 130 to 149 us).
    typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
    __builtin_nontemporal_store(u32x4_t{w[0], w[1], w[2], w[3]}, reinterpret_cast<u32x4_t*>(cp));
  }
};

// Writes a wave's accumulators to C through the form the call needs.
template <int kWaveN, int kBlkM>
__device__ __forceinline__ void store_bf16(const f32x16_t (&acc)[kBlkM][kWaveN / 32],
                                           unsigned char HK_LDS* area, int lane, const Epi& ep,
                                           uint16_t* Cb, int64_t ldc, int M, int N, int wrow0,
                                           int wcol0) {
  if (ep.ragged) {
    if (ep.bias)
      staged_rows<kWaveN, kBlkM>(acc, area, lane,
                                 Bf16RowOut<true, true>{ep, Cb, ldc, M, N, wrow0, wcol0});
    else
      staged_rows<kWaveN, kBlkM>(acc, area, lane,
                                 Bf16RowOut<false, true>{ep, Cb, ldc, M, N, wrow0, wcol0});
  } else if (ep.bias) {
    staged_rows<kWaveN, kBlkM>(acc, area, lane,
                               Bf16RowOut<true>{ep, Cb, ldc, M, N, wrow0, wcol0});
  } else {
    staged_rows<kWaveN, kBlkM>(acc, area, lane,
                               Bf16RowOut<false>{ep, Cb, ldc, M, N, wrow0, wcol0});
  }
}

// fp32 output: C = alpha * acc + beta * C + bias_scale * bias (hk::F32Out), N % 8 == 0.
template <int kWaveN, int kBlkM>
__device__ __forceinline__ void store_f32(const f32x16_t (&acc)[kBlkM][kWaveN / 32],
                                          unsigned char HK_LDS* area, int lane,
                                          const hk::F32Out& fo, int batch, int M, int N, int wrow0,
                                          int wcol0) {
  float* cb = fo.C + static_cast<int64_t>(batch) * fo.sC;
  staged_rows<kWaveN, kBlkM>(acc, area, lane, [&](int rr, int cc, const f32x4_t& a, const f32x4_t& b) {
    const int row = wrow0 + rr, col = wcol0 + cc;
    if (row >= M || col >= N) return;  // N % 8 == 0
    f32x4_t* dst = reinterpret_cast<f32x4_t*>(cb + static_cast<int64_t>(row) * fo.ldc + col);
    f32x4_t v0 = fo.alpha * a, v1 = fo.alpha * b;
    if (fo.beta != 0.0f) {
      v0 += fo.beta * dst[0];
      v1 += fo.beta * dst[1];
    }
    if (fo.bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v0[e] += fo.bias_scale * f32out_bias(fo, M, N, batch, col + e);
        v1[e] += fo.bias_scale * f32out_bias(fo, M, N, batch, col + 4 + e);
      }
    }
    dst[0] = v0;
    dst[1] = v1;
  });
}

// Adds the accumulators of the T::KG k groups of a workgroup, in group order, into those of group 0,
// through LDS behind the groups' staging areas (T::kSums bytes for each further group). True for the
// waves of the other groups, which are done then.
template <class T>
__device__ __forceinline__ bool merge_groups(f32x16_t (&acc)[T::kBlkM][T::kBlkN],
                                             unsigned char HK_LDS* lds, int group, int wave,
                                             int lane) {
  unsigned char HK_LDS* sums = lds + T::kGroupWaves * T::kStaging;
  constexpr int kPerWave = T::kBlkM * T::kBlkN * 4;
  auto at = [&](int grp, int b, int q) {
    return reinterpret_cast<f32x4_t HK_LDS*>(
        sums + (grp - 1) * T::kSums + ((wave * kPerWave + b * 4 + q) * 64 + lane) * 16);
  };
  if (group > 0) {
#pragma unroll
    for (int b = 0; b < T::kBlkM * T::kBlkN; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x16_t& v = acc[b / T::kBlkN][b % T::kBlkN];
        *at(group, b, q) = f32x4_t{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
      }
  }
  __syncthreads();
  if (group > 0) return true;
#pragma unroll
  for (int grp = 1; grp < T::KG; ++grp)
#pragma unroll
    for (int b = 0; b < T::kBlkM * T::kBlkN; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4_t v = *at(grp, b, q);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[b / T::kBlkN][b % T::kBlkN][4 * q + e] += v[e];
      }
  return false;
}

// Row pitch (elements) of the fp32 split-K partials: whole 32-byte groups for any N.
__host__ __device__ __forceinline__ int part_pitch(int N) { return (N + 7) & ~7; }

// One split's fp32 sums: out = the [M][part_pitch(N)] partials of its batch.
template <int kWaveN, int kBlkM>
__device__ __forceinline__ void store_partial(const f32x16_t (&acc)[kBlkM][kWaveN / 32],
                                              unsigned char HK_LDS* area, int lane, float* out,
                                              int M, int N, int wrow0, int wcol0) {
  const int64_t pitch = part_pitch(N);
  staged_rows<kWaveN, kBlkM>(acc, area, lane, [&](int rr, int cc, const f32x4_t& a, const f32x4_t& b) {
    const int row = wrow0 + rr, col = wcol0 + cc;
    if (row >= M || col >= N) return;
    f32x4_t* dst = reinterpret_cast<f32x4_t*>(out + row * pitch + col);
    dst[0] = a;
    dst[1] = b;
  });
}

}  // namespace gemm
}  // namespace hk
