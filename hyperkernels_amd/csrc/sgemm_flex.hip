// sgemm_flex.hip - fp32 GEMM on the fp32 MFMA for rows of any length and alignment and for products
// that 256 x 256 tiles leave most CUs idle on: C = alpha * op(A) op(B) + beta * C + bias, exact
// fp32 products, fp32 accumulation in a fixed order. Contract: sgemm.hip.
//
// Design (gfx950): v_mfma_f32_32x32x2_f32 takes 64 cycles for 2 k of a 32 x 32 block, so a
// workgroup of 4 waves keeps its CU's matrix cores busy on any tile; what a tile's size decides is
// how many CUs a product covers and how often its operands are read. Tiles of 32 x 32 (the four
// waves are k groups that take alternate k-tiles, summed in group order through LDS), 64 x 64 and
// 128 x 128 (2 x 2 waves). K-tiles of 32 fp32 are loaded 16 bytes per lane at any 4-byte address
// into registers, one k-tile ahead, and written to a ring of two LDS slots; a vector that would
// cross the end of K, or of the matrix in its last k-row, is read element by element, with zeros
// past K. An output's fp32 sum is formed from KG x NA serial ones (NA accumulator sets per wave, MFMA
// steps in turn): 8, 4 and 1 for the three tiles, at no cost in time (1500 x 1500 x 772 NN 47 us with
// one set and with four, error against 64 bits 5.0e-7 and 2.5e-7; 260 x 260 x 16388 NT 110 us, 1.15e-6
// with 4 sums, 8.1e-7 with 8, as 8 k splits of the 256 x 256 tiles have). LDS holds K-major operands
// as [row][32 k] and M/N-major ones as [32 k][row], as in sgemm.hip: lane (r, h) of a wave feeds
// k = 16 h + s of each k-tile at MFMA step s.
#include <mutex>

#include "bgemm_tile.h"
#include "sgemm_flex.h"

namespace {

using namespace hk::gemm;
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes anywhere

constexpr int KT = 32;  // k-tile (fp32 elements)

// One operand of a k-tile: ROWS rows by 32 k. Bank placement as in sgemm.hip: K-major rows are
// 128 bytes whose 16-byte chunk c sits at c ^ ((row >> 1) & 7); M/N-major k-rows 16 .. 31 have
// their chunks at c ^ 8, so the two halves of a wave read opposite bank halves (ROWS >= 64; at 32
// rows the k-rows of the two halves share banks).
template <bool KMAJOR, int ROWS>
struct Operand32 {
  static constexpr int kLanesPerRow = ROWS / 4;  // M/N-major: lanes of one k-row
  __device__ static void source(int ii, int lane, int& row, int& k) {
    if (KMAJOR) {
      row = ii * 8 + (lane >> 3);
      k = ((lane & 7) ^ ((row >> 1) & 7)) * 4;
    } else {
      const int at = ii * 64 + lane;
      k = at / kLanesPerRow;
      row = ((at % kLanesPerRow) ^ flip(k)) * 4;
    }
  }
  __device__ static int flip(int k) { return ROWS >= 64 ? 8 * ((k >> 4) & 1) : 0; }
  // Operands of MFMA steps 4 qd .. 4 qd + 3 of the 32-row block at row `r0`.
  __device__ static f32x4_t read(const unsigned char HK_LDS* st, int r0, int qd, int lane) {
    const int r = r0 + (lane & 31), h = lane >> 5;
    if (KMAJOR) {
      const int c = 4 * h + qd;
      return *reinterpret_cast<const f32x4_t HK_LDS*>(st + r * 128 + ((c ^ ((r >> 1) & 7)) * 16));
    }
    const float HK_LDS* col =
        reinterpret_cast<const float HK_LDS*>(st) + (16 * h + 4 * qd) * ROWS + (r ^ (4 * flip(16 * h)));
    return f32x4_t{col[0], col[ROWS], col[2 * ROWS], col[3 * ROWS]};
  }
};

// 1 to 4 fp32 (n of them) from p, zeros behind.
__device__ __forceinline__ f32x4_t load_some(const float* p, int n) {
  f32x4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = e < n ? p[e] : 0.f;
  return v;
}

template <int BMT_, int BNT_, int WM_, int WN_, int KG_, int NA_>
struct Tile {
  static constexpr int BMT = BMT_, BNT = BNT_, WM = WM_, WN = WN_, KG = KG_, NA = NA_;
  static constexpr int kChains = KG * NA;  // serial sums that an output is formed from
  static constexpr int kGroupWaves = WM * WN, kThreads = kGroupWaves * KG * 64;
  static constexpr int kWaveM = BMT / WM, kWaveN = BNT / WN;
  static constexpr int kBlkM = kWaveM / 32, kBlkN = kWaveN / 32;
  static constexpr int kStageA = BMT * KT * 4, kStageB = BNT * KT * 4, kStage = kStageA + kStageB;
  static constexpr int kCopiesA = kStageA / 1024 / kGroupWaves;
  static constexpr int kCopiesB = kStageB / 1024 / kGroupWaves;
  static constexpr int kCopies = kCopiesA + kCopiesB;
  static constexpr int kStaging = 32 * (kWaveN * 4 + 16);
  static constexpr int kSums = BMT * BNT * 4;
  static constexpr size_t kRing = static_cast<size_t>(KG) * 2 * kStage;
  static constexpr size_t kEnd = static_cast<size_t>(kGroupWaves) * kStaging + (KG - 1) * kSums;
  static constexpr size_t kLds = kRing > kEnd ? kRing : kEnd;
  static_assert(kCopiesA * kGroupWaves * 1024 == kStageA, "whole copies per wave");
  static_assert(kCopiesB * kGroupWaves * 1024 == kStageB, "whole copies per wave");
};

template <class T, bool A_KMAJOR, bool B_KMAJOR>
__global__ __launch_bounds__(T::kThreads, 2) void sgemm_flex(hk::SgemmFlexCall g) {
  using OA = Operand32<A_KMAJOR, T::BMT>;
  using OB = Operand32<B_KMAJOR, T::BNT>;
  constexpr int kBlkM = T::kBlkM, kBlkN = T::kBlkN;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  unsigned char HK_LDS* lds = (unsigned char HK_LDS*)lds_raw;
  const int M = g.M, N = g.N, K = g.K, batch = blockIdx.z;
  const int tiles_m = (M + T::BMT - 1) / T::BMT, tiles_n = (N + T::BNT - 1) / T::BNT;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * T::BMT, n0 = tn * T::BNT;
  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = wave_all / T::kGroupWaves, wave = wave_all - group * T::kGroupWaves;
  const int wm = wave / T::WN, wn = wave % T::WN;

  // Group `group` takes k-tiles group, group + KG, ...; every wave passes `loops` barriers.
  const int all_tiles = (K + KT - 1) / KT;
  const int loops = (all_tiles + T::KG - 1) / T::KG;
  const int ktiles = (all_tiles - group + T::KG - 1) / T::KG;
  const int k0 = group * KT, klen = K - k0;
  constexpr int kStep = T::KG * KT;
  const float* pA = g.A + batch * g.sA + (A_KMAJOR ? m0 * g.lda + k0 : k0 * g.lda + m0);
  const float* pB = g.B + batch * g.sB + (B_KMAJOR ? n0 * g.ldb + k0 : k0 * g.ldb + n0);
  const int64_t stepA = A_KMAJOR ? kStep : kStep * g.lda;
  const int64_t stepB = B_KMAJOR ? kStep : kStep * g.ldb;
  // Rows past M (N) are clamped to the last row or 4-row vector: they feed no stored output.
  uint32_t off[T::kCopies];
  int kq[T::kCopies], nrow[T::kCopies];
#pragma unroll
  for (int q = 0; q < T::kCopies; ++q) {
    const bool isA = q < T::kCopiesA;
    int row, k;
    if (isA) OA::source(wave * T::kCopiesA + q, lane, row, k);
    else OB::source(wave * T::kCopiesB + q - T::kCopiesA, lane, row, k);
    const int left = (isA ? M - m0 : N - n0) - 1;
    const bool km = isA ? A_KMAJOR : B_KMAJOR;
    row = km ? min(row, left) : min(row, left & ~3);
    nrow[q] = km ? 4 : min(4, left - row + 1);
    const int64_t ld = isA ? g.lda : g.ldb;
    off[q] = static_cast<uint32_t>(km ? row * ld + k : k * ld + row);
    kq[q] = k;
  }
  unsigned char HK_LDS* ring = lds + group * 2 * T::kStage;
  auto src = [&](int q, int kt) {
    return reinterpret_cast<const char*>(q < T::kCopiesA ? pA + kt * stepA : pB + kt * stepB) +
           4 * off[q];
  };
  // Guarded loads only in the last k-tile: a vector across the end of K, or (M/N-major) across
  // the end of the matrix's last k-row; elsewhere the rest of the matrix covers the overhang
  // (ld >= 4).
  const bool tail = ktiles > 0 && klen - (ktiles - 1) * kStep < KT;
  const bool guard = tail || (!A_KMAJOR && (M & 3) != 0) || (!B_KMAJOR && (N & 3) != 0);
  f32x4_t reg[T::kCopies];
  auto load_whole = [&](int kt) {
#pragma unroll
    for (int q = 0; q < T::kCopies; ++q) reg[q] = *reinterpret_cast<const f32x4u_t*>(src(q, kt));
  };
  auto load = [&](int kt) {
    if (kt < ktiles - 1 || !guard) {
      load_whole(kt);
      return;
    }
#pragma unroll
    for (int q = 0; q < T::kCopies; ++q) {
      const bool km = q < T::kCopiesA ? A_KMAJOR : B_KMAJOR;
      const int left = klen - (kt * kStep + kq[q]);
      const int n = km ? max(0, min(4, left)) : left > 0 ? nrow[q] : 0;
      if (n == 4) reg[q] = *reinterpret_cast<const f32x4u_t*>(src(q, kt));
      else reg[q] = load_some(reinterpret_cast<const float*>(src(q, kt)), n);
    }
  };
  auto store = [&](int slot) {
#pragma unroll
    for (int q = 0; q < T::kCopies; ++q)
      *reinterpret_cast<f32x4_t HK_LDS*>(
          ring + slot * T::kStage +
          (q < T::kCopiesA ? (wave * T::kCopiesA + q) * 1024
                           : T::kStageA + (wave * T::kCopiesB + q - T::kCopiesA) * 1024) +
          16 * lane) = reg[q];
  };

  f32x16_t sum[T::NA][kBlkM][kBlkN];  // MFMA step s adds into set s % NA
#pragma unroll
  for (int a = 0; a < T::NA; ++a)
#pragma unroll
    for (int i = 0; i < kBlkM; ++i)
#pragma unroll
      for (int j = 0; j < kBlkN; ++j) sum[a][i][j] = f32x16_t{};

  if (ktiles > 0) {
    load(0);
    store(0);
  }
  if (ktiles > 1) load(1);
  __syncthreads();

  f32x4_t fa[2][kBlkM], fb[2][kBlkN];
  auto read = [&](int slot, int qd, int buf) {
    const unsigned char HK_LDS* sa = ring + slot * T::kStage;
#pragma unroll
    for (int i = 0; i < kBlkM; ++i) fa[buf][i] = OA::read(sa, wm * T::kWaveM + 32 * i, qd, lane);
#pragma unroll
    for (int j = 0; j < kBlkN; ++j)
      fb[buf][j] = OB::read(sa + T::kStageA, wn * T::kWaveN + 32 * j, qd, lane);
  };
  auto mma = [&](int buf) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < kBlkM; ++i)
#pragma unroll
        for (int j = 0; j < kBlkN; ++j)
          sum[e % T::NA][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
              fb[buf][j][e], fa[buf][i][e], sum[e % T::NA][i][j], 0, 0, 0);
  };
  if (ktiles > 0) read(0, 0, 0);
  // Quads 0 .. 2 read the next quad's operands while they multiply, and the next k-tile is written
  // to the other slot; the barrier before quad 3 publishes it and frees this slot.
  auto ktile = [&](int kt, auto steady_tag) {
    constexpr bool STEADY = decltype(steady_tag)::value;
    const int slot = kt & 1;
    const bool on = STEADY || kt < ktiles;
    if (on) {
#pragma unroll
      for (int qd = 0; qd < 3; ++qd) {
        read(slot, qd + 1, (qd + 1) & 1);
        mma(qd & 1);
        if (qd == 1 && (STEADY || kt + 1 < ktiles)) {
          store(slot ^ 1);
          if (STEADY) load_whole(kt + 2);
          else if (kt + 2 < ktiles) load(kt + 2);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (on) {
      if (STEADY || kt + 1 < ktiles) read(slot ^ 1, 0, 0);
      mma(1);
    }
  };
  int kt = 0;
  for (; kt + 2 < ktiles - 1; ++kt) ktile(kt, std::true_type{});
  for (; kt < loops; ++kt) ktile(kt, std::false_type{});

  __syncthreads();
  f32x16_t (&acc)[kBlkM][kBlkN] = sum[0];
#pragma unroll
  for (int a = 1; a < T::NA; ++a)
#pragma unroll
    for (int i = 0; i < kBlkM; ++i)
#pragma unroll
      for (int j = 0; j < kBlkN; ++j) acc[i][j] += sum[a][i][j];
  if constexpr (T::KG > 1) {
    if (merge_groups<T>(acc, lds, group, wave, lane)) return;
  }
  float* Cb = g.out.C + batch * g.out.sC;
  const int wrow0 = m0 + wm * T::kWaveM, wcol0 = n0 + wn * T::kWaveN;
  staged_rows<T::kWaveN, kBlkM>(
      acc, lds + wave * T::kStaging, lane, [&](int rr, int cc, const f32x4_t& a, const f32x4_t& b) {
        const int row = wrow0 + rr, col = wcol0 + cc;
        if (row >= M || col >= N) return;
        float* cp = Cb + static_cast<int64_t>(row) * g.out.ldc + col;
        const hk::F32Out& fo = g.out;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          f32x4_t v = fo.alpha * (half ? b : a);
          const int c0 = col + 4 * half, n = N - c0;
          if (n <= 0) break;
          float* p = cp + 4 * half;
          if (fo.beta != 0.0f)
            v += fo.beta * (n >= 4 ? static_cast<f32x4_t>(*reinterpret_cast<const f32x4u_t*>(p))
                                   : load_some(p, n));
          if (fo.bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              v[e] += fo.bias_scale * f32out_bias(fo, M, N, batch, min(c0 + e, N - 1));
          }
          if (n >= 4) {
            *reinterpret_cast<f32x4u_t*>(p) = v;
          } else {
#pragma unroll
            for (int e = 0; e < 3; ++e)
              if (e < n) p[e] = v[e];
          }
        }
      });
}

template <class T, bool AK, bool BKM>
hipError_t launch(const hk::SgemmFlexCall& c, hipStream_t stream) {
  static_assert(T::kLds <= 64 * 1024, "no LDS limit to raise");
  const int64_t tiles = hk::ceil_div(c.M, T::BMT) * hk::ceil_div(c.N, T::BNT);
  HK_CHECK_ARG(tiles <= INT32_MAX && c.batch <= 65535);
  hipLaunchKernelGGL((sgemm_flex<T, AK, BKM>), dim3(static_cast<unsigned>(tiles), 1, c.batch),
                     dim3(T::kThreads), T::kLds, stream, c);
  return hk::launch_status();
}
template <class T>
hipError_t layouts(const hk::SgemmFlexCall& c, hipStream_t stream) {
  HK_CHECK_ARG(!(c.ta && c.tb));  // the fp32 entry points have NT, TN and NN
  if (c.ta) return launch<T, false, false>(c, stream);
  return c.tb ? launch<T, true, true>(c, stream) : launch<T, true, false>(c, stream);
}

// The tile shapes: us per k of one workgroup that has its CU alone, of each of several that share
// one, and the fixed time of a launch. On MI355X, us (TFLOP/s; the fallback ran at about 2):
//   4095^3 NT / NN / TN       1170 / 1058 / 1000 (117 / 130 / 137) on 128 x 128
//   2049 x 2047 x 1025 NN       98 (88) on 64 x 64
//   511 x 511 x 2049 NN       20.0 (53) on 32 x 32
struct Shape {
  int bm, bn, chains;
  double alone, shared, fixed;
  hipError_t (*run)(const hk::SgemmFlexCall&, hipStream_t);
};
template <class T>
constexpr Shape shape(double alone, double shared, double fixed) {
  return Shape{T::BMT, T::BNT, T::kChains, alone, shared, fixed, &layouts<T>};
}
const Shape kShapes[] = {
    shape<Tile<32, 32, 1, 1, 4, 2>>(0.0063, 0.0060, 3.8),
    shape<Tile<64, 64, 2, 2, 1, 4>>(0.0205, 0.0178, 3.4),
    shape<Tile<128, 128, 2, 2, 1, 1>>(0.070, 0.0643, 5.0),
};
constexpr int kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);

}  // namespace

namespace hk {

int sgemm_flex_plan(int M, int N, int K, int batch, int min_chains) {
  const int64_t cus = device_cu_count();
  int best = 0;  // the first shape has the most chains
  double cost = 0.0;
  for (int i = 0; i < kNumShapes; ++i) {
    const Shape& s = kShapes[i];
    if (i > 0 && s.chains < min_chains) continue;
    const int64_t wgs = ceil_div(M, s.bm) * ceil_div(N, s.bn) * batch;
    const double share = static_cast<double>(ceil_div(wgs, cus)) * s.shared;
    const double t = s.fixed + K * (share > s.alone ? share : s.alone);
    if (i == 0 || t < cost) {
      cost = t;
      best = i;
    }
  }
  return best;
}

hipError_t sgemm_flex_run(int shape, const SgemmFlexCall& call, hipStream_t stream) {
  return kShapes[shape].run(call, stream);
}

}  // namespace hk
