// bgemm_flex.hip - the BF16 GEMM on small tiles and on operands of any alignment: the products that
// the 256-wide tiles of bgemm.hip leave most CUs idle on, and those whose rows are not whole
// 16-byte vectors (an odd vocabulary, an odd sequence length). Same contract: C = alpha * op(A)
// op(B) + beta * C (or + beta * bias), bf16 operands, fp32 accumulation, one rounding to bf16, all
// four transpose layouts, the k order of the sums fixed (deterministic).
//
// Design (gfx950): the LDS layout, MFMA operand order and epilogue of bgemm_tile.h on output tiles
// of BMT x BNT. Each wave owns kWaveM x kWaveN of the tile in 32 x 32 MFMA blocks. KG groups of
// waves share one output tile and take alternate k-tiles, each with an LDS ring of its own; their
// sums are added in group order through LDS before the epilogue. KG > 1 shortens the serial chain
// of k-tiles (copy, barrier, multiply), which bounds a product of few output tiles.
// Two ways for the operands to reach LDS:
//   - direct (16-byte aligned rows): global -> LDS copies that bypass registers, a ring of S
//     k-tiles, tile kt + S copied while tile kt + 1 .. kt + S - 1 wait or land;
//   - staged (RAGGED): 16-byte loads at any 2-byte address into registers (gfx950 serves
//     unaligned vector loads at 80% of the aligned rate when the rows sit in cache and 92% from
//     HBM: 6.7 against 8.4 TB/s and 5.8 against 6.3 TB/s), written to a ring of two LDS slots one
//     k-tile after they were issued.
// The last k-tile of a staged operand reads element by element where a vector would cross the end
// of K or of the matrix, and fills zeros past K.
#include <mutex>
#include <type_traits>

#include "bgemm_flex.h"
#include "bgemm_tile.h"

namespace {

using namespace hk::gemm;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

struct Operand {
  const uint16_t* p;
  int64_t ld, stride;  // leading dimension and batch stride (elements)
};
struct Args {
  int M, N, K;
  Epi ep;
  Operand a, b;
  uint16_t* C;
  int64_t ldc, sC;
  int split_k, k_per_split;
  bool by_matrix;  // matrix_order
  float* part;     // not NULL: fp32 partials [split][batch][M][part_pitch(N)] instead of C
  hk::F32Out fo;   // fo.C not NULL: fp32 C through its own epilogue instead
};

// Tile shape: BMT x BNT on WM x WN waves per k group, KG k groups, S ring slots (direct copies).
template <int BMT_, int BNT_, int WM_, int WN_, int KG_, int S_>
struct Tile {
  static constexpr int BMT = BMT_, BNT = BNT_, WM = WM_, WN = WN_, KG = KG_, S = S_;
  static constexpr int kGroupWaves = WM * WN;
  static constexpr int kThreads = kGroupWaves * KG * 64;
  static constexpr int kWaveM = BMT / WM, kWaveN = BNT / WN;
  static constexpr int kBlkM = kWaveM / 32, kBlkN = kWaveN / 32;
  static constexpr int kStageA = BMT * BK * 2, kStageB = BNT * BK * 2, kStage = kStageA + kStageB;
  static constexpr int kCopiesA = kStageA / 1024 / kGroupWaves;
  static constexpr int kCopiesB = kStageB / 1024 / kGroupWaves;
  static constexpr int kCopies = kCopiesA + kCopiesB;
  static constexpr int kStaging = 32 * (kWaveN * 4 + 16);  // epilogue area of one wave
  static constexpr int kSums = BMT * BNT * 4;              // one k group's accumulators
  static constexpr size_t lds(bool ragged) {
    const size_t ring = static_cast<size_t>(KG) * (ragged ? 2 : S) * kStage;
    const size_t end = static_cast<size_t>(kGroupWaves) * kStaging + (KG - 1) * kSums;
    return ring > end ? ring : end;
  }
  static_assert(kCopiesA * kGroupWaves * 1024 == kStageA, "whole copies per wave");
  static_assert(kCopiesB * kGroupWaves * 1024 == kStageB, "whole copies per wave");
};

// n (0 .. 8) elements from p, zeros behind them.
__device__ __forceinline__ u32x4_t load_some(const uint16_t* p, int n) {
  u32x4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t lo = 2 * e < n ? p[2 * e] : 0, hi = 2 * e + 1 < n ? p[2 * e + 1] : 0;
    v[e] = lo | (hi << 16);
  }
  return v;
}

template <class T, bool A_KMAJOR, bool B_KMAJOR, bool RAGGED>
__global__ __launch_bounds__(T::kThreads, T::kThreads >= 512 ? 1 : 2) void bgemm_flex(Args g) {
  using OA = TileOperand<A_KMAJOR, T::BMT>;
  using OB = TileOperand<B_KMAJOR, T::BNT>;
  constexpr int kSlots = RAGGED ? 2 : T::S;
  constexpr int kBlkM = T::kBlkM, kBlkN = T::kBlkN;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  unsigned char HK_LDS* lds = (unsigned char HK_LDS*)lds_raw;

  const int M = g.M, N = g.N;
  const int tiles_m = (M + T::BMT - 1) / T::BMT, tiles_n = (N + T::BNT - 1) / T::BNT;
  int tile = blockIdx.x, z = blockIdx.z, tm, tn;
  if (g.by_matrix) matrix_order(gridDim.x, gridDim.z, tile, z);
  const int batch = z / g.split_k;
  const int split = z - batch * g.split_k;
  tile_coords(tile, tiles_m, tiles_n, tm, tn, g.by_matrix);
  const int m0 = tm * T::BMT, n0 = tn * T::BNT;
  const int kbeg = split * g.k_per_split;
  const int kend = min(g.K, kbeg + g.k_per_split);

  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = wave_all / T::kGroupWaves, wave = wave_all - group * T::kGroupWaves;
  const int wm = wave / T::WN, wn = wave % T::WN;

  // Group `group` takes k-tiles group, group + KG, ... of the split. Every wave passes the same
  // number of barriers (loops = the most k-tiles of any group).
  const int all_tiles = (kend - kbeg + BK - 1) / BK;
  const int loops = (all_tiles + T::KG - 1) / T::KG;
  const int ktiles = (all_tiles - group + T::KG - 1) / T::KG;  // >= 0: group < KG
  const int k0 = kbeg + group * BK;
  const int klen = kend - k0;  // may be <= 0 when ktiles == 0
  constexpr int kStep = T::KG * BK;

  const uint16_t* pA = g.a.p + batch * g.a.stride +
                       (A_KMAJOR ? m0 * g.a.ld + k0 : k0 * g.a.ld + m0);
  const uint16_t* pB = g.b.p + batch * g.b.stride +
                       (B_KMAJOR ? n0 * g.b.ld + k0 : k0 * g.b.ld + n0);
  const int64_t stepA = A_KMAJOR ? kStep : kStep * g.a.ld;
  const int64_t stepB = B_KMAJOR ? kStep : kStep * g.b.ld;

  // Source of this wave's copies: element offsets from the k-tile's base, k within the tile, and
  // (row-major k) how many of the 8 rows exist. Rows past M (N) are clamped to the last row or
  // chunk; they only feed outputs that are not stored.
  uint32_t off[T::kCopies];
  int kq[T::kCopies], nrow[T::kCopies];
#pragma unroll
  for (int q = 0; q < T::kCopies; ++q) {
    const bool isA = q < T::kCopiesA;
    int row, k;
    if (isA) OA::source(wave * T::kCopiesA + q, lane, row, k);
    else OB::source(wave * T::kCopiesB + q - T::kCopiesA, lane, row, k);
    const int left = (isA ? M - m0 : N - n0) - 1;  // last row of the matrix, from the tile's first
    const bool km = isA ? A_KMAJOR : B_KMAJOR;
    row = km ? min(row, left) : min(row, left & ~7);
    nrow[q] = km ? 8 : min(8, left - row + 1);
    const int64_t ld = isA ? g.a.ld : g.b.ld;
    off[q] = static_cast<uint32_t>(km ? row * ld + k : k * ld + row);
    kq[q] = k;
  }

  const unsigned ring = static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds)) +
                        group * kSlots * T::kStage;
  // LDS address of copy q in ring slot `slot`
  auto dst = [&](int q, int slot) {
    return ring + slot * T::kStage +
           (q < T::kCopiesA ? (wave * T::kCopiesA + q) * 1024
                            : T::kStageA + (wave * T::kCopiesB + q - T::kCopiesA) * 1024);
  };
  auto put = [&](int q, int slot, u32x4_t v) {
    *reinterpret_cast<u32x4_t HK_LDS*>((unsigned char HK_LDS*)(uintptr_t)dst(q, slot) +
                                       16 * lane) = v;
  };
  auto src = [&](int q, int kt) {
    return (q < T::kCopiesA ? pA + kt * stepA : pB + kt * stepB);
  };
  // this group's last k-tile when it is the last of the split and K ends inside it
  const bool tail = ktiles > 0 && klen - (ktiles - 1) * kStep < BK;

  // ---- direct copies
  auto copy = [&](int kt, int slot, bool steady) {
    const bool fill = !steady && tail && kt == ktiles - 1;
#pragma unroll
    for (int q = 0; q < T::kCopies; ++q) {
      if (!fill || kt * kStep + kq[q] < klen)
        copy16_to_lds(src(q, kt), static_cast<int>(2 * off[q]), dst(q, slot));
      else
        put(q, slot, u32x4_t{0u, 0u, 0u, 0u});
    }
  };
  // ---- staged loads
  // Vectors that would cross the end of K (a partial last k-tile) or, in the matrix's last k-row,
  // the end of a row (the rest of the matrix covers every other row's overhang, ld >= 8).
  const bool guardA = RAGGED && ktiles > 0 && kend == g.K &&
                      (tail || (!A_KMAJOR && (M & 7) != 0));
  const bool guardB = RAGGED && ktiles > 0 && kend == g.K &&
                      (tail || (!B_KMAJOR && (N & 7) != 0));
  u32x4_t reg[T::kCopies];
  auto load_whole = [&](int kt) {
#pragma unroll
    for (int q = 0; q < T::kCopies; ++q)
      __builtin_memcpy(&reg[q], reinterpret_cast<const char*>(src(q, kt)) + 2 * off[q], 16);
  };
  auto load = [&](int kt) {
    if (kt < ktiles - 1 || !(guardA || guardB)) {
      load_whole(kt);
      return;
    }
#pragma unroll
    for (int q = 0; q < T::kCopies; ++q) {
      const bool isA = q < T::kCopiesA;
      const bool km = isA ? A_KMAJOR : B_KMAJOR;
      const char* p = reinterpret_cast<const char*>(src(q, kt)) + 2 * off[q];
      const int left = klen - (kt * kStep + kq[q]);  // k values from here to the end of K
      int n = km ? max(0, min(8, left)) : left > 0 ? nrow[q] : 0;
      if (!(isA ? guardA : guardB)) n = 8;
      if (n == 8) __builtin_memcpy(&reg[q], p, 16);
      else reg[q] = load_some(reinterpret_cast<const uint16_t*>(p), n);
    }
  };
  auto store = [&](int slot) {
#pragma unroll
    for (int q = 0; q < T::kCopies; ++q) put(q, slot, reg[q]);
  };

  f32x16_t acc[kBlkM][kBlkN];
#pragma unroll
  for (int i = 0; i < kBlkM; ++i)
#pragma unroll
    for (int j = 0; j < kBlkN; ++j) acc[i][j] = f32x16_t{};

  if constexpr (RAGGED) {
    if (ktiles > 0) {
      load(0);
      store(0);
    }
    if (ktiles > 1) load(1);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  } else {
#pragma unroll
    for (int p = 0; p < kSlots; ++p)
      if (p < ktiles) copy(p, p, false);
    // k-tile 0 landed; a partial last k-tile may have issued fewer copies than counted here
    if (ktiles > kSlots - 1 && !(tail && ktiles == kSlots))
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kSlots - 1) * T::kCopies) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  }
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");  // no LDS access moves across

  const unsigned char HK_LDS* ringp = (const unsigned char HK_LDS*)(uintptr_t)ring;
  auto read = [&](int slot, int s, bf16x8_t (&a)[kBlkM], bf16x8_t (&b)[kBlkN]) {
    const unsigned char HK_LDS* sa = ringp + slot * T::kStage;
#pragma unroll
    for (int i = 0; i < kBlkM; ++i) a[i] = OA::read(sa, wm * T::kWaveM, i, s, lane);
#pragma unroll
    for (int j = 0; j < kBlkN; ++j) b[j] = OB::read(sa + T::kStageA, wn * T::kWaveN, j, s, lane);
  };
  auto mma = [&](const bf16x8_t (&a)[kBlkM], const bf16x8_t (&b)[kBlkN]) {
#pragma unroll
    for (int i = 0; i < kBlkM; ++i)
#pragma unroll
      for (int j = 0; j < kBlkN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
  };
  constexpr int kSteps = BK / 16;
  bf16x8_t fa[2][kBlkM], fb[2][kBlkN];  // the operands of two 16-deep k steps
  if (ktiles > 0) read(0, 0, fa[0], fb[0]);
  // Before the barrier of k-tile kt: this wave's part of tile kt + 1 is in LDS, its operand reads
  // of tile kt are done.
  auto landed = [&](int kt, bool steady) {
    if constexpr (RAGGED) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    } else {
      // k-tiles kt + 2 .. kt + S - 1 may still be in flight
      const int last = kt + kSlots - 1;
      if (steady || (last < ktiles && !(tail && last == ktiles - 1)))
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kSlots - 2) * T::kCopies)
                     : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  constexpr int kReads = (A_KMAJOR ? 1 : 2) * kBlkM + (B_KMAJOR ? 1 : 2) * kBlkN;
  int slot = 0;
  // One k-tile. STEADY (compile-time): tiles kt + 1 .. kt + kAhead exist and are whole, so nothing
  // is tested inside the loop body.
  constexpr int kAhead = RAGGED ? 2 : kSlots;
  auto ktile = [&](int kt, auto steady_tag) {
    constexpr bool STEADY = decltype(steady_tag)::value;
    // Steps 0 .. 2 read the operands of the next step while they multiply; the barrier before
    // step 3 publishes tile kt + 1 and frees this tile's slot (every wave holds its step-3
    // operands).
    const int next = slot == kSlots - 1 ? 0 : slot + 1;
    const bool on = STEADY || kt < ktiles;
    if (on) {
#pragma unroll
      for (int s = 0; s < kSteps - 1; ++s) {
        read(slot, s + 1, fa[(s + 1) & 1], fb[(s + 1) & 1]);
        mma(fa[s & 1], fb[s & 1]);
        interleave_reads<kBlkM * kBlkN, kReads>();
        if (RAGGED && s == 1 && (STEADY || kt + 1 < ktiles)) {
          store(next);
          if (STEADY) load_whole(kt + 2);
          else if (kt + 2 < ktiles) load(kt + 2);
        }
      }
    }
    landed(kt, STEADY);
    if (on) {
      if (STEADY || kt + 1 < ktiles) read(next, 0, fa[0], fb[0]);
      if (!RAGGED && (STEADY || kt + kSlots < ktiles)) copy(kt + kSlots, slot, STEADY);
      mma(fa[(kSteps - 1) & 1], fb[(kSteps - 1) & 1]);
    }
    slot = next;
  };
  int kt = 0;
  for (; kt + kAhead < ktiles - 1; ++kt) ktile(kt, std::true_type{});
  for (; kt < loops; ++kt) ktile(kt, std::false_type{});

  // Epilogue. The ring is free after this barrier; the k groups' sums are added in group order.
  __syncthreads();
  if constexpr (T::KG > 1) {
    if (merge_groups<T>(acc, lds, group, wave, lane)) return;
  }
  unsigned char HK_LDS* area = lds + wave * T::kStaging;
  const int wrow0 = m0 + wm * T::kWaveM, wcol0 = n0 + wn * T::kWaveN;
  if (g.fo.C) {
    store_f32<T::kWaveN, kBlkM>(acc, area, lane, g.fo, batch, M, N, wrow0, wcol0);
    return;
  }
  if (g.part) {
    store_partial<T::kWaveN, kBlkM>(
        acc, area, lane,
        g.part + (static_cast<int64_t>(split) * (gridDim.z / g.split_k) + batch) * M * part_pitch(N),
        M, N, wrow0, wcol0);
    return;
  }
  store_bf16<T::kWaveN, kBlkM>(acc, area, lane, g.ep, g.C + batch * g.sC, g.ldc, M, N, wrow0,
                               wcol0);
}

template <class T, bool AK, bool BKM, bool RAGGED>
hipError_t launch(const Args& g, int batch, hipStream_t stream) {
  constexpr size_t kLds = T::lds(RAGGED);
  static_assert(kLds <= 160 * 1024, "fits gfx950's 160 KiB of LDS");
  static std::once_flag once;
  static hipError_t attr_status = hipSuccess;
  std::call_once(once, [] {
    attr_status = hipFuncSetAttribute(reinterpret_cast<const void*>(&bgemm_flex<T, AK, BKM, RAGGED>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(kLds));
  });
  HK_RETURN_IF_ERROR(attr_status);
  const int64_t tiles = hk::ceil_div(g.M, T::BMT) * hk::ceil_div(g.N, T::BNT);
  HK_CHECK_ARG(tiles <= INT32_MAX && static_cast<int64_t>(batch) * g.split_k <= 65535);
  Args a = g;
  a.by_matrix = batch > 1 && tiles * batch * g.split_k <= INT32_MAX;
  hipLaunchKernelGGL((bgemm_flex<T, AK, BKM, RAGGED>),
                     dim3(static_cast<unsigned>(tiles), 1, batch * g.split_k), dim3(T::kThreads),
                     kLds, stream, a);
  return hk::launch_status();
}

template <class T, bool RAGGED>
hipError_t layouts(bool ta, bool tb, const Args& g, int batch, hipStream_t stream) {
  // A is k-major unless transposed; B is k-major only when transposed.
  if (!ta) return tb ? launch<T, true, true, RAGGED>(g, batch, stream)
                     : launch<T, true, false, RAGGED>(g, batch, stream);
  return tb ? launch<T, false, true, RAGGED>(g, batch, stream)
            : launch<T, false, false, RAGGED>(g, batch, stream);
}
// The tile shapes, with what each costs: us per k-tile of one workgroup on a mostly idle device
// (alone), of each of those that share a CU of a busy one (shared), how many a CU holds, and the
// fixed time of a launch (fill, epilogue). A product of few tiles is bound by the serial chain of
// its k-tiles, which k groups shorten; one of many by the CU's copies and LDS reads per multiply,
// which fall with the tile's area. Fitted to back-to-back launches of random shapes on MI355X,
// where the plan's time came within 2% (aligned rows) and 4% (ragged) of the best shape and split
// of each. Times (us) on the 256-wide tiles, finalize included, and here:
//   512 x 2304 x 768 NN   22.0   8.2        2048^3 NN              39.9  21.8
//   512 x 768 x 2304 NT   22.0   9.9        1024 x 4096 x 4096 TN  54.0  37.8
//   768 x 2304 x 512 TN   10.3   6.9        64 x 256 x 192 NT       7.2   4.1
// Rows of odd length ran at about 2 TFLOP/s on the fallback kernel; here 50257 x 768 x 2048 TN takes
// 187 us (845 TFLOP/s) and 2048 x 768 x 50257 NN in 10 splits 190 us (833).
struct Shape {
  int bm, bn;
  bool ragged;
  double alone, shared;
  int per_cu;
  double fixed;
  hipError_t (*run)(bool, bool, const Args&, int, hipStream_t);
};
const Shape kShapes[] = {
    {64, 64, false, 0.26, 0.20, 3, 3.0, &layouts<Tile<64, 64, 2, 2, 1, 3>, false>},
    {64, 64, false, 0.21, 0.28, 1, 3.3, &layouts<Tile<64, 64, 2, 2, 2, 3>, false>},
    {64, 64, false, 0.19, 0.29, 1, 4.8, &layouts<Tile<64, 64, 2, 2, 4, 2>, false>},
    {128, 64, false, 0.38, 0.32, 2, 3.4, &layouts<Tile<128, 64, 2, 2, 1, 3>, false>},
    {128, 64, false, 0.34, 0.35, 1, 3.6, &layouts<Tile<128, 64, 2, 2, 2, 3>, false>},
    {128, 128, false, 0.56, 0.60, 1, 4.0, &layouts<Tile<128, 128, 2, 2, 2, 2>, false>},
    {64, 64, true, 0.37, 0.33, 4, 3.2, &layouts<Tile<64, 64, 2, 2, 1, 2>, true>},
    {64, 64, true, 0.31, 0.35, 2, 3.9, &layouts<Tile<64, 64, 2, 2, 2, 2>, true>},
    {64, 64, true, 0.28, 0.38, 1, 4.9, &layouts<Tile<64, 64, 2, 2, 4, 2>, true>},
    {128, 64, true, 0.60, 0.60, 1, 3.8, &layouts<Tile<128, 64, 2, 2, 2, 2>, true>},
    {128, 128, true, 0.92, 0.69, 2, 4.0, &layouts<Tile<128, 128, 2, 2, 1, 2>, true>},
    {256, 256, true, 1.70, 1.90, 1, 8.0, &layouts<Tile<256, 256, 2, 4, 1, 2>, true>},
};
constexpr int kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);

}  // namespace

namespace hk {

FlexPlan bgemm_flex_plan(int M, int N, int K, int batch, int split_k, bool ragged) {
  const int64_t cus = device_cu_count(), ktiles = ceil_div(K, BK);
  FlexPlan best{0, 1, K, 0.0};
  // A further round of workgroups on the CUs: its fill and the stores of its outputs. At 1.5 us the
  // aligned shapes were taken over the 256-wide tiles for large outputs of few k, up to twice as slow
  // (5208 x 6880 x 80: 43.4 us against 28.3); at 3.0 us, over 333 random products of 64 to 13,000
  // rows and columns and 8 to 6,000 k, 5 are more than 5% slower than those tiles (at most 16%)
  // where 33 were.
  const double round = ragged ? 1.5 : 3.0;
  for (int i = 0; i < kNumShapes; ++i) {
    const Shape& s = kShapes[i];
    if (s.ragged != ragged) continue;
    const int64_t tiles = ceil_div(M, s.bm) * ceil_div(N, s.bn) * batch;
    // what each further split costs at least: the partials' finalize, a launch and an HBM pass
    auto finalize = [&](int64_t used) {
      return 4.5 + 0.35 * static_cast<double>(used) +
             static_cast<double>(4 * used + 2) * M * static_cast<double>(N) * batch / 6.0e6;
    };
    for (int want = split_k > 0 ? split_k : 1; want <= (split_k > 0 ? split_k : 32); ++want) {
      // the k range of a split is a whole number of k-tiles; `used` splits are not empty
      const int64_t kt = ceil_div(ktiles, want), used = ceil_div(ktiles, kt);
      if (split_k == 0 && want > 1) {
        // no later `want` can be better: its ranges are no longer, its finalize no cheaper
        if (kt < 4 || batch * used > 65535) break;
        if (best.tile && s.fixed + finalize(want) >= best.cost) break;
        if (used != want) continue;
      }
      const int64_t wgs = tiles * used, held = cus * s.per_cu;
      const int64_t full = wgs / held, last = wgs % held;
      // `share` workgroups on each CU: the slower of one's serial chain and the CU's throughput;
      // a launch that fills under half of the CUs meets less contention
      auto per_ktile = [&](int64_t wg) {
        const double share = static_cast<double>(ceil_div(wg, cus));
        const double busy = 2 * wg < cus ? s.alone : s.shared * share;
        return busy > s.alone ? busy : s.alone;
      };
      double cost = s.fixed + round * static_cast<double>(full + (last > 0) - 1);
      if (full > 0) cost += static_cast<double>(kt * full) * per_ktile(held);
      if (last > 0) cost += static_cast<double>(kt) * per_ktile(last);
      if (used > 1) cost += finalize(used);
      if (best.tile == 0 || cost < best.cost)
        best = FlexPlan{i + 1, static_cast<int>(used), static_cast<int>(kt * BK), cost};
    }
  }
  return best;
}

int bgemm_flex_tile_rows(int tile) { return tile ? kShapes[tile - 1].bm : 0; }

hipError_t bgemm_flex_run(int tile, const FlexCall& c, hipStream_t stream) {
  HK_CHECK_ARG(tile >= 1 && tile <= kNumShapes && c.used >= 1 && (c.used == 1 || c.part));
  Args g{};
  g.M = c.M, g.N = c.N, g.K = c.K;
  if (c.ep) g.ep = *c.ep;
  g.a = Operand{c.A, c.lda, c.sA};
  g.b = Operand{c.B, c.ldb, c.sB};
  g.C = c.C, g.ldc = c.ldc, g.sC = c.sC;
  g.split_k = c.used, g.k_per_split = c.used > 1 ? c.kps : c.K;
  g.part = c.used > 1 ? c.part : nullptr;
  if (c.used == 1 && c.out) g.fo = *c.out;
  return kShapes[tile - 1].run(c.ta, c.tb, g, c.batch, stream);
}

}  // namespace hk
