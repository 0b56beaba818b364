// layernorm.hip - LayerNorm forward / backward over rows [rows, cols] of fp32, bf16 or fp16
// (statistics, gamma/beta gradients and all arithmetic in fp32).
//
// Reference behaviour:
//   forward            kernels/layernorm/layer_norm_forward_sm89_kernel.cu:27-209
//                      mean, rstd = 1/sqrt(var + eps) (biased var), y = (x - mean) * rstd * g + b
//   backward (input)   kernels/layernorm/ln_backward_input_sm89_kernel.cu:33-105
//                      dx = rstd * (dy g - (s1 + xhat s2) / cols), s1 = sum dy g,
//                      s2 = sum dy g xhat
//   backward (g, b)    kernels/layernorm/ln_backward_gamma_beta_sm89_kernel.cu:15-49
//                      dgamma += sum_r dy xhat, dbeta += sum_r dy
//
// Design (gfx950): one 64-lane wave owns one row; a row of at most 16 16-byte vectors per lane
// (cols <= 4096 fp32, 8192 16-bit) is held in VGPRs in its storage format, so x is read from HBM
// once and mean/variance are computed in two exact passes over registers (no Welford merge). Rows
// of any length and alignment take this path (Vec): gfx950 serves unaligned 16-byte accesses, and a
// row that is no whole number of vectors ends with one that overlaps the vector before it. The
// gamma/beta gradient is accumulated per lane in registers across the rows a wave visits,
// reduced across the workgroup's waves in LDS, written as one partial per workgroup, and summed over
// the workgroups in a fixed order by a second small kernel: the result is deterministic, unlike
// the reference's atomics. Rows of 2049 to 4096 columns are shared by four waves there; few rows
// take one launch for both gradients (ln_bwd_few_rows). Longer rows use a workgroup-per-row
// fallback and a column-slab reduction.
#include <initializer_list>
#include <mutex>
#include <type_traits>

#include "hk_device.h"
#include "hk_host.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / HK_WAVE;

// Storage type of a format tag, in a form that template argument deduction does not look at.
template <typename T>
using St = typename T::storage;

__device__ __forceinline__ uint4 u4_zero() { return make_uint4(0u, 0u, 0u, 0u); }

// Vector c of a row of `cols` elements. RAGGED: rows start at any element, and when cols is no
// multiple of the vector length (and at least one vector) the last vector starts early and
// repeats `skip` elements of the one before it, which its lane leaves out.
typedef uint32_t any_t __attribute__((ext_vector_type(4), aligned(2)));  // 16 bytes anywhere
template <typename T, bool RAGGED>
struct Vec {
  using S = typename T::storage;
  static constexpr int P = T::kPerVec;
  __device__ static int start(int c, int cols) { return RAGGED ? min(c * P, cols - P) : c * P; }
  __device__ static int skip(int c, int cols) { return RAGGED ? c * P - start(c, cols) : 0; }
  __device__ static uint4 load_nt(const S* row, int c, int cols) {
    if (!RAGGED) return hk::ld_nt(reinterpret_cast<const uint4*>(row) + c);
    const any_t v =
        __builtin_nontemporal_load(reinterpret_cast<const any_t*>(row + start(c, cols)));
    return make_uint4(v.x, v.y, v.z, v.w);
  }
  __device__ static uint4 load(const S* row, int c, int cols) {
    if (!RAGGED) return reinterpret_cast<const uint4*>(row)[c];
    const any_t v = *reinterpret_cast<const any_t*>(row + start(c, cols));
    return make_uint4(v.x, v.y, v.z, v.w);
  }
  __device__ static void unpack(const uint4& v, int c, int cols, float* f) {
    T::unpack(v, f);
    if (RAGGED) {
      const int n = skip(c, cols);
#pragma unroll
      for (int k = 0; k < P; ++k) f[k] = k < n ? 0.f : f[k];
    }
  }
  __device__ static void store_nt(S* row, int c, int cols, const float* f) {
    const uint4 v = T::pack(f);
    if (!RAGGED) {
      hk::st_nt(reinterpret_cast<uint4*>(row) + c, v);
      return;
    }
    S* p = row + start(c, cols);
    const int n = skip(c, cols);
    if (n == 0) {
      __builtin_nontemporal_store(any_t{v.x, v.y, v.z, v.w}, reinterpret_cast<any_t*>(p));
      return;
    }
#pragma unroll
    for (int k = 0; k < P; ++k)
      if (k >= n) T::store(p, k, f[k]);
  }
};

// One 16-byte vector of gamma (or beta) as fp32, or `dflt` everywhere when the pointer is NULL.
template <typename T, bool RAGGED>
__device__ __forceinline__ void affine(const St<T>* p, int c, int cols, float dflt, float* f) {
  if (p) {
    T::unpack(Vec<T, RAGGED>::load(p, c, cols), f);
  } else {
#pragma unroll
    for (int k = 0; k < T::kPerVec; ++k) f[k] = dflt;
  }
}

// ------------------------------------------------------------------------------------------
// Forward, register-resident rows: VPL 16-byte vectors per lane, nvec vectors per row.
// ------------------------------------------------------------------------------------------
template <typename T, int VPL, bool RAGGED>
__global__ __launch_bounds__(kThreads) void ln_fwd_reg(const St<T>* __restrict__ x,
                                                       const St<T>* __restrict__ gamma,
                                                       const St<T>* __restrict__ beta,
                                                       St<T>* __restrict__ y,
                                                       float* __restrict__ mean_out,
                                                       float* __restrict__ rstd_out, int rows,
                                                       int cols, float inv_cols, float eps) {
  using V = Vec<T, RAGGED>;
  constexpr int P = T::kPerVec;
  const int nvec = (cols + P - 1) / P;
  const int lane = threadIdx.x & (HK_WAVE - 1);
  const int row = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const St<T>* xr = x + static_cast<int64_t>(row) * cols;
  uint4 v[VPL];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = lane + i * HK_WAVE;
    v[i] = (c < nvec) ? V::load_nt(xr, c, cols) : u4_zero();
    float f[P];
    V::unpack(v[i], c < nvec ? c : 0, cols, f);
    s += hk::tree_sum<P>(f);
  }
  const float mu = hk::wave_sum(s) * inv_cols;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = lane + i * HK_WAVE;
    if (c < nvec) {
      float f[P];
      T::unpack(v[i], f);
#pragma unroll
      for (int k = 0; k < P; ++k)
        f[k] = RAGGED && k < V::skip(c, cols) ? 0.f : (f[k] - mu) * (f[k] - mu);
      q += hk::tree_sum<P>(f);
    }
  }
  const float var = hk::wave_sum(q) * inv_cols;
  const float rs = 1.0f / sqrtf(var + eps);
  if (lane == 0) {
    if (mean_out) mean_out[row] = mu;
    if (rstd_out) rstd_out[row] = rs;
  }
  St<T>* yr = y + static_cast<int64_t>(row) * cols;
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = lane + i * HK_WAVE;
    if (c < nvec) {
      float f[P], g[P], b[P];
      T::unpack(v[i], f);
      affine<T, RAGGED>(gamma, c, cols, 1.f, g);
      affine<T, RAGGED>(beta, c, cols, 0.f, b);
#pragma unroll
      for (int k = 0; k < P; ++k) f[k] = (f[k] - mu) * rs * g[k] + b[k];
      V::store_nt(yr, c, cols, f);
    }
  }
}

// Waves per workgroup of the backward kernels that accumulate gamma/beta: 8 when the flat
// LDS reduction of 8 waves fits 64 KiB (cols <= 1024), else 4. The grid is one workgroup
// per CU (8 waves) or two (4 waves), so each CU holds 8 waves and writes one or two partials
// for the finalize to read back. Measured at 4096 x 768 on MI355X against 4 waves and two
// workgroups per CU (512 partials): 12.2 against 12.9 us per fused backward (fp32), 9.8
// against 10.7 us (bf16); a tree reduction over the waves instead of the flat one was slower.
constexpr int gb_waves(int cols) { return cols <= 1024 ? 8 : 4; }

// One row per wave: when every row fits one round of 16-wave workgroups, one per CU
// (rows <= CUs x 16, cols <= kOneRowMaxCols<T>, so the flat reduction's 16 x 2 x cols floats fit
// 128 KiB), the gamma/beta backward runs the ONE_ROW form of ln_bwd_reg: no prefetch registers
// (108 VGPRs at 768 fp32 columns, 4 waves per SIMD), each wave's row in flight at once, still
// one partial per CU. fp32 rows of 4 vectors per lane (769-1024 columns) would spill at the
// 128-VGPR limit of 4 waves per SIMD and keep the prefetching form.
// 4096 x 768 fp32 fused backward on MI355X, one buffer set: 11.87 -> 11.27 us per call (the
// kernel alone 8.90 -> 8.37 us); eight such waves with two workgroups per CU made the kernel
// 8.02 us but its 512 partials cost the finalize more than that.
constexpr int kOneRowWaves = 16;
template <typename T>
constexpr int kOneRowMaxCols = T::kPerVec == 4 ? 768 : 1024;

// ------------------------------------------------------------------------------------------
// Backward, register-resident rows. WRITE_DX: produce grad_x. DO_GB: accumulate the
// per-workgroup gamma/beta partials into part[blockIdx.x][2 * cols] (gamma then beta).
// Each wave walks its rows with the next row's dy / x already in flight (software prefetch),
// so the two wave reductions of one row overlap the loads of the next; ONE_ROW drops the
// prefetch (each row is loaded at the top of its iteration) for grids where each wave has one
// row. dy, x and gamma stay in registers in their storage format and are widened to fp32
// where they are used. NW > 1: NW waves share a row (vectors dealt to them 64 by 64) and
// exchange their two sums through LDS, so rows of up to 4096 columns keep their gamma/beta sums
// in registers; every wave of the workgroup then makes the same number of iterations.
// ------------------------------------------------------------------------------------------
template <typename T, int VPL, bool WRITE_DX, bool DO_GB, int WAVES, bool ONE_ROW = false,
          bool RAGGED = false, int NW = 1>
__global__ __launch_bounds__(WAVES * HK_WAVE, ONE_ROW && WAVES == 16 ? 4 : 1) void ln_bwd_reg(
    const St<T>* __restrict__ dy, const St<T>* __restrict__ x, const float* __restrict__ mean,
    const float* __restrict__ rstd, const St<T>* __restrict__ gamma, St<T>* __restrict__ dx,
    float* __restrict__ part, int rows, int cols, float inv_cols) {
  // Every product below is rounded on its own (as the reference formula is written), so a
  // row whose terms cancel exactly (cols == 1) gives exactly zero.
#pragma clang fp contract(off)
  using V = Vec<T, RAGGED>;
  constexpr int P = T::kPerVec;
  constexpr int SLOTS = WAVES / NW;  // rows in flight per workgroup
  extern __shared__ float4 lds4[];   // [SLOTS][2][cols] floats when DO_GB
  __shared__ float2 row_sums[2][NW > 1 ? WAVES : 1];
  const int nvec = (cols + P - 1) / P;
  const int lane = threadIdx.x & (HK_WAVE - 1);
  const int wave = threadIdx.x >> 6;
  const int slot = wave / NW, share = wave % NW;
  auto col = [&](int i) { return lane + (share + NW * i) * HK_WAVE; };  // vector i of this lane
  uint4 graw[VPL];
  float acc_g[VPL][P], acc_b[VPL][P];
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = col(i);
    // NW > 1 reads gamma where it is used (from cache): held here, 4096 columns would spill
    if (NW == 1) graw[i] = (gamma && c < nvec) ? V::load(gamma, c, cols) : u4_zero();
#pragma unroll
    for (int k = 0; k < P; ++k) acc_g[i][k] = acc_b[i][k] = 0.f;
  }
  const int stride = gridDim.x * SLOTS;
  int row = blockIdx.x * SLOTS + slot;
  uint4 dn[VPL], xn[VPL];
  float mn = 0.f, rn = 0.f;
  auto fetch = [&](int r) {
    const St<T>* dyr = dy + static_cast<int64_t>(r) * cols;
    const St<T>* xr = x + static_cast<int64_t>(r) * cols;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const int c = col(i);
      dn[i] = (c < nvec) ? V::load_nt(dyr, c, cols) : u4_zero();
      xn[i] = (c < nvec) ? V::load_nt(xr, c, cols) : u4_zero();
    }
    mn = mean[r];
    rn = rstd[r];
  };
  // dy, x-hat and dy * gamma of vector i of the current row (zero past the row end and for the
  // repeated elements of a ragged row's last vector).
  auto widen = [&](const uint4& draw, const uint4& xraw, int i, float m, float rs, float* d,
                   float* n, float* a) {
    const int c = col(i);
    const bool in = c < nvec;
    const int skip = RAGGED && in ? V::skip(c, cols) : 0;
    float g[P];
    T::unpack(draw, d);
    T::unpack(xraw, n);
    if (gamma) {
      T::unpack(NW == 1 ? graw[i] : V::load(gamma, in ? c : 0, cols), g);
    } else {
#pragma unroll
      for (int k = 0; k < P; ++k) g[k] = 1.f;
    }
#pragma unroll
    for (int k = 0; k < P; ++k) {
      const bool own = in && (!RAGGED || k >= skip);
      n[k] = own ? (n[k] - m) * rs : 0.f;
      if (RAGGED) d[k] = own ? d[k] : 0.f;
      a[k] = d[k] * g[k];
    }
  };
  if (!ONE_ROW && row < rows) fetch(row);
  int parity = 0;
  // NW > 1: `row - slot` is the same for the whole workgroup, which iterates together
  for (; (NW > 1 ? row - slot : row) < rows; row += stride) {
    const bool live = NW == 1 || row < rows;
    if (ONE_ROW && live) fetch(row);
    uint4 dcur[VPL], xcur[VPL];
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      dcur[i] = dn[i];
      xcur[i] = xn[i];
    }
    const float m = mn, rs = rn;
    if (!ONE_ROW && row + stride < rows) fetch(row + stride);
    float s1 = 0.f, s2 = 0.f;
    if (live) {
#pragma unroll
      for (int i = 0; i < VPL; ++i) {
        float d[P], n[P], a[P];
        widen(dcur[i], xcur[i], i, m, rs, d, n, a);
        if (DO_GB) {
#pragma unroll
          for (int k = 0; k < P; ++k) {
            acc_g[i][k] += d[k] * n[k];
            acc_b[i][k] += d[k];
          }
        }
        if (WRITE_DX) {
          s1 += hk::tree_sum<P>(a);
#pragma unroll
          for (int k = 0; k < P; ++k) n[k] = a[k] * n[k];
          s2 += hk::tree_sum<P>(n);
        }
      }
    }
    if (WRITE_DX) {
      float t1 = hk::wave_sum(s1), t2 = hk::wave_sum(s2);
      if constexpr (NW > 1) {
        // two buffers: the next row's sums are written while a slower wave still reads these
        if (lane == 0) row_sums[parity][wave] = make_float2(t1, t2);
        __syncthreads();
        t1 = t2 = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          const float2 v = row_sums[parity][slot * NW + w];
          t1 += v.x;
          t2 += v.y;
        }
        parity ^= 1;
      }
      if (live) {
        St<T>* dxr = dx + static_cast<int64_t>(row) * cols;
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
          const int c = col(i);
          if (c < nvec) {
            float d[P], n[P], a[P], o[P];
            widen(dcur[i], xcur[i], i, m, rs, d, n, a);
#pragma unroll
            for (int k = 0; k < P; ++k) o[k] = rs * (a[k] - (t1 + n[k] * t2) * inv_cols);
            V::store_nt(dxr, c, cols, o);
          }
        }
      }
    }
  }
  if constexpr (DO_GB) {
    // LDS holds [slot][gamma | beta][cols] floats
    float* ldsf = reinterpret_cast<float*>(lds4);
    float* my = ldsf + static_cast<int64_t>(slot) * 2 * cols;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const int c = col(i);
      if (c >= nvec) continue;
      float* g = my + V::start(c, cols);
      float* b = g + cols;
      if constexpr (RAGGED) {
        const int skip = V::skip(c, cols);
#pragma unroll
        for (int k = 0; k < P; ++k)
          if (k >= skip) {
            g[k] = acc_g[i][k];
            b[k] = acc_b[i][k];
          }
      } else {
#pragma unroll
        for (int q = 0; q < P; q += 4) {
          *reinterpret_cast<float4*>(g + q) =
              make_float4(acc_g[i][q], acc_g[i][q + 1], acc_g[i][q + 2], acc_g[i][q + 3]);
          *reinterpret_cast<float4*>(b + q) =
              make_float4(acc_b[i][q], acc_b[i][q + 1], acc_b[i][q + 2], acc_b[i][q + 3]);
        }
      }
    }
    __syncthreads();
    if constexpr (RAGGED) {
      float* out = part + static_cast<int64_t>(blockIdx.x) * 2 * cols;
      for (int c = threadIdx.x; c < 2 * cols; c += WAVES * HK_WAVE) {
        float t = ldsf[c];
#pragma unroll
        for (int w = 1; w < SLOTS; ++w) t += ldsf[static_cast<int64_t>(w) * 2 * cols + c];
        out[c] = t;
      }
    } else {
      const int cols4 = cols / 4;
      float4* out = reinterpret_cast<float4*>(part) + static_cast<int64_t>(blockIdx.x) * 2 * cols4;
      for (int c = threadIdx.x; c < 2 * cols4; c += WAVES * HK_WAVE) {
        float4 s = lds4[c];
#pragma unroll
        for (int w = 1; w < SLOTS; ++w) {
          const float4 t = lds4[static_cast<int64_t>(w) * 2 * cols4 + c];
          s.x += t.x; s.y += t.y; s.z += t.z; s.w += t.w;
        }
        out[c] = s;
      }
    }
  }
}

// Sums nparts partials [nparts][2 * cols] in a fixed order and adds them into grad_gamma /
// grad_beta. A workgroup owns kFinCols columns and spreads the partials over kFinGroups lane
// groups: group g sums partials g, g + kFinGroups, ... (eight loads in flight per lane, one
// round for up to 256 partials), then the group sums are added in group order in LDS. Narrow
// column slices spread the read of the partials over 2 x cols / 16 workgroups.
constexpr int kFinCols = 16;
constexpr int kFinGroups = 32;
__global__ __launch_bounds__(kFinCols * kFinGroups) void ln_gb_finalize(
    const float* __restrict__ part, int nparts, int cols, float* __restrict__ grad_gamma,
    float* __restrict__ grad_beta) {
  __shared__ float red[kFinGroups][kFinCols];
  const int col = threadIdx.x % kFinCols;
  const int grp = threadIdx.x / kFinCols;
  const int c = blockIdx.x * kFinCols + col;
  const int width = 2 * cols;
  // The value this thread adds into is loaded before the partials, so its latency overlaps
  // theirs instead of following the reduction (4096 x 768 fp32 fused backward on MI355X:
  // 12.15 -> 11.84 us per call, same bits).
  float* dst = nullptr;
  if (grp == 0 && c < width) dst = c < cols ? (grad_gamma ? grad_gamma + c : nullptr)
                                            : (grad_beta ? grad_beta + (c - cols) : nullptr);
  const float prev = dst ? *dst : 0.f;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (c < width) {
    int p = grp;
    for (; p + 7 * kFinGroups < nparts; p += 8 * kFinGroups) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        acc[u] += part[static_cast<int64_t>(p + u * kFinGroups) * width + c];
    }
    for (; p < nparts; p += kFinGroups) acc[0] += part[static_cast<int64_t>(p) * width + c];
  }
  red[grp][col] = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
  __syncthreads();
  if (grp == 0 && c < width) {
    float s = red[0][col];
#pragma unroll
    for (int g = 1; g < kFinGroups; ++g) s += red[g][col];
    if (dst) *dst = prev + s;
  }
}

// Few rows: grad_x and the gamma/beta gradients in one launch. The first `row_groups` workgroups
// take one row per wave; each of the others owns kFinCols columns and sums them over every row (32
// row groups, added pairwise), reading dy and x a second time, from cache. Saves the partials'
// round trip and the finalize launch, which at 64 x 768 cost more than the second read.
template <typename T, int VPL, bool RAGGED>
__global__ __launch_bounds__(kFinCols * kFinGroups) void ln_bwd_few_rows(
    const St<T>* __restrict__ dy, const St<T>* __restrict__ x, const float* __restrict__ mean,
    const float* __restrict__ rstd, const St<T>* __restrict__ gamma, St<T>* __restrict__ dx,
    float* __restrict__ grad_gamma, float* __restrict__ grad_beta, int rows, int cols,
    float inv_cols, int row_groups) {
#pragma clang fp contract(off)
  using V = Vec<T, RAGGED>;
  constexpr int P = T::kPerVec;
  if (static_cast<int>(blockIdx.x) < row_groups) {
    const int nvec = (cols + P - 1) / P;
    const int lane = threadIdx.x & (HK_WAVE - 1);
    const int row = blockIdx.x * (kFinCols * kFinGroups / HK_WAVE) + (threadIdx.x >> 6);
    if (row >= rows) return;
    const St<T>* dyr = dy + static_cast<int64_t>(row) * cols;
    const St<T>* xr = x + static_cast<int64_t>(row) * cols;
    uint4 dv[VPL], xv[VPL];
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const int c = lane + i * HK_WAVE;
      dv[i] = c < nvec ? V::load(dyr, c, cols) : u4_zero();
      xv[i] = c < nvec ? V::load(xr, c, cols) : u4_zero();
    }
    const float m = mean[row], rs = rstd[row];
    auto widen = [&](int i, float* n, float* a) {
      const int c = lane + i * HK_WAVE;
      const int skip = RAGGED && c < nvec ? V::skip(c, cols) : 0;
      float d[P], g[P];
      T::unpack(dv[i], d);
      T::unpack(xv[i], n);
      affine<T, RAGGED>(gamma, c < nvec ? c : 0, cols, 1.f, g);
#pragma unroll
      for (int k = 0; k < P; ++k) {
        const bool own = c < nvec && (!RAGGED || k >= skip);
        n[k] = own ? (n[k] - m) * rs : 0.f;
        a[k] = own ? d[k] * g[k] : 0.f;
      }
    };
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      float n[P], a[P];
      widen(i, n, a);
      s1 += hk::tree_sum<P>(a);
#pragma unroll
      for (int k = 0; k < P; ++k) n[k] = a[k] * n[k];
      s2 += hk::tree_sum<P>(n);
    }
    const float t1 = hk::wave_sum(s1), t2 = hk::wave_sum(s2);
    St<T>* dxr = dx + static_cast<int64_t>(row) * cols;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const int c = lane + i * HK_WAVE;
      if (c < nvec) {
        float n[P], a[P], o[P];
        widen(i, n, a);
#pragma unroll
        for (int k = 0; k < P; ++k) o[k] = rs * (a[k] - (t1 + n[k] * t2) * inv_cols);
        V::store_nt(dxr, c, cols, o);
      }
    }
    return;
  }
  __shared__ float red[2][kFinGroups][kFinCols];
  const int col = threadIdx.x % kFinCols, grp = threadIdx.x / kFinCols;
  const int c = (blockIdx.x - row_groups) * kFinCols + col;
  // the values added into are loaded first, as in the finalize above
  const float* into = grp == 0 ? grad_gamma : grp == 1 ? grad_beta : nullptr;
  const float prev = into && c < cols ? into[c] : 0.f;
  float sg = 0.f, sb = 0.f;
  if (c < cols) {
#pragma unroll 4
    for (int r = grp; r < rows; r += kFinGroups) {
      const int64_t o = static_cast<int64_t>(r) * cols + c;
      const float d = T::load(dy, o);
      sg = __builtin_fmaf(d, (T::load(x, o) - mean[r]) * rstd[r], sg);
      sb += d;
    }
  }
  red[0][grp][col] = sg;
  red[1][grp][col] = sb;
  __syncthreads();
  if (grp < 2 && c < cols) {  // group 0: gamma, group 1: beta, each a pairwise sum of the groups
    float v[kFinGroups];
#pragma unroll
    for (int g = 0; g < kFinGroups; ++g) v[g] = red[grp][g][col];
    float* dst = grp == 0 ? grad_gamma : grad_beta;
    if (dst) dst[c] = prev + hk::tree_sum<kFinGroups>(v);
  }
}

// ------------------------------------------------------------------------------------------
// Fallback kernels (any cols, any alignment): one workgroup per row, row re-read from cache.
// ------------------------------------------------------------------------------------------
__device__ float block_sum(float v, float* red) {
  v = hk::wave_sum(v);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < kWavesPerBlock; ++w) t += red[w];
  return t;
}

template <typename T, typename S = typename T::storage>
__global__ __launch_bounds__(kThreads) void ln_fwd_rowblock(const S* __restrict__ x,
                                                            const S* __restrict__ gamma,
                                                            const S* __restrict__ beta,
                                                            S* __restrict__ y,
                                                            float* __restrict__ mean_out,
                                                            float* __restrict__ rstd_out,
                                                            int cols, float eps) {
  __shared__ float red[kWavesPerBlock];
  const int64_t row = blockIdx.x;
  const S* xr = x + row * cols;
  float s = 0.f;
  for (int c = threadIdx.x; c < cols; c += kThreads) s += T::load(xr, c);
  const float mu = block_sum(s, red) / static_cast<float>(cols);
  float q = 0.f;
  for (int c = threadIdx.x; c < cols; c += kThreads) {
    const float d = T::load(xr, c) - mu;
    q += d * d;
  }
  const float var = block_sum(q, red) / static_cast<float>(cols);
  const float rs = 1.0f / sqrtf(var + eps);
  if (threadIdx.x == 0) {
    if (mean_out) mean_out[row] = mu;
    if (rstd_out) rstd_out[row] = rs;
  }
  S* yr = y + row * cols;
  for (int c = threadIdx.x; c < cols; c += kThreads) {
    const float g = gamma ? T::load(gamma, c) : 1.f, b = beta ? T::load(beta, c) : 0.f;
    T::store(yr, c, (T::load(xr, c) - mu) * rs * g + b);
  }
}

template <typename T, typename S = typename T::storage>
__global__ __launch_bounds__(kThreads) void ln_bwd_input_rowblock(
    const S* __restrict__ dy, const S* __restrict__ x, const float* __restrict__ mean,
    const float* __restrict__ rstd, const S* __restrict__ gamma, S* __restrict__ dx, int cols) {
#pragma clang fp contract(off)
  __shared__ float red[kWavesPerBlock];
  const int64_t row = blockIdx.x;
  const float m = mean[row], rs = rstd[row];
  const S* dyr = dy + row * cols;
  const S* xr = x + row * cols;
  float s1 = 0.f, s2 = 0.f;
  for (int c = threadIdx.x; c < cols; c += kThreads) {
    const float a = T::load(dyr, c) * (gamma ? T::load(gamma, c) : 1.f);
    s1 += a;
    s2 += a * ((T::load(xr, c) - m) * rs);
  }
  const float t1 = block_sum(s1, red);
  const float t2 = block_sum(s2, red);
  const float ic = 1.0f / static_cast<float>(cols);
  S* dxr = dx + row * cols;
  for (int c = threadIdx.x; c < cols; c += kThreads) {
    const float n = (T::load(xr, c) - m) * rs;
    T::store(dxr, c, rs * (T::load(dyr, c) * (gamma ? T::load(gamma, c) : 1.f) - (t1 + n * t2) * ic));
  }
}

// Gamma/beta gradient of rows that the register path does not hold: a lane per column, the rows in
// gridDim.y slabs of `slab` rows, each summed in row order into part[slab][2 * cols] (gamma then
// beta) for ln_gb_finalize. One slab (gridDim.y == 1) adds into the gradients itself.
template <typename T, typename S = typename T::storage>
__global__ __launch_bounds__(kThreads) void ln_gb_slab(const S* __restrict__ dy,
                                                       const S* __restrict__ x,
                                                       const float* __restrict__ mean,
                                                       const float* __restrict__ rstd,
                                                       float* __restrict__ part,
                                                       float* __restrict__ grad_gamma,
                                                       float* __restrict__ grad_beta, int rows,
                                                       int cols, int slab) {
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c >= cols) return;
  const int r0 = blockIdx.y * slab, r1 = min(rows, r0 + slab);
  float sg = 0.f, sb = 0.f;
#pragma unroll 8
  for (int r = r0; r < r1; ++r) {
    const int64_t o = static_cast<int64_t>(r) * cols + c;
    const float d = T::load(dy, o);
    sg += d * ((T::load(x, o) - mean[r]) * rstd[r]);
    sb += d;
  }
  if (gridDim.y > 1) {
    float* out = part + static_cast<int64_t>(blockIdx.y) * 2 * cols;
    out[c] = sg;
    out[cols + c] = sb;
    return;
  }
  if (grad_gamma) grad_gamma[c] += sg;
  if (grad_beta) grad_beta[c] += sb;
}

// ------------------------------------------------------------------------------------------
// Dispatch helpers
// ------------------------------------------------------------------------------------------
int pick_vpl(int cols4) {
  static const int kVpl[] = {1, 2, 3, 4, 6, 8, 12, 16};
  for (int v : kVpl)
    if (cols4 <= v * HK_WAVE) return v;
  return 0;
}

template <typename F>
hipError_t with_vpl(int vpl, F&& f) {
  switch (vpl) {
    case 1: return f(std::integral_constant<int, 1>{});
    case 2: return f(std::integral_constant<int, 2>{});
    case 3: return f(std::integral_constant<int, 3>{});
    case 4: return f(std::integral_constant<int, 4>{});
    case 6: return f(std::integral_constant<int, 6>{});
    case 8: return f(std::integral_constant<int, 8>{});
    case 12: return f(std::integral_constant<int, 12>{});
    case 16: return f(std::integral_constant<int, 16>{});
    default: return hipErrorInvalidValue;
  }
}

// Rows of whole, 16-byte aligned vectors (else the RAGGED forms).
template <typename T>
bool vec_rows(int cols, std::initializer_list<const void*> ptrs) {
  if (cols % T::kPerVec != 0) return false;
  for (const void* p : ptrs)
    if (p && !hk::aligned16(p)) return false;
  return true;
}

// 16-byte vectors per lane of a row over `waves` waves; 0: no register path (longer than 16 per
// lane, or shorter than one vector).
template <typename T>
int row_vpl(int cols, int waves = 1) {
  if (cols < T::kPerVec) return 0;
  return pick_vpl(static_cast<int>(hk::ceil_div(hk::ceil_div(cols, T::kPerVec), waves)));
}

constexpr int kMaxGbCols = 2048;      // one wave per row with gamma/beta sums in registers
constexpr int kMaxWideCols = 4096;    // four waves per row
// Rows up to which both gradients come from one launch (ln_bwd_few_rows). Fused backward on MI355X,
// one launch against two, us per call back to back (a call costs its caller 3.4): 64 x 768 fp32 3.4
// against 6.9, 512 x 768 4.1 against 7.0, 300 x 4096 bf16 7.6 against 11.3.
constexpr int kFewRows = 512;
// The same for rows of more than kMaxWideCols columns, whose slabs are the other way (gradients alone,
// us, one launch against slabs: 20 x 8200 fp32 7.7 against 10.5, 100 x 8200 7.7 and 10.4, 512 x 8200 12.7
// and 10.0).
constexpr int kFewLongRows = 128;
template <typename T>
constexpr int kMaxFewVpl = T::kPerVec == 4 ? 12 : 8;  // fp32 rows of 16 vectors per lane spill
template <typename T>
constexpr int kMaxBwdVpl = 4096 / (HK_WAVE * T::kPerVec);

// Lets a kernel use `bytes` of dynamic LDS (set once per kernel, before its first launch).
template <auto Kernel>
hipError_t lds_limit(size_t bytes) {
  static std::once_flag once;
  static hipError_t status = hipSuccess;
  std::call_once(once, [bytes] {
    status = hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel),
                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                 static_cast<int>(bytes));
  });
  return status;
}

// Whether two arrays of n elements share memory.
template <typename S>
bool overlap(const S* a, const S* b, int64_t n) {
  const uintptr_t pa = reinterpret_cast<uintptr_t>(a), pb = reinterpret_cast<uintptr_t>(b);
  const uintptr_t bytes = static_cast<uintptr_t>(n) * sizeof(S);
  return pa < pb + bytes && pb < pa + bytes;
}

// Workgroups of a gamma/beta backward: one per `waves` rows, at most 8 / waves per CU.
int bwd_gb_grid(int rows, int waves) {
  const int64_t want = hk::ceil_div(rows, waves);
  const int64_t cap = static_cast<int64_t>(hk::device_cu_count()) * (8 / waves);
  return static_cast<int>(want < cap ? want : cap);
}

template <typename T>
hipError_t launch_fwd(const St<T>* x, const St<T>* gamma, const St<T>* beta, St<T>* y,
                      float* mean_out, float* rstd_out, int rows, int cols, float eps,
                      hipStream_t stream) {
  HK_CHECK_ARG(rows >= 0 && cols >= 0);
  if (rows == 0 || cols == 0) return hipSuccess;
  HK_CHECK_ARG(x && y);
  if (const int vpl = row_vpl<T>(cols)) {
    const bool vec = vec_rows<T>(cols, {x, gamma, beta, y});
    const unsigned grid = static_cast<unsigned>(hk::ceil_div(rows, kWavesPerBlock));
    const float inv_cols = 1.0f / static_cast<float>(cols);
    return with_vpl(vpl, [&](auto vpl_c) -> hipError_t {
      constexpr int V = decltype(vpl_c)::value;
      hipLaunchKernelGGL((vec ? ln_fwd_reg<T, V, false> : ln_fwd_reg<T, V, true>), dim3(grid),
                         dim3(kThreads), 0, stream, x, gamma, beta, y, mean_out, rstd_out, rows,
                         cols, inv_cols, eps);
      return hk::launch_status();
    });
  }
  hipLaunchKernelGGL(ln_fwd_rowblock<T>, dim3(rows), dim3(kThreads), 0, stream, x, gamma, beta, y,
                     mean_out, rstd_out, cols, eps);
  return hk::launch_status();
}

template <typename T>
using BwdKernel = void (*)(const St<T>*, const St<T>*, const float*, const float*, const St<T>*,
                           St<T>*, float*, int, int, float);

// The fused gamma/beta forms of the register path: kernel, workgroup and grid of a shape.
template <typename T>
struct GbForm {
  BwdKernel<T> kernel = nullptr;
  int waves = 0, grid = 0;
  size_t lds = 0;
};

template <typename T, bool RAGGED>
hipError_t gb_form(int rows, int cols, bool write_dx, GbForm<T>* out) {
  const int64_t cus = hk::device_cu_count();
  if (cols > kMaxGbCols) {
    // Four waves per row, four rows in flight per workgroup, one workgroup per CU, LDS for 4 x 2 x
    // cols floats (128 KiB at most). Fused backward on MI355X: 4096 x 2560 bf16 23.6 us (two waves
    // per row and 8 per workgroup 23.6, too: 34.4 against 31.0 at 4096 columns), fp32 29.3 us (31.4).
    // These rows ran a workgroup per row for grad_x and one lane per column over all rows for the
    // gradients, 1,278 and 1,235 us.
    return with_vpl(row_vpl<T>(cols, 4), [&](auto vpl_c) -> hipError_t {
      constexpr int V = decltype(vpl_c)::value;
      if constexpr (V * T::kPerVec > kMaxWideCols / (4 * HK_WAVE)) {
        return hipErrorInvalidValue;
      } else {
        constexpr int W = 16, kSlots = W / 4;
        constexpr size_t kLds = kSlots * 2 * kMaxWideCols * sizeof(float);
        const int64_t want = hk::ceil_div(rows, kSlots);
        constexpr auto dx_gb = ln_bwd_reg<T, V, true, true, W, true, RAGGED, 4>;
        constexpr auto gb = ln_bwd_reg<T, V, false, true, W, true, RAGGED, 4>;
        HK_RETURN_IF_ERROR(write_dx ? lds_limit<dx_gb>(kLds) : lds_limit<gb>(kLds));
        *out = GbForm<T>{write_dx ? dx_gb : gb, W, static_cast<int>(want < cus ? want : cus),
                         static_cast<size_t>(kSlots) * 2 * cols * sizeof(float)};
        return hipSuccess;
      }
    });
  }
  // The gamma/beta partials of one workgroup live in LDS: 8 (cols <= 1024) or 4 waves x 2 x
  // cols floats, kept within 64 KiB (cols <= kMaxGbCols); the one-row form's 16 waves take up
  // to 128 KiB (cols <= kOneRowMaxCols<T>).
  const bool one_row = !RAGGED && cols <= kOneRowMaxCols<T> && rows <= cus * kOneRowWaves;
  return with_vpl(row_vpl<T>(cols), [&](auto vpl_c) -> hipError_t {
    constexpr int V = decltype(vpl_c)::value;
    constexpr int kCols = V * HK_WAVE * T::kPerVec;  // the widest row of this VPL
    if constexpr (kCols > kMaxGbCols) {
      return hipErrorInvalidValue;
    } else {
      if constexpr (!RAGGED && kCols <= kOneRowMaxCols<T>) {
        if (one_row) {
          constexpr int W = kOneRowWaves;
          constexpr size_t kLds = W * 2 * kOneRowMaxCols<T> * sizeof(float);
          constexpr auto dx_gb = ln_bwd_reg<T, V, true, true, W, true>;
          constexpr auto gb = ln_bwd_reg<T, V, false, true, W, true>;
          HK_RETURN_IF_ERROR(write_dx ? lds_limit<dx_gb>(kLds) : lds_limit<gb>(kLds));
          *out = GbForm<T>{write_dx ? dx_gb : gb, W, static_cast<int>(hk::ceil_div(rows, W)),
                           static_cast<size_t>(W) * 2 * cols * sizeof(float)};
          return hipSuccess;
        }
      }
      // row_vpl takes the smallest VPL that holds the row, so cols <= 1024 exactly when
      // kCols <= 1024: the wave count is fixed by V
      constexpr int W = gb_waves(kCols);
      *out = GbForm<T>{write_dx ? ln_bwd_reg<T, V, true, true, W, false, RAGGED>
                                : ln_bwd_reg<T, V, false, true, W, false, RAGGED>,
                       W, bwd_gb_grid(rows, W), static_cast<size_t>(W) * 2 * cols * sizeof(float)};
      return hipSuccess;
    }
  });
}

template <typename T>
hipError_t launch_finalize(const float* part, int nparts, int cols, float* dgamma, float* dbeta,
                           hipStream_t stream) {
  hipLaunchKernelGGL(ln_gb_finalize, dim3(static_cast<unsigned>(hk::ceil_div(2 * cols, kFinCols))),
                     dim3(kFinCols * kFinGroups), 0, stream, part, nparts, cols, dgamma, dbeta);
  return hk::launch_status();
}

// grad_x alone.
template <typename T>
hipError_t launch_dx(const St<T>* dy, const St<T>* x, const float* mean, const float* rstd,
                     const St<T>* gamma, St<T>* dx, int rows, int cols, bool vec,
                     hipStream_t stream) {
  // The backward keeps dy, x and their prefetch in registers; past kMaxBwdVpl vectors per lane
  // (4096 columns for every storage type) it would spill, so wider rows take a workgroup per row.
  const int vpl = row_vpl<T>(cols);
  if (vpl == 0 || vpl > kMaxBwdVpl<T>) {
    hipLaunchKernelGGL(ln_bwd_input_rowblock<T>, dim3(rows), dim3(kThreads), 0, stream, dy, x,
                       mean, rstd, gamma, dx, cols);
    return hk::launch_status();
  }
  return with_vpl(vpl, [&](auto vpl_c) -> hipError_t {
    constexpr int V = decltype(vpl_c)::value;
    if constexpr (V > kMaxBwdVpl<T>) {
      return hipErrorInvalidValue;
    } else {
      constexpr int W = kWavesPerBlock;
      hipLaunchKernelGGL((vec ? ln_bwd_reg<T, V, true, false, W>
                              : ln_bwd_reg<T, V, true, false, W, false, true>),
                         dim3(static_cast<unsigned>(hk::ceil_div(rows, W))), dim3(W * HK_WAVE), 0,
                         stream, dy, x, mean, rstd, gamma, dx, static_cast<float*>(nullptr), rows,
                         cols, 1.0f / static_cast<float>(cols));
      return hk::launch_status();
    }
  });
}

// Few rows: `row_groups` workgroups of grad_x rows (0: the gradients alone) and those of the columns.
template <typename T>
hipError_t launch_few_rows(void (*kernel)(const St<T>*, const St<T>*, const float*, const float*,
                                          const St<T>*, St<T>*, float*, float*, int, int, float, int),
                           const St<T>* dy, const St<T>* x, const float* mean, const float* rstd,
                           const St<T>* gamma, St<T>* dx, float* dgamma, float* dbeta, int rows,
                           int cols, int row_groups, hipStream_t stream) {
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(row_groups + hk::ceil_div(cols, kFinCols))),
                     dim3(kFinCols * kFinGroups), 0, stream, dy, x, mean, rstd, gamma, dx, dgamma,
                     dbeta, rows, cols, 1.0f / static_cast<float>(cols), row_groups);
  return hk::launch_status();
}

template <typename T>
hipError_t launch_bwd(const St<T>* dy, const St<T>* x, const float* mean, const float* rstd,
                      const St<T>* gamma, St<T>* dx, float* dgamma, float* dbeta, int rows,
                      int cols, bool write_dx, bool do_gb, hipStream_t stream) {
  HK_CHECK_ARG(rows >= 0 && cols >= 0);
  if (rows == 0 || cols == 0) return hipSuccess;
  HK_CHECK_ARG(dy && x && mean && rstd);
  HK_CHECK_ARG(!write_dx || dx);
  const bool vec = vec_rows<T>(cols, {dy, x, gamma, dx});
  // grad_x may be dy or x itself. The register forms load a row before they store it, and the
  // workgroup-per-row form reads and writes an element in the same lane; ln_bwd_few_rows reads whole
  // columns while other workgroups store rows, and the slabs read after a grad_x launch of their own
  // would, so the first is left out for such calls and the second run before it.
  const int64_t n = static_cast<int64_t>(rows) * cols;
  const bool in_place = write_dx && (overlap(dx, dy, n) || overlap(dx, x, n));
  if (!do_gb) return launch_dx<T>(dy, x, mean, rstd, gamma, dx, rows, cols, vec, stream);
  const int vpl = row_vpl<T>(cols);
  const float inv_cols = 1.0f / static_cast<float>(cols);
  if (rows <= kFewRows && write_dx && vpl > 0 && vpl <= kMaxFewVpl<T> && !in_place) {
    const int row_groups = static_cast<int>(hk::ceil_div(rows, kFinCols * kFinGroups / HK_WAVE));
    return with_vpl(vpl, [&](auto vpl_c) -> hipError_t {
      constexpr int V = decltype(vpl_c)::value;
      if constexpr (V > kMaxFewVpl<T>) {
        return hipErrorInvalidValue;
      } else {
        return launch_few_rows<T>(vec ? ln_bwd_few_rows<T, V, false> : ln_bwd_few_rows<T, V, true>,
                                  dy, x, mean, rstd, gamma, dx, dgamma, dbeta, rows, cols,
                                  row_groups, stream);
      }
    });
  }
  // The gradients of few rows alone, of any length, since no row is held; rows of less than a vector get
  // their grad_x from a second launch (it may be written over dy or x).
  const int few = cols > kMaxWideCols ? kFewLongRows : kFewRows;
  if (rows <= few && (!write_dx || cols < T::kPerVec)) {
    HK_RETURN_IF_ERROR(launch_few_rows<T>(ln_bwd_few_rows<T, 1, false>, dy, x, mean, rstd, gamma, dx,
                                          dgamma, dbeta, rows, cols, 0, stream));
    if (write_dx) return launch_dx<T>(dy, x, mean, rstd, gamma, dx, rows, cols, vec, stream);
    return hipSuccess;
  }
  // Whole vectors of up to kMaxGbCols columns have always used the stream's workspace. The other
  // shapes do without it while a graph is being captured: the graph would keep its address, and a
  // later call may grow it.
  const bool capturing = (!vec || cols > kMaxGbCols) && hk::stream_capturing(stream);
  if (cols >= T::kPerVec && cols <= kMaxWideCols && !capturing) {
    GbForm<T> f;
    HK_RETURN_IF_ERROR(vec ? (gb_form<T, false>(rows, cols, write_dx, &f))
                           : (gb_form<T, true>(rows, cols, write_dx, &f)));
    void* ws = nullptr;
    HK_RETURN_IF_ERROR(hk::device_workspace(static_cast<size_t>(f.grid) * 2 * cols * sizeof(float),
                                            stream, &ws));
    float* part = static_cast<float*>(ws);
    hipLaunchKernelGGL(f.kernel, dim3(f.grid), dim3(f.waves * HK_WAVE), f.lds, stream, dy, x, mean,
                       rstd, gamma, dx, part, rows, cols, inv_cols);
    HK_RETURN_IF_ERROR(hk::launch_status());
    return launch_finalize<T>(part, f.grid, cols, dgamma, dbeta, stream);
  }
  // slabs of at least 16 rows, at most four workgroups per CU
  const int64_t blocks = hk::ceil_div(cols, kThreads);
  int64_t nslab = capturing ? 1 : hk::ceil_div(4 * static_cast<int64_t>(hk::device_cu_count()), blocks);
  if (nslab > hk::ceil_div(rows, 16)) nslab = hk::ceil_div(rows, 16);
  const int slab = static_cast<int>(hk::ceil_div(rows, nslab));
  nslab = hk::ceil_div(rows, slab);
  float* part = nullptr;
  if (nslab > 1) {
    void* ws = nullptr;
    HK_RETURN_IF_ERROR(hk::device_workspace(static_cast<size_t>(nslab) * 2 * cols * sizeof(float),
                                            stream, &ws));
    part = static_cast<float*>(ws);
  }
  hipLaunchKernelGGL(ln_gb_slab<T>,
                     dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(nslab)),
                     dim3(kThreads), 0, stream, dy, x, mean, rstd, part, dgamma, dbeta, rows, cols,
                     slab);
  HK_RETURN_IF_ERROR(hk::launch_status());
  if (nslab > 1)
    HK_RETURN_IF_ERROR(
        launch_finalize<T>(part, static_cast<int>(nslab), cols, dgamma, dbeta, stream));
  if (write_dx) return launch_dx<T>(dy, x, mean, rstd, gamma, dx, rows, cols, vec, stream);
  return hipSuccess;
}

}  // namespace

// One set of four entry points per storage type: fp32 (the float kernels), and the
// reference's __half / __nv_bfloat16 instantiations (layer_norm_forward_sm89_kernel.cu:205-210;
// ln_backward_input_sm89_kernel.cu:107-113; ln_backward_gamma_beta_sm89_kernel.cu:51-56).
#define HK_LN_ENTRY_POINTS(SUFFIX, TAG, S)                                                       \
  extern "C" hipError_t hk_layer_norm_forward_##SUFFIX(const S* x, const S* gamma,              \
                                                       const S* beta, S* y, float* mean_out,    \
                                                       float* rstd_out, int rows, int cols,     \
                                                       float eps, hipStream_t stream) {         \
    return launch_fwd<TAG>(x, gamma, beta, y, mean_out, rstd_out, rows, cols, eps, stream);     \
  }                                                                                             \
  extern "C" hipError_t hk_ln_backward_input_##SUFFIX(const S* grad_y, const S* x,              \
                                                      const float* mean, const float* rstd,     \
                                                      const S* gamma, S* grad_x, int rows,      \
                                                      int cols, hipStream_t stream) {           \
    return launch_bwd<TAG>(grad_y, x, mean, rstd, gamma, grad_x, nullptr, nullptr, rows, cols,  \
                           true, false, stream);                                                \
  }                                                                                             \
  extern "C" hipError_t hk_ln_backward_gamma_beta_##SUFFIX(                                     \
      const S* grad_y, const S* x, const float* mean, const float* rstd, float* grad_gamma,     \
      float* grad_beta, int rows, int cols, hipStream_t stream) {                               \
    HK_CHECK_ARG(grad_gamma || grad_beta || rows == 0 || cols == 0);                            \
    return launch_bwd<TAG>(grad_y, x, mean, rstd, nullptr, nullptr, grad_gamma, grad_beta, rows, \
                           cols, false, true, stream);                                          \
  }                                                                                             \
  extern "C" hipError_t hk_layer_norm_backward_##SUFFIX(                                        \
      const S* grad_y, const S* x, const float* mean, const float* rstd, const S* gamma,        \
      S* grad_x, float* grad_gamma, float* grad_beta, int rows, int cols, hipStream_t stream) { \
    return launch_bwd<TAG>(grad_y, x, mean, rstd, gamma, grad_x, grad_gamma, grad_beta, rows,   \
                           cols, true, grad_gamma || grad_beta, stream);                        \
  }

HK_LN_ENTRY_POINTS(f32, hk::F32, float)
HK_LN_ENTRY_POINTS(bf16, hk::BF16, hk_bf16)
HK_LN_ENTRY_POINTS(f16, hk::F16, hk_f16)
