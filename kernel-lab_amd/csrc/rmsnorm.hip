// RMSNorm and fused residual-add + RMSNorm for gfx950.
//
// Math (reference: csrc/rmsnorm.cu:17-62 and kernel_lab/reference.py:13-30):
//   res = dtype(f32(x) + f32(res))                  (fused variant only)
//   rstd = 1 / sqrt(sum(f32(res)^2) / hidden + eps)
//   out = dtype((f32(res) * rstd) * f32(weight))
// The sum is rounded to the storage dtype before it is normalised, because
// that rounded value is what the residual stream keeps; the residual output is
// therefore bit-identical to PyTorch's.
//
// Design: one workgroup per row, several rows per workgroup where a row is
// narrow. Each thread loads its share of the row as 16-byte packs, strided by
// the row's threads so every wave load is contiguous, and keeps the values in
// registers. The sum of squares is reduced within each wave by DPP, across
// waves (if the row has several) through LDS with one barrier, and the output
// is written from registers: one read of x and the residual, one write of the
// residual and the output, nothing re-read.
//   rms_norm_reg_kernel     wide rows, 16-byte aligned
//   rms_norm_rows_kernel    narrow rows: a row per 4 .. 64 lanes
//   rms_norm_ragged_kernel  wide rows at any address and width
//   rms_norm_staged_kernel  rows too wide for the register budget: two passes,
//                           the rounded sum kept in LDS (and formed again for
//                           what LDS cannot hold)
#include <algorithm>
#include <type_traits>

#include "hip_common.h"
#include "kl_internal.h"

namespace kl {
namespace {

template <typename S, int N>
struct alignas(sizeof(S) * N) Pack {
  S v[N];
};

// Pack loads and stores keep the default cache policy: measured on MI355X for
// this read/write mix, non-temporal stores lose ~10% of HBM bandwidth and
// non-temporal loads ~7%.
template <typename S, int N>
__device__ __forceinline__ Pack<S, N> load_pack(const Pack<S, N>* p) {
  return *p;
}

// Packs per thread the launch aims for (threads = packs / 2, in whole waves,
// 64..1024): measured on MI355X at hidden 8192 bf16, one, four and eight
// 16-byte packs per tensor per thread were slower than two.
constexpr int kPacksPerThread = 2;

template <typename S, int N>
__device__ __forceinline__ void store_pack(Pack<S, N>* p, const Pack<S, N>& v) {
  *p = v;
}

constexpr int kMaxThreads = 1024;

// Where x's rows are, in elements: row i of group g at g * group_stride + i *
// row_stride, inner rows to a group; out and the residuals hold row g * inner +
// i there. A strided view of two leading dimensions (the heads of one part of a
// fused projection) is read in place; copied first, 2,048 x 32 heads of 128
// bf16 took 15.7 us a call, the copy 9.7 of them, and 6.9 read in place (calls back
// to back; the kernel alone traces at 7.3 with the profiler's gaps).
//
// A workgroup per row takes (i, g) from the grid, the larger of the two counts
// along x: a division before the first load cost the large sizes 2 %.
struct RowMap {
  int64_t inner, row_stride, group_stride;
  int swapped;  // the grid's x counts groups
  __device__ __forceinline__ void of_workgroup(int64_t* row, int64_t* x_off) const {
    const int64_t i = swapped ? blockIdx.y : blockIdx.x;
    const int64_t g = swapped ? blockIdx.x : blockIdx.y;
    *row = g * inner + i;
    *x_off = g * group_stride + i * row_stride;
  }
  __device__ __forceinline__ int64_t x_of_row(int64_t r) const {
    if (group_stride == 0) return r * row_stride;  // one group
    const uint32_t g = static_cast<uint32_t>(r) / static_cast<uint32_t>(inner);
    return g * group_stride + (r - g * inner) * row_stride;
  }
};

__device__ __forceinline__ float inv_rms(float sum_sq, int hidden, float eps) {
  // Division and square root are IEEE-rounded here (no fast-math), matching
  // torch.rsqrt on the CPU, which computes 1 / sqrt(x).
  return 1.0f / sqrtf(sum_sq / static_cast<float>(hidden) + eps);
}

// The new residual's place, `bytes` past the old one's: 0 in place. Reached
// from the same pointer, so that pointer can be __restrict__ in both forms
// (without it the large sizes lost 1 %: the weights' loads went ahead of the
// residual's).
template <typename S>
__device__ __forceinline__ S* residual_out(S* res, int64_t bytes) {
  return reinterpret_cast<S*>(reinterpret_cast<char*>(res) + bytes);
}

// The 16 bytes at element offset `off` of a row. Unaligned rows (any element
// alignment) use the same 16-byte memory instructions, which gfx950 takes at
// any address.
template <bool ALIGNED, typename P, typename S>
__device__ __forceinline__ P load_at(const S* row, int off) {
  P v;
  if constexpr (ALIGNED) {
    v = *reinterpret_cast<const P*>(row + off);
  } else {
    __builtin_memcpy(&v, row + off, sizeof(P));
  }
  return v;
}
template <bool ALIGNED, typename P, typename S>
__device__ __forceinline__ void store_at(S* row, int off, const P& v) {
  if constexpr (ALIGNED) {
    *reinterpret_cast<P*>(row + off) = v;
  } else {
    __builtin_memcpy(row + off, &v, sizeof(P));
  }
}

// One thread's share of a row: packs t, t + nt, ..., NPACK of them, held in
// registers. reduce(v) sums v over the row's threads. live false: a row past
// the last, loaded like the last and not stored.
//
// ALIGNED: every row starts on 16 bytes and holds whole packs. Otherwise the
// last pack is the row's last VEC elements, which overlap the pack before it
// when the width is not a multiple of VEC: it leaves those elements out of the
// sum and writes the same values to them. The residual may be updated in place
// (res_out 0), so without ALIGNED it is stored after the reduction, which
// every thread of the row reaches with its loads done.
template <typename E, int VEC, int NPACK, bool HAS_RES, bool ALIGNED, typename Reduce>
__device__ __forceinline__ void norm_row(typename E::S* out, const typename E::S* x, typename E::S* res,
                                         int64_t res_out, const typename E::S* weight, int hidden, float eps,
                                         int t, int nt, bool live, Reduce&& reduce) {
  using S = typename E::S;
  using P = Pack<S, VEC>;
  const int packs = ALIGNED ? hidden / VEC : (hidden + VEC - 1) / VEC;
  int off[NPACK];
  int skip[NPACK];  // leading elements of the pack that the one before it holds
  bool valid[NPACK];
#pragma unroll
  for (int k = 0; k < NPACK; ++k) {
    const int p = t + k * nt;
    valid[k] = p < packs;
    const int at = (valid[k] ? p : packs - 1) * VEC;
    off[k] = ALIGNED ? at : min(at, hidden - VEC);
    skip[k] = at - off[k];
  }
  P a[NPACK], b[NPACK], w[NPACK];
#pragma unroll
  for (int k = 0; k < NPACK; ++k) {
    a[k] = load_at<ALIGNED, P>(x, off[k]);
    if constexpr (HAS_RES) b[k] = load_at<ALIGNED, P>(res, off[k]);
  }
  // At most four packs: the weights travel through the reduction.
#pragma unroll
  for (int k = 0; k < NPACK; ++k) w[k] = load_at<ALIGNED, P>(weight, off[k]);
  float sum_sq = 0.0f;
#pragma unroll
  for (int k = 0; k < NPACK; ++k) {
    float part = 0.0f;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      if constexpr (HAS_RES) a[k].v[j] = E::from_f32(E::to_f32(a[k].v[j]) + E::to_f32(b[k].v[j]));
      const float f = E::to_f32(a[k].v[j]);
      part += ALIGNED || j >= skip[k] ? f * f : 0.0f;
    }
    sum_sq += valid[k] ? part : 0.0f;
  }
  if constexpr (HAS_RES && ALIGNED) {
#pragma unroll
    for (int k = 0; k < NPACK; ++k) {
      if (valid[k] && live) store_at<ALIGNED>(residual_out(res, res_out), off[k], a[k]);
    }
  }
  const float rstd = inv_rms(reduce(sum_sq), hidden, eps);
  if constexpr (HAS_RES && !ALIGNED) {
#pragma unroll
    for (int k = 0; k < NPACK; ++k) {
      if (valid[k] && live) store_at<ALIGNED>(residual_out(res, res_out), off[k], a[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < NPACK; ++k) {
    P o;
#pragma unroll
    for (int j = 0; j < VEC; ++j) o.v[j] = E::from_f32((E::to_f32(a[k].v[j]) * rstd) * E::to_f32(w[k].v[j]));
    if (valid[k] && live) store_at<ALIGNED>(out, off[k], o);
  }
}

// Sum over the LANES (4 .. 64) lanes of a row, in every one of them.
template <int LANES>
__device__ __forceinline__ float lanes_sum(float v) {
  v += dpp<kDppQuadSwap1>(v);
  v += dpp<kDppQuadSwap2>(v);
  if constexpr (LANES >= 8) v += dpp<kDppRowHalfMirror>(v);  // the quads of each half row agree, so a mirror is a swap
  if constexpr (LANES >= 16) v += dpp<kDppRowRor8>(v);
  if constexpr (LANES >= 32) v = sum_xor16(v);
  if constexpr (LANES >= 64) v = sum_xor32(v);
  return v;
}

// Workgroup-wide sum; every thread receives the same value. `scratch` holds one
// float per wave. Wave sums are added in wave order, so the result is
// deterministic.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const float w = wave_sum(v);
  const int nw = blockDim.x >> 6;
  if (__lane_id() == 0) scratch[threadIdx.x >> 6] = w;
  __syncthreads();
  float total = 0.0f;
  for (int i = 0; i < nw; ++i) total += scratch[i];
  return total;
}

// Register-resident single pass. Thread t owns packs t, t + NT, ..., so NPACK
// loads per tensor per thread; NT * NPACK * VEC >= hidden. Every load is
// issued unconditionally (indexes past the row are clamped to its last pack
// and their values masked to zero), so all of a thread's loads are in flight
// together; a branch per pack would make the compiler wait for each load
// before issuing the next. Only stores are guarded.
template <typename E, int VEC, int NPACK, bool HAS_RES>
__global__ void __launch_bounds__(kMaxThreads)
    rms_norm_reg_kernel(typename E::S* __restrict__ out, const typename E::S* __restrict__ x,
                        typename E::S* __restrict__ res, int64_t res_out, const typename E::S* __restrict__ weight,
                        int hidden, RowMap x_rows, float eps) {
  using S = typename E::S;
  using P = Pack<S, VEC>;
  __shared__ float scratch[kMaxThreads / 64];

  int64_t row, x_off;
  x_rows.of_workgroup(&row, &x_off);
  const int packs = hidden / VEC;
  const int nt = blockDim.x;
  const P* xr = reinterpret_cast<const P*>(x + x_off);
  P* rr = HAS_RES ? reinterpret_cast<P*>(res + row * static_cast<int64_t>(hidden)) : nullptr;
  P* rw = HAS_RES ? residual_out(rr, res_out) : nullptr;
  P* orow = reinterpret_cast<P*>(out + row * static_cast<int64_t>(hidden));
  const P* wr = reinterpret_cast<const P*>(weight);

  int idx[NPACK];
  bool valid[NPACK];
#pragma unroll
  for (int k = 0; k < NPACK; ++k) {
    const int p = threadIdx.x + k * nt;
    valid[k] = p < packs;
    idx[k] = valid[k] ? p : packs - 1;
  }

  P a[NPACK];
  P b[NPACK];
#pragma unroll
  for (int k = 0; k < NPACK; ++k) {
    a[k] = load_pack(xr + idx[k]);
    if constexpr (HAS_RES) b[k] = load_pack(rr + idx[k]);
  }
  // Weights are loaded before the reduction so their latency overlaps it,
  // except at NPACK = 8, where their registers beside x's and the residual's
  // would exceed the 128 a lane has at 1024 threads and spill.
  constexpr bool kEarlyWeights = NPACK <= 4;
  P w[NPACK];
  if constexpr (kEarlyWeights) {
#pragma unroll
    for (int k = 0; k < NPACK; ++k) w[k] = wr[idx[k]];
  }

  // The rounded sum stays packed across the block reduction and is widened
  // again for the output: keeping an fp32 copy live as well would need
  // NPACK * VEC more registers and spill at NPACK = 8.
  P s[NPACK];
  float sum_sq = 0.0f;
#pragma unroll
  for (int k = 0; k < NPACK; ++k) {
    if constexpr (HAS_RES) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) s[k].v[j] = E::from_f32(E::to_f32(a[k].v[j]) + E::to_f32(b[k].v[j]));
    } else {
      s[k] = a[k];
    }
    float part = 0.0f;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float f = E::to_f32(s[k].v[j]);
      part += f * f;
    }
    sum_sq += valid[k] ? part : 0.0f;
  }
  if constexpr (HAS_RES) {
#pragma unroll
    for (int k = 0; k < NPACK; ++k) {
      if (valid[k]) store_pack(rw + idx[k], s[k]);
    }
  }

  if constexpr (!kEarlyWeights) {
#pragma unroll
    for (int k = 0; k < NPACK; ++k) w[k] = wr[idx[k]];
  }
  const float rstd = inv_rms(block_sum(sum_sq, scratch), hidden, eps);
  if constexpr (!kEarlyWeights && sizeof(P) == 16) {
    // Keep the sums packed until here: widened ahead of the reduction (the
    // compiler's choice otherwise) they would take twice the registers.
#pragma unroll
    for (int k = 0; k < NPACK; ++k) {
      u32x4 r = __builtin_bit_cast(u32x4, s[k]);
      asm volatile("" : "+v"(r));
      s[k] = __builtin_bit_cast(P, r);
    }
  }

#pragma unroll
  for (int k = 0; k < NPACK; ++k) {
    P o;
#pragma unroll
    for (int j = 0; j < VEC; ++j) o.v[j] = E::from_f32((E::to_f32(s[k].v[j]) * rstd) * E::to_f32(w[k].v[j]));
    if (valid[k]) store_pack(orow + idx[k], o);
  }
}

// Rows wider than the register-resident kernel holds (more than 8 packs per
// thread at 1024 threads, 4 unaligned: 65,536 16-bit or 32,768 fp32 elements
// aligned, half of them unaligned). Two passes over the row with the rounded sum kept in LDS:
//   pass 1  reads x (and the residual), forms the rounded sum, accumulates its
//           squares, and keeps the sum of the row's first kStagedPacks packs in
//           LDS (writing their residual now);
//   pass 2  normalises from LDS; packs beyond the LDS window are formed again
//           from x and the residual, whose original value is still in memory
//           because pass 1 did not write those packs, and their residual is
//           written then.
// A thread takes the same packs in both passes, so neither pass waits for
// another thread beyond the reduction's barrier; the squares are summed in the
// same order either way, so the bits do not depend on the LDS window.
constexpr int kStageBytes = 48 * 1024;

template <typename E, int VEC, bool HAS_RES>
__global__ void __launch_bounds__(kMaxThreads)
    rms_norm_staged_kernel(typename E::S* __restrict__ out, const typename E::S* __restrict__ x,
                           typename E::S* __restrict__ res, int64_t res_out,
                           const typename E::S* __restrict__ weight, int hidden, RowMap x_rows, float eps) {
  using S = typename E::S;
  using P = Pack<S, VEC>;
  constexpr int kStagedPacks = kStageBytes / static_cast<int>(sizeof(P));
  __shared__ P staged[kStagedPacks];
  __shared__ float scratch[kMaxThreads / 64];

  int64_t row, x_off;
  x_rows.of_workgroup(&row, &x_off);
  const int packs = hidden / VEC;
  const int window = min(packs, kStagedPacks);
  const P* xr = reinterpret_cast<const P*>(x + x_off);
  P* rr = HAS_RES ? reinterpret_cast<P*>(res + row * static_cast<int64_t>(hidden)) : nullptr;
  P* rw = HAS_RES ? residual_out(rr, res_out) : nullptr;
  P* orow = reinterpret_cast<P*>(out + row * static_cast<int64_t>(hidden));
  const P* wr = reinterpret_cast<const P*>(weight);

  // The value the residual stream carries for pack p: dtype(x + residual), or x.
  auto rounded_sum = [&](int p) {
    P v = xr[p];
    if constexpr (HAS_RES) {
      const P r = rr[p];
#pragma unroll
      for (int j = 0; j < VEC; ++j) v.v[j] = E::from_f32(E::to_f32(v.v[j]) + E::to_f32(r.v[j]));
    }
    return v;
  };

  float sum_sq = 0.0f;
  for (int p = threadIdx.x; p < packs; p += blockDim.x) {
    const P v = rounded_sum(p);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float f = E::to_f32(v.v[j]);
      sum_sq += f * f;
    }
    if (p < window) {
      staged[p] = v;
      if constexpr (HAS_RES) rw[p] = v;
    }
  }
  const float rstd = inv_rms(block_sum(sum_sq, scratch), hidden, eps);

  for (int p = threadIdx.x; p < packs; p += blockDim.x) {
    P v;
    if (p < window) {
      v = staged[p];
    } else {
      v = rounded_sum(p);
      if constexpr (HAS_RES) rw[p] = v;
    }
    const P g = wr[p];
    P o;
#pragma unroll
    for (int j = 0; j < VEC; ++j) o.v[j] = E::from_f32((E::to_f32(v.v[j]) * rstd) * E::to_f32(g.v[j]));
    orow[p] = o;
  }
}

// Rows of at most kRowsMaxPacks packs: LANES lanes per row and 256 / LANES rows
// per workgroup, so a narrow row neither leaves lanes idle nor costs a
// workgroup of its own, and the reduction stays in a wave (no barrier). What
// bounds it: memory for many rows, the launch for few. Measured, a workgroup
// per row -> this (us, bf16): 65,536 rows of 128 16.9 -> 6.9 (4.9 TB/s), of 64
// 16.6 -> 4.6, 16,384 rows of 512 7.2 -> 6.8; 16 rows of 128 equal.
constexpr int kRowsThreads = 256;

template <typename E, int LANES, bool HAS_RES, bool ALIGNED>
__global__ void __launch_bounds__(kRowsThreads)
    rms_norm_rows_kernel(typename E::S* __restrict__ out, const typename E::S* __restrict__ x,
                         typename E::S* __restrict__ res, int64_t res_out, const typename E::S* __restrict__ weight,
                         int rows, int hidden, RowMap x_rows, float eps) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * (kRowsThreads / LANES) + threadIdx.x / LANES;
  const bool live = r < rows;
  const int64_t row = live ? r : rows - 1;
  norm_row<E, 16 / E::kBytes, 1, HAS_RES, ALIGNED>(
      out + row * hidden, x + x_rows.x_of_row(row), HAS_RES ? res + row * hidden : nullptr,
      res_out, weight, hidden, eps, threadIdx.x % LANES, LANES, live, [](float v) { return lanes_sum<LANES>(v); });
}

// Wide rows whose width or addresses are not multiples of 16 bytes: one
// workgroup per row on unaligned 16-byte accesses, in place of element-wide
// ones. Memory bounds it. Measured, element-wide -> this (us): add + norm 4,096
// rows of 5,003 bf16 54.5 -> 35.4, 2,048 of 4,099 fp32 30.7 -> 24.8, norm of
// 2,048 of 4,099 fp16 12.1 -> 8.8.
template <typename E, int NPACK, bool HAS_RES>
__global__ void __launch_bounds__(kMaxThreads)
    rms_norm_ragged_kernel(typename E::S* __restrict__ out, const typename E::S* __restrict__ x,
                           typename E::S* __restrict__ res, int64_t res_out,
                           const typename E::S* __restrict__ weight, int hidden, RowMap x_rows, float eps) {
  __shared__ float scratch[kMaxThreads / 64];
  int64_t row, x_off;
  x_rows.of_workgroup(&row, &x_off);
  norm_row<E, 16 / E::kBytes, NPACK, HAS_RES, false>(
      out + row * hidden, x + x_off, HAS_RES ? res + row * hidden : nullptr,
      res_out, weight, hidden, eps, threadIdx.x, blockDim.x, true, [&](float v) { return block_sum(v, scratch); });
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Calls f(IntC<N>) with the smallest N of 2, 4, 8 that holds npack (a row of one
// pack per thread is narrow enough for rms_norm_rows_kernel).
template <int N>
using IntC = std::integral_constant<int, N>;
template <typename F>
void with_packs(int npack, F&& f) {
  if (npack <= 2) {
    f(IntC<2>{});
  } else if (npack <= 4) {
    f(IntC<4>{});
  } else {
    f(IntC<8>{});
  }
}

// Widest row, in packs, that rms_norm_rows_kernel takes: a pack per lane of one
// wave. With two packs a lane it lost to a workgroup per row (8,192 rows of
// 1,024 bf16: 7.5 against 6.7 us).
constexpr int kRowsMaxPacks = 64;

template <typename E, bool HAS_RES>
int launch_typed(void* out, const void* x, const void* res, void* res_out, const void* w, int64_t rows, int hidden,
                 const RowMap& xm, float eps, hipStream_t stream) {
  using S = typename E::S;
  constexpr int VEC = 16 / E::kBytes;
  auto* o = static_cast<S*>(out);
  auto* xi = static_cast<const S*>(x);
  auto* r = static_cast<S*>(const_cast<void*>(res));  // read only, but for the in-place form
  const int64_t rw = reinterpret_cast<intptr_t>(res_out) - reinterpret_cast<intptr_t>(res);
  auto* wi = static_cast<const S*>(w);
  const bool aligned = hidden % VEC == 0 && xm.row_stride % VEC == 0 && xm.group_stride % VEC == 0 &&
                       aligned16(out) && aligned16(x) && aligned16(w) && aligned16(res) && aligned16(res_out);
  const int packs = static_cast<int>(cdiv(hidden, VEC));
  const auto gx = static_cast<unsigned>(xm.swapped ? rows / xm.inner : xm.inner);
  const dim3 grid(gx, static_cast<unsigned>(rows / gx));
  if (hidden < VEC) {  // less than a pack: element by element
    rms_norm_reg_kernel<E, 1, 1, HAS_RES><<<grid, 64, 0, stream>>>(o, xi, r, rw, wi, hidden, xm, eps);
    return check_launch("rms_norm kernel launch");
  }
  if (packs <= kRowsMaxPacks) {
    auto rows_kernel = [&](auto lanes) {
      constexpr int L = decltype(lanes)::value;
      const unsigned wgs = static_cast<unsigned>(cdiv(rows, kRowsThreads / L));
      if (aligned) {
        rms_norm_rows_kernel<E, L, HAS_RES, true><<<wgs, kRowsThreads, 0, stream>>>(
            o, xi, r, rw, wi, static_cast<int>(rows), hidden, xm, eps);
      } else {
        rms_norm_rows_kernel<E, L, HAS_RES, false><<<wgs, kRowsThreads, 0, stream>>>(
            o, xi, r, rw, wi, static_cast<int>(rows), hidden, xm, eps);
      }
    };
    if (packs <= 4) {
      rows_kernel(IntC<4>{});
    } else if (packs <= 8) {
      rows_kernel(IntC<8>{});
    } else if (packs <= 16) {
      rows_kernel(IntC<16>{});
    } else if (packs <= 32) {
      rows_kernel(IntC<32>{});
    } else {
      rows_kernel(IntC<64>{});
    }
    return check_launch("rms_norm kernel launch");
  }
  // About kPacksPerThread packs per thread, in whole waves, 64..1024 threads.
  const int threads = static_cast<int>(
      std::min<int64_t>(kMaxThreads, std::max<int64_t>(64, cdiv(cdiv(packs, kPacksPerThread), 64) * 64)));
  const int npack = static_cast<int>(cdiv(packs, threads));
  if (npack > (aligned ? 8 : 4)) {  // eight unaligned packs of x and the residual would spill
    if (aligned) {
      rms_norm_staged_kernel<E, VEC, HAS_RES>
          <<<grid, kMaxThreads, 0, stream>>>(o, xi, r, rw, wi, hidden, xm, eps);
    } else {
      rms_norm_staged_kernel<E, 1, HAS_RES>
          <<<grid, kMaxThreads, 0, stream>>>(o, xi, r, rw, wi, hidden, xm, eps);
    }
  } else {
    with_packs(npack, [&](auto np) {
      constexpr int NP = decltype(np)::value;
      if (aligned) {
        rms_norm_reg_kernel<E, VEC, NP, HAS_RES>
            <<<grid, threads, 0, stream>>>(o, xi, r, rw, wi, hidden, xm, eps);
      } else if constexpr (NP <= 4) {
        rms_norm_ragged_kernel<E, NP, HAS_RES>
            <<<grid, threads, 0, stream>>>(o, xi, r, rw, wi, hidden, xm, eps);
      }
    });
  }
  return check_launch("rms_norm kernel launch");
}

template <typename E>
int launch_any(void* out, const void* x, const void* res, void* res_out, const void* w, int64_t rows, int hidden,
               const RowMap& xm, float eps, hipStream_t stream) {
  return res ? launch_typed<E, true>(out, x, res, res_out, w, rows, hidden, xm, eps, stream)
             : launch_typed<E, false>(out, x, nullptr, nullptr, w, rows, hidden, xm, eps, stream);
}

}  // namespace
}  // namespace kl

extern "C" int kl_rms_norm_grouped(kl_dtype dtype, void* out, const void* x, const void* residual, void* residual_out,
                                   const void* weight, int64_t groups, int64_t rows_per_group, int64_t hidden,
                                   int64_t x_group_stride, int64_t x_row_stride, float eps, kl_stream_t stream) {
  using namespace kl;
  if (groups < 0 || rows_per_group < 0 || hidden < 0) {
    return fail(KL_ERR_INVALID_ARGUMENT, "rows and hidden must be >= 0");
  }
  if (groups == 0 || rows_per_group == 0 || hidden == 0) return ok();
  if (groups > 0x7fffffffLL || rows_per_group > 0x7fffffffLL || groups * rows_per_group > 0x7fffffffLL) {
    return fail(KL_ERR_UNSUPPORTED, "rows must be < 2^31");
  }
  if (hidden > 0x7fffffffLL) return fail(KL_ERR_UNSUPPORTED, "hidden must be < 2^31");
  if (out == nullptr || x == nullptr || weight == nullptr) {
    return fail(KL_ERR_INVALID_ARGUMENT, "out, x and weight must be non-null");
  }
  if ((residual == nullptr) != (residual_out == nullptr)) {
    return fail(KL_ERR_INVALID_ARGUMENT, "residual and residual_out go together");
  }
  if ((x_row_stride < hidden && rows_per_group > 1) || (x_group_stride < hidden && groups > 1)) {
    return fail(KL_ERR_INVALID_ARGUMENT, "x_row_stride and x_group_stride must be >= hidden");
  }
  const auto s = reinterpret_cast<hipStream_t>(stream);
  const int h = static_cast<int>(hidden);
  const int64_t rows = groups * rows_per_group;
  // One row per group, or one group: a single stride. The grid's y is at most
  // 65,535, which the smaller of two counts whose product is below 2^31 meets.
  const RowMap xm = groups == 1           ? RowMap{rows, x_row_stride, 0, 0}
                    : rows_per_group == 1 ? RowMap{rows, x_group_stride, 0, 0}
                                          : RowMap{rows_per_group, x_row_stride, x_group_stride, groups > rows_per_group};
  switch (dtype) {
    case KL_DTYPE_F32:
      return launch_any<F32>(out, x, residual, residual_out, weight, rows, h, xm, eps, s);
    case KL_DTYPE_F16:
      return launch_any<F16>(out, x, residual, residual_out, weight, rows, h, xm, eps, s);
    case KL_DTYPE_BF16:
      return launch_any<BF16>(out, x, residual, residual_out, weight, rows, h, xm, eps, s);
  }
  return fail(KL_ERR_UNSUPPORTED, "dtype must be f32, f16 or bf16");
}

extern "C" int kl_rms_norm(kl_dtype dtype, void* out, const void* x, void* residual, const void* weight,
                           int64_t rows, int64_t hidden, int64_t x_row_stride, float eps,
                           kl_stream_t stream) {
  return kl_rms_norm_grouped(dtype, out, x, residual, residual, weight, 1, rows, hidden, 0, x_row_stride, eps, stream);
}
