// kernels.hpp -- device building blocks shared by the operator and solver
// kernels: the sliced-ELLPACK row product, XCD-aware block mapping and
// deterministic block / grid reductions.
#pragma once

#include "internal.hpp"

namespace nosh {

template <class T>
using V2 = typename Vec2<T>::type;

// Meshes up to this many rows use P = 4, larger ones P = 2 (see RowBlock), in
// 2D (3 + 3 slots a row) as in 3D (7 + 7) and in FP32 as in FP64. A Newton step
// of 16 MINRES iterations, P = 4 | 2, in us:
//   rows                 FP64          FP32
//   10,201  (100^2)    595 |  636    615 |  668
//   68,921  (40^3)     772 |  862    781 |  809
//   90,601  (300^2)    753 |  746    762 |  747
//   91,125  (44^3)     857 |  893    839 |  830
//   117,649 (48^3)    1085 | 1031    921 |  908
//   160,801 (400^2)    985 |  874    961 |  822
//   491,401 (700^2)   2331 | 2218   1923 | 1646
//   912,673 (96^3)    5554 | 4935   3887 | 3514
constexpr int64_t kSplitRows = 90000;

// MI355X dispatches consecutive workgroups round-robin over its 8 XCDs.
// Remap so that XCD x processes one contiguous range of workgroup indices,
// keeping each XCD's gathers of x within its own L2.
__device__ __forceinline__ int64_t xcd_block(bool remap) {
  const int64_t b = blockIdx.x;
  if (!remap) return b;
  const int64_t nb = gridDim.x;
  const int64_t q = nb / 8, r = nb % 8;
  const int64_t xcd = b % 8, idx = b / 8;
  return xcd < r ? xcd * (q + 1) + idx : r * (q + 1) + (xcd - r) * q + idx;
}

__device__ __forceinline__ int32_t uniform(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Load of a value that no kernel writes, at a wave-uniform address, through
// the constant address space (a scalar load).
__device__ __forceinline__ int32_t ld_uniform(const int32_t* p) {
#if __HIP_DEVICE_COMPILE__
  return *reinterpret_cast<const __attribute__((address_space(4))) int32_t*>(
      reinterpret_cast<uintptr_t>(p));
#else
  return *p;  // host pass only parses device functions
#endif
}

// Row products of one workgroup of 256 threads. P waves share a 64-row slice:
// P = 4: two take its upper slots and two its lower ones (FP64: every other slot
// each; FP32: the first and the second half of them); P = 2: one takes the upper
// slots, one the lower ones. The first of them adds the sums (FP32: the terms,
// see sell_ordered) through LDS and owns the slice's rows. One wave a slice
// walks a chain of some twelve dependent loads (slot pointer, columns,
// gathers, first above then below the diagonal); P waves are P times as many,
// with a part of the chain each. A Newton step of 16 MINRES iterations (112
// products) with one, two and four waves a slice: 20^3 cube 878 / 746 / 664 us,
// 48^3 1310 / 1010 / 1126 us, 96^3 5997 / 5025 / 5597 us in FP64. Columns and
// positions are ordinary loads: as non-temporal ones they miss the Infinity
// Cache when the next product reads them again (96^3: 5219 us). Eight slots at
// a time instead of four: 6126 us.
//
// The slice's slot ranges come with the row, before anything that the kernel
// decides by a load (a solver's `done` flag): both loads are then under way
// together. FP64: the range of the wave's half; FP32: those of both halves
// (see sell_ordered).
template <class T, int P>
struct RowBlock {
  static constexpr int kSlices = 4 / P;  // per workgroup
  int64_t row;
  int part;    // of the slice, wave-uniform
  bool owner;  // this thread owns `row`
  int32_t beg[sizeof(T) == 4 ? 2 : 1], end[sizeof(T) == 4 ? 2 : 1];
  __device__ __forceinline__ RowBlock(int64_t n, const SellView& S) : beg{}, end{} {
    const int w = uniform(int(threadIdx.x >> 6));
    const int64_t slice = xcd_block(true) * kSlices + w / P;
    part = w % P;
    row = slice * kSliceH + (threadIdx.x & 63);
    owner = row < n && part == 0;
    if (slice * kSliceH < n) {
      const int32_t s = uniform(int32_t(slice));
      if constexpr (sizeof(T) == 4) {
        beg[0] = ld_uniform(S.uptr + s), end[0] = ld_uniform(S.uptr + s + 1);
        beg[1] = ld_uniform(S.lptr + s), end[1] = ld_uniform(S.lptr + s + 1);
      } else {
        const int32_t* p = part < P / 2 ? S.uptr : S.lptr;
        beg[0] = ld_uniform(p + s), end[0] = ld_uniform(p + s + 1);
      }
    }
  }
};

template <class T, bool OFF16, int P>
__device__ __forceinline__ V2<T> sell_part(const RowBlock<T, P>& rb, const SellView& S,
                                           const V2<T>* __restrict__ val,
                                           const V2<T>* __restrict__ x) {
  constexpr int H = P / 2;  // waves per half
  const int32_t r32 = int32_t(rb.row), b = rb.beg[0], e = rb.end[0];
  const int32_t first = kSliceH * (rb.part % H) + (r32 & 63);
  T ar = T(0), ai = T(0);
  if (rb.part < H) {
#pragma unroll 4
    for (int32_t j = b + first; j < e; j += H * kSliceH) {
      const int32_t c = OFF16 ? r32 + int32_t(S.uoff[j]) : S.ucol[j];
      const V2<T> v = val[j];
      const V2<T> xv = x[c];
      ar += v.x * xv.x - v.y * xv.y;
      ai += v.x * xv.y + v.y * xv.x;
    }
  } else {
#pragma unroll 4
    for (int32_t j = b + first; j < e; j += H * kSliceH) {
      const int32_t c = OFF16 ? r32 + int32_t(S.loff[j]) : S.lcol[j];
      const V2<T> v = val[S.lpos[j]];
      const V2<T> xv = x[c];
      ar += v.x * xv.x + v.y * xv.y;
      ai += v.x * xv.y - v.y * xv.x;
    }
  }
  V2<T> r;
  r.x = ar;
  r.y = ai;
  return r;
}

// The FP32 product of a slice's rows with its terms added in slot order, upper
// then lower, whatever P: the rounding of an FP32 solve, some 1e-8 of the state
// it updates, is then that of one wave a slice, to the bit, and P is free to
// follow the speed alone. The owner adds its own slots as it gathers them; the
// other waves leave up to kTerms terms in LDS, and slots beyond those (rows of
// more than twice that many slots) are the owner's as well.
// (53 x 41 x 47 box, two Newton steps: 1.80 ms with per-wave sums, 1.79 with
// these; the error against 64 bits moved by up to a factor of 5 either way from
// state to state with the former.)
template <bool OFF16>
__device__ __forceinline__ float2 sell_term(bool up, int32_t j, int32_t r32, const SellView& S,
                                            const float2* __restrict__ val,
                                            const float2* __restrict__ x) {
  const int32_t c = up ? (OFF16 ? r32 + int32_t(S.uoff[j]) : S.ucol[j])
                       : (OFF16 ? r32 + int32_t(S.loff[j]) : S.lcol[j]);
  const float2 v = val[up ? j : S.lpos[j]];
  const float2 xv = x[c];
  float2 t;
  if (up) {
    t.x = v.x * xv.x - v.y * xv.y;
    t.y = v.x * xv.y + v.y * xv.x;
  } else {
    t.x = v.x * xv.x + v.y * xv.y;
    t.y = v.x * xv.y - v.y * xv.x;
  }
  return t;
}

// The rows of a Kuhn cube have 7 + 7 slots, more about jittered or irregular
// vertices. Twice as many terms (24 KB of LDS with P = 4, 32 with P = 2) leave
// too few workgroups a CU: 16 iterations at 96^3 take 4523 us against 3512, at
// 700^2 2123 against 1645. Half as many: 3460 and 1626, but a half row of 9
// slots with P = 2 is then partly one wave's.
template <int P>
constexpr int kTerms = P == 4 ? 8 : 16;

template <bool OFF16, int P>
__device__ __forceinline__ float2 sell_ordered(const RowBlock<float, P>& rb, int64_t n,
                                               const SellView& S, const float2* __restrict__ val,
                                               const float2* __restrict__ x,
                                               float2 (&mine)[P - 1][kTerms<P>][kSliceH]) {
  const int lane = int(threadIdx.x & 63);
  const int32_t r32 = int32_t(rb.row);
  float2 acc = make_float2(0.f, 0.f);
  // Slots of part q: [from[q], to[q]) of its half.
  int32_t from[P] = {}, to[P] = {};
  if (rb.row < n) {
    const int32_t len[2] = {(rb.end[0] - rb.beg[0]) / kSliceH, (rb.end[1] - rb.beg[1]) / kSliceH};
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int32_t l = len[q / (P / 2)], cut = P == 4 ? (l + 1) / 2 : l;
      from[q] = P == 4 && (q & 1) ? cut : 0;
      to[q] = P == 4 && (q & 1) ? l : cut;
    }
#pragma unroll
    for (int q = 0; q < P; ++q) {
      if (rb.part != q) continue;
      const bool up = q < P / 2;
      const int32_t at = rb.beg[up ? 0 : 1] + lane;
      if (q == 0) {
#pragma unroll 4
        for (int32_t k = from[q]; k < to[q]; ++k) {
          const float2 t = sell_term<OFF16>(up, at + k * kSliceH, r32, S, val, x);
          acc.x += t.x;
          acc.y += t.y;
        }
      } else {
        const int32_t cnt = min(to[q] - from[q], kTerms<P>);
#pragma unroll 4
        for (int32_t k = 0; k < cnt; ++k)
          mine[q - 1][k][lane] =
              sell_term<OFF16>(up, at + (from[q] + k) * kSliceH, r32, S, val, x);
      }
    }
  }
  __syncthreads();
  if (rb.owner) {
#pragma unroll
    for (int q = 1; q < P; ++q) {
      const bool up = q < P / 2;
      const int32_t at = rb.beg[up ? 0 : 1] + lane, cnt = min(to[q] - from[q], kTerms<P>);
#pragma unroll 4
      for (int32_t k = 0; k < cnt; ++k) {
        const float2 t = mine[q - 1][k][lane];
        acc.x += t.x;
        acc.y += t.y;
      }
      for (int32_t k = from[q] + cnt; k < to[q]; ++k) {
        const float2 t = sell_term<OFF16>(up, at + k * kSliceH, r32, S, val, x);
        acc.x += t.x;
        acc.y += t.y;
      }
    }
  }
  return acc;
}

// Off-diagonal row product of rb.row, valid where rb.owner: upper slots, then
// lower slots conjugated at their mirrored positions (a gather that the
// neighbouring rows' waves have just brought into L2). The columns come as
// 16-bit offsets from the row when the layout has them (2 bytes a slot
// instead of 4), else as 32-bit indices. Every thread of the workgroup calls
// it (there is a barrier).
template <class T, int P>
__device__ __forceinline__ V2<T> row_product(const RowBlock<T, P>& rb, int64_t n,
                                             const SellView& S, const V2<T>* __restrict__ val,
                                             const V2<T>* __restrict__ x) {
  if constexpr (sizeof(T) == 4) {
    __shared__ float2 terms[RowBlock<T, P>::kSlices][P - 1][kTerms<P>][kSliceH];
    auto& mine = terms[uniform(int(threadIdx.x >> 6)) / P];
    return S.uoff ? sell_ordered<true, P>(rb, n, S, val, x, mine)
                  : sell_ordered<false, P>(rb, n, S, val, x, mine);
  } else {
    __shared__ V2<T> sums[4][kSliceH];
    const int w = uniform(int(threadIdx.x >> 6)), lane = int(threadIdx.x & 63);
    V2<T> acc;
    acc.x = acc.y = T(0);
    if (rb.row < n)
      acc = S.uoff ? sell_part<T, true, P>(rb, S, val, x) : sell_part<T, false, P>(rb, S, val, x);
    if (rb.part > 0) sums[w][lane] = acc;
    __syncthreads();
    if (rb.part == 0) {
      if constexpr (P == 4) {
        const V2<T> a = sums[1][lane], b = sums[2][lane], c = sums[3][lane];
        acc.x = (acc.x + a.x) + (b.x + c.x);
        acc.y = (acc.y + a.y) + (b.y + c.y);
      } else {
        const V2<T> b = sums[w + 1][lane];
        acc.x += b.x;
        acc.y += b.y;
      }
    }
    return acc;
  }
}

// P of a mesh, and its number of workgroups and of slices they cover.
inline int row_split(const MeshCache& m) { return m.n <= kSplitRows ? 4 : 2; }
inline unsigned row_blocks(const MeshCache& m) {
  return grid_for(m.n, kSliceH * (4 / row_split(m)));
}
inline unsigned row_slices(const MeshCache& m) { return row_blocks(m) * (4 / row_split(m)); }

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  return v;
}

// Sum of v over each slice's rows (lanes of its owning wave; v = 0 where no row
// is owned) to partials[slice].
template <class T, int P>
__device__ __forceinline__ void slice_partials(const RowBlock<T, P>& rb, double v,
                                               double* __restrict__ partials) {
  if (rb.part != 0) return;
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0)
    partials[blockIdx.x * RowBlock<T, P>::kSlices + (threadIdx.x >> 6) / P] = v;
}

// Block-wide sums of NV values; the totals end up in every lane of wave 0.
// lds must hold 16*NV doubles (blockDim <= 1024).
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* lds) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    v[q] = wave_sum(v[q]);
    if (lane == 0) lds[q * 16 + wid] = v[q];
  }
  __syncthreads();
  if (wid == 0) {
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] = wave_sum(lane < nw ? lds[q * 16 + lane] : 0.0);
  }
  __syncthreads();
}

// Phase one of a grid-wide deterministic sum: each block stores its NV
// partial sums at partials[q * gridDim.x + blockIdx.x]. Phase two is a
// separate one-block kernel (finalize_sum) that adds them in block order;
// the kernel boundary makes the partials visible across XCDs without a
// per-block device-scope fence (which on gfx950 writes back the L2).
template <int NV>
__device__ __forceinline__ void block_partials(double (&v)[NV], double* __restrict__ partials) {
  __shared__ double lds[16 * NV];
  block_sum<NV>(v, lds);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < NV; ++q) partials[q * gridDim.x + blockIdx.x] = v[q];
  }
}

constexpr int kFinalizeThreads = 256;

// Sums nb partials per value in fixed order; totals valid in thread 0. The
// order is that of a block of kFinalizeThreads threads whatever the block
// size (a multiple of 64): virtual thread t adds partials t, t + 256, ...,
// each virtual wave of 64 is reduced by lane shuffles, and the 4 wave sums
// by a last one, so the persistent kernel (blocks of 128 to 1024 threads)
// and the separate finalize kernels (256) give the same bits.
template <int NV>
__device__ __forceinline__ void finalize_sum(double (&v)[NV], const double* __restrict__ partials,
                                             int nb) {
  __shared__ double lds[16 * NV];
  constexpr int kVw = kFinalizeThreads / 64;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = max(1, int(blockDim.x) >> 6);
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    for (int vw = wid; vw < kVw; vw += nw) {
      double s = 0.0;
      for (int i = vw * 64 + lane; i < nb; i += kFinalizeThreads) s += partials[q * nb + i];
      s = wave_sum(s);
      if (lane == 0) lds[q * 16 + vw] = s;
    }
  }
  __syncthreads();
  if (wid == 0) {
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] = wave_sum(lane < kVw ? lds[q * 16 + lane] : 0.0);
  }
  __syncthreads();
}

// Sum of nb partials by one workgroup of kFinThreads (valid in thread 0, fixed
// order). 1024 threads: a solve on 10^6 rows leaves 14 k partials, 14 loads
// a thread, all in flight.
constexpr int kFinThreads = 1024;
__device__ __forceinline__ double fin_sum(const double* __restrict__ partials, int nb) {
  __shared__ double w[kFinThreads / 64];
  double v = 0.0;
#pragma unroll 16
  for (int i = threadIdx.x; i < nb; i += kFinThreads) v += partials[i];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
  __syncthreads();
  v = 0.0;
  if (threadIdx.x < 64) v = wave_sum(threadIdx.x < kFinThreads / 64 ? w[threadIdx.x] : 0.0);
  return v;
}

}  // namespace nosh
