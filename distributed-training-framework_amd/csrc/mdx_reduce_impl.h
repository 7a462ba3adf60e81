// W-way streaming reductions over contributions resident in HBM (kernel
// templates; instantiated per dtype by the mdx_reduce_*.hip translation units).
//
// allreduce_kernel<T, G, W, UNPACK>: DDP's bucket all-reduce.  For element j
// of a piece (replica position p = pos + j):
//     acc = x_0[p]; acc = rnd_T(acc + x_r[p]) for r = 1..W-1      (rank order)
//     out[p] = acc                                  (the in-place all-reduce)
//   UNPACK additionally writes the bucket slice straight into the gradient,
//   with the loss scaler's epilogue:
//     g = cvt_G(acc); g = rnd_G(g * inv_scale); grad[j] = g; bad |= !isfinite(g)
//   which is scatter_from_buffer's copy_ followed by unscale_'s mul_ and
//   isfinite, fused so the bucket is not read back.
//
// allreduce_wide_kernel<In, T, G, W> (+ _dev): the same fused all-reduce +
// unpack for contributions that travel in a narrower dtype In than the bucket
// dtype T (bf16 or fp16 gradients summed into fp32 buckets).  Each contribution is
// widened and pre-scaled at the receiver, x_r = rnd_T(cvt_T(c_r[p]) * pre),
// which is exactly the value the sender's pack (`copy_` into a T bucket, then
// `mul_(1/W)`) would have put on the wire; the rank-ordered sum, the write of
// the T bucket and the unpack epilogue are as above.
//
// allreduce_pack_kernel<In, T, W> (+ _dev): the pack fused in front of the
// fused all-reduce + unpack, for gradients of the wire dtype In.  Replica
// `rank` is read from the run's gradient (NULL = zeros) and packed in
// registers, c = rnd_T(g * pre) for a bucket of the same dtype (the pack's
// `copy_` + `mul_(1/W)`) or the raw gradient for a widening bucket (which
// pre-scales every contribution where it is widened, as above); c is stored
// to replica `rank`'s row -- what the peers read -- and enters the rank-ordered
// sum without being read back, and the bucket is a separate output.  Per
// element: the gradient and W-1 peer rows read; the packed row, the bucket
// and the gradient written.  The dispatch also clears the loss scaler's flag
// for the next step (ReduceParams::clear).
//
// share_kernel<In, Acc, Out, WMAX>: FSDP's reduce-scatter share, runtime
// W <= WMAX.  x_r = cvt_Acc(contribution_r[p]); x_r = rnd_Acc(x_r * pre | x_r / pre);
// acc = rank-ordered sum in Acc; y = cvt_Out(acc); y = rnd_Out(out + y) when
// accumulating; optional unscale + found-inf epilogue.  The pre-scale is a
// compile-time variant selected once per workgroup.  A piece
// may carry its own destination (PieceRun::grad), so that one dispatch writes
// the shard gradients of several FSDP units (the multi-unit share); otherwise
// it writes out + its position.
//
// Every contribution is read once per step, so every load is non-temporal;
// each lane keeps U fragments of all W contributions in flight before the
// first add (about 128 bytes per lane: U * W = 8 16-byte loads for the fp32
// all-reduce at W = 8).
#pragma once

#include <type_traits>

#include "mdx_internal.h"

namespace mdx {
namespace reduce_impl {

// ---------------------------------------------------------------------------
// Fragment arithmetic
// ---------------------------------------------------------------------------

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

// Element `i` of a run, as a scalar base plus a 32-bit byte offset (a run holds
// at most kMaxRunElems elements): no 64-bit vector arithmetic per stream.
static_assert(kMaxRunElems * 4 <= int64_t(UINT32_MAX), "a run's byte offsets fit 32 bits");
template <typename T>
__device__ __forceinline__ T* at(T* base, uint32_t i) {
  using Byte = std::conditional_t<std::is_const_v<T>, const char, char>;
  return reinterpret_cast<T*>(reinterpret_cast<Byte*>(base) + i * uint32_t(sizeof(T)));
}

// Two fp32 values rounded to T, the low half first; NaNs as from_f32<T> stores
// them (bf16: 0xFFFF; `kRaw` leaves the instruction's own quiet NaN, which a
// following from_f32 or RankSum::get makes 0xFFFF).
template <typename T, bool kRaw = false>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if constexpr (std::is_same_v<T, bf16>) {
    uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
    if constexpr (!kRaw) {
      w = __builtin_isnan(lo) ? w | 0xffffu : w;
      w = __builtin_isnan(hi) ? w | 0xffff0000u : w;
    }
    return w;
  } else {
    asm("" : "+v"(lo), "+v"(hi));  // as in from_f32<f16>
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, f16x2));
  }
}

// The rank-ordered sum of E elements of T, one rounding to T per add: `first`
// takes rank 0's values, `add` the next rank's, `get` gives the sums.  The
// results are those of acc = from_f32<T>(to_f32(acc) + to_f32(x)), bit for bit.
template <typename T, int E>
struct RankSum;

template <int E>
struct RankSum<float, E> {
  float a[E];
  __device__ __forceinline__ void first(const float (&x)[E]) {
#pragma unroll
    for (int k = 0; k < E; ++k) a[k] = x[k];
  }
  __device__ __forceinline__ void add(const float (&x)[E]) {
#pragma unroll
    for (int k = 0; k < E; ++k) a[k] += x[k];
  }
  __device__ __forceinline__ void get(float (&y)[E]) const {
#pragma unroll
    for (int k = 0; k < E; ++k) y[k] = a[k];
  }
};

// bf16: the running sum is kept as the fp32 value of its rounding, two elements
// per v_cvt_pk_bf16_f32, and the NaN encoding is settled once, in `get` (a NaN
// stays a NaN through the adds): 3.5 instructions per element and add instead
// of 6 with a conversion, compare and select of its own for each.
template <int E>
struct RankSum<bf16, E> {
  float a[E];
  __device__ __forceinline__ void first(const bf16 (&x)[E]) {
#pragma unroll
    for (int k = 0; k < E; ++k) a[k] = to_f32(x[k]);
  }
  __device__ __forceinline__ void add(const bf16 (&x)[E]) {
#pragma unroll
    for (int k = 0; k < E; k += 2) {
      const uint32_t w = pack2<bf16, true>(a[k] + to_f32(x[k]), a[k + 1] + to_f32(x[k + 1]));
      a[k] = __uint_as_float(w << 16);
      a[k + 1] = __uint_as_float(w & 0xffff0000u);
    }
  }
  __device__ __forceinline__ void get(bf16 (&y)[E]) const {
#pragma unroll
    for (int k = 0; k < E; k += 2) {
      uint32_t w = (__float_as_uint(a[k]) >> 16) | (__float_as_uint(a[k + 1]) & 0xffff0000u);
      w = __builtin_isnan(a[k]) ? w | 0xffffu : w;
      w = __builtin_isnan(a[k + 1]) ? w | 0xffff0000u : w;
      __builtin_memcpy(&y[k], &w, 4);
    }
  }
};

// fp16: v_pk_add_f16, two elements per instruction.  One fp16 rounding of the
// exact sum is the fp32 sum rounded to fp16 (an fp32 significand holds 2 * 11 +
// 2 bits, so rounding twice is rounding once), as over all 2^32 pairs of
// patterns on the device (of two NaNs, either may be the one that stays).
template <int E>
struct RankSum<f16, E> {
  f16x2 a[E / 2];
  __device__ __forceinline__ void first(const f16 (&x)[E]) { __builtin_memcpy(a, x, sizeof(a)); }
  __device__ __forceinline__ void add(const f16 (&x)[E]) {
    f16x2 b[E / 2];
    __builtin_memcpy(b, x, sizeof(b));
#pragma unroll
    for (int k = 0; k < E / 2; ++k) a[k] = a[k] + b[k];
  }
  __device__ __forceinline__ void get(f16 (&y)[E]) const { __builtin_memcpy(y, a, sizeof(a)); }
};

// A fragment multiplied by `s`, each product rounded to T.
template <typename T, int E>
__device__ __forceinline__ void scale_fragment(T (&x)[E], float s) {
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int k = 0; k < E; ++k) x[k] = x[k] * s;
  } else {
#pragma unroll
    for (int k = 0; k < E; k += 2) {
      const uint32_t w = pack2<T>(to_f32(x[k]) * s, to_f32(x[k + 1]) * s);
      __builtin_memcpy(&x[k], &w, 4);
    }
  }
}

template <typename S, typename D, int E>
__device__ __forceinline__ void convert_fragment(const S (&x)[E], D (&y)[E]) {
  if constexpr (std::is_same_v<S, D> || sizeof(D) == 4) {
#pragma unroll
    for (int k = 0; k < E; ++k) y[k] = Cvt<S, D>::run(x[k]);
  } else {
#pragma unroll
    for (int k = 0; k < E; k += 2) {
      const uint32_t w = pack2<D>(to_f32(x[k]), to_f32(x[k + 1]));
      __builtin_memcpy(&y[k], &w, 4);
    }
  }
}

// Whether any element of the fragment is an inf or a NaN.
template <typename T, int E>
__device__ __forceinline__ bool any_nonfinite(const T (&x)[E]) {
  if constexpr (sizeof(T) == 4) {
    bool bad = false;
#pragma unroll
    for (int k = 0; k < E; ++k) bad |= !is_finite(x[k]);
    return bad;
  } else {
    // an all-ones exponent leaves a zero half in the complement
    constexpr uint32_t kExp = std::is_same_v<T, bf16> ? 0x7f807f80u : 0x7c007c00u;
    u16x2 least{0xffff, 0xffff};
#pragma unroll
    for (int k = 0; k < E; k += 2) {
      uint32_t w;
      __builtin_memcpy(&w, &x[k], 4);
      least = __builtin_elementwise_min(least, __builtin_bit_cast(u16x2, ~w & kExp));
    }
    return least.x == 0 || least.y == 0;
  }
}

// ---------------------------------------------------------------------------
// all-reduce (+ fused unpack)
// ---------------------------------------------------------------------------

template <typename In, typename T, typename G, int W, bool UNPACK, bool PRE, bool PACK, typename View>
__device__ __forceinline__ void allreduce_body(const View& tab, const ReduceParams& p) {
  static_assert(!PACK || (UNPACK && sizeof(G) == sizeof(In)), "the fused pack reads gradients of the wire dtype");
  constexpr int E = UNPACK ? reduce_frag_elems(int(sizeof(In)), int(sizeof(T)), int(sizeof(G)))
                            : store_frag_elems(int(sizeof(T)));
  constexpr int U = PACK ? pack_allreduce_unroll() : allreduce_unroll(W, E * int(sizeof(In)));
  constexpr int VPB = kBlock * U;
  constexpr int EPB = VPB * E;
  // 32-byte fragments of a stored type go out through vstore_wave8, which
  // every lane of the wave takes part in: lanes past the end then compute on
  // zeros (finite: they never raise the flag) and store nothing.
  constexpr bool kWaveT = E * int(sizeof(T)) == 32;
  constexpr bool kWaveG = UNPACK && E * int(sizeof(G)) == 32;
  constexpr bool kWave = kWaveT || kWaveG;
  static_assert(!kWave || E == 8, "wave-permuted stores take 8 four-byte elements per lane");

  const int blk = tab.block();
  const PieceRun run = tab.piece_run(blk);
  const int c = run.c;
  const int nblk = run.nblk;
  const int64_t pos = run.pos;
  // A run holds at most kMaxRunElems elements, so its element indices and byte
  // offsets fit 32 bits: every access is a scalar base plus a 32-bit offset.
  const int n = int(run.numel);
  const int h = run.head;
  const int rank = p.rank;
  const int t = int(threadIdx.x);
  const bool unscale = (p.flags & kRedUnscale) != 0;
  const float inv = p.inv_scale;
  const float pre = p.pre;

  // Replica `rank` is read through the run's own pointer: the rank's packed
  // row, or with PACK its gradient, packed here.  A NULL gradient counts as
  // zeros; the row it is packed into is read in its place and not used.
  const bool own_zero = PACK && run.own == nullptr;
  In* own_row = PACK ? static_cast<In*>(const_cast<void*>(p.own_row)) + pos : nullptr;
  const In* own = own_zero ? own_row : static_cast<const In*>(run.own);
  const In* src[W];
#pragma unroll
  for (int r = 0; r < W; ++r) src[r] = (r == rank) ? own : static_cast<const In*>(p.peer[r]) + pos;
  const bool pack_scale = PACK && !PRE && (p.flags & kRedPackScale) != 0;
  T* out = p.out ? static_cast<T*>(p.out) + pos : nullptr;
  G* grad = static_cast<G*>(run.grad);
  bool bad = false;
  // The next step's found-inf flag rides on the fused pack (nothing reads or
  // sets it during this step): one lane of the first workgroup.
  if (PACK && p.clear != nullptr && blk == 0 && t == 0) *p.clear = 0;

  // The pack's `copy_` + `mul_(1/W)` of this rank's gradient (same-dtype
  // buckets; a widening bucket carries the raw gradient and pre-scales where
  // every contribution is widened).
  auto pack_op = [&](In x) -> In {
    if constexpr (PACK && !PRE) {
      const In xs = from_f32<In>(to_f32(x) * pre);
      return pack_scale ? xs : x;
    }
    return x;
  };
  auto widen = [&](In x) -> T {
    T a = Cvt<In, T>::run(x);
    if constexpr (PRE) a = from_f32<T>(to_f32(a) * pre);
    return a;
  };

  auto finish = [&](T acc) -> G {
    G g = Cvt<T, G>::run(acc);
    const G gs = from_f32<G>(to_f32(g) * inv);
    g = unscale ? gs : g;
    bad |= !is_finite(g);
    return g;
  };
  auto element = [&](int i) {
    T acc = zero_of<T>();
    In packed = zero_of<In>();
#pragma unroll
    for (int r = 0; r < W; ++r) {
      In xr = src[r][i];
      if (PACK && r == rank) {
        xr = pack_op(own_zero ? zero_of<In>() : xr);
        packed = xr;
      }
      const T a = widen(xr);
      acc = (r == 0) ? a : from_f32<T>(to_f32(acc) + to_f32(a));
    }
    if constexpr (PACK) own_row[i] = packed;
    if (out) out[i] = acc;
    if constexpr (UNPACK) grad[i] = finish(acc);
  };

  if (h >= 0) {
    const int nvec = (n - h) / E;
    In x[U][W][E];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v = c * VPB + u * kBlock + t;
      if constexpr (kWave) {
#pragma unroll
        for (int r = 0; r < W; ++r) {
#pragma unroll
          for (int e = 0; e < E; ++e) x[u][r][e] = zero_of<In>();
        }
      }
      if (v < nvec) {
#pragma unroll
        for (int r = 0; r < W; ++r) vload<In, E, true>(x[u][r], at(src[r], uint32_t(h + v * E)));
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v0 = c * VPB + u * kBlock;  // the fragment of lane 0
      const int v = v0 + t;
      const bool active = v < nvec;
      // elements of this wave's fragment that exist (wave-permuted stores only)
      const int limit = max_size(0, min_size(nvec - v0, kBlock)) * E;
      if (kWave || active) {
        const uint32_t i = uint32_t(h + v * E);
        if constexpr (PACK) {
          // This rank's fragment, packed in registers (static indices: the
          // branch on the wave-uniform rank picks the replica slot).
          In po[E];
#pragma unroll
          for (int r = 0; r < W; ++r) {
            if (r == rank) {
              __builtin_amdgcn_sched_barrier(0);  // keeps the branch: as selects this runs for every r
              if (own_zero) {
#pragma unroll
                for (int e = 0; e < E; ++e) x[u][r][e] = zero_of<In>();
              }
              if constexpr (!PRE) {
                if (pack_scale) scale_fragment(x[u][r], pre);
              }
#pragma unroll
              for (int e = 0; e < E; ++e) po[e] = x[u][r][e];
            }
          }
          if (active) vstore<In, E, true>(at(own_row, i), po);
        }
        T y[E];
        if constexpr (PRE) {
#pragma unroll
          for (int e = 0; e < E; ++e) {
            T acc = widen(x[u][0][e]);
#pragma unroll
            for (int r = 1; r < W; ++r) acc = from_f32<T>(to_f32(acc) + to_f32(widen(x[u][r][e])));
            y[e] = acc;
          }
        } else if constexpr (W == 1) {
#pragma unroll
          for (int e = 0; e < E; ++e) y[e] = x[u][0][e];
        } else {
          RankSum<T, E> sum;
          sum.first(x[u][0]);
#pragma unroll
          for (int r = 1; r < W; ++r) sum.add(x[u][r]);
          sum.get(y);
        }
        if (out) {
          if constexpr (kWaveT) {
            vstore_wave8<T>(out + uint32_t(h + v0 * E), y, t, limit);
          } else if (active) {
            vstore<T, E, true>(at(out, i), y);
          }
        }
        if constexpr (UNPACK) {
          G gy[E];
          convert_fragment(y, gy);
          if (unscale) scale_fragment(gy, inv);
          bad |= any_nonfinite(gy);
          if constexpr (kWaveG) {
            vstore_wave8<G>(grad + uint32_t(h + v0 * E), gy, t, limit);
          } else if (active) {
            vstore<G, E, true>(at(grad, i), gy);
          }
        }
      }
    }
    if (c == 0 && t < h && t < n) element(t);
    const int tail0 = h + nvec * E;
    if (c == nblk - 1 && tail0 + t < n) element(tail0 + t);
  } else {
#pragma unroll 4
    for (int k = 0; k < U * E; ++k) {
      const int i = c * EPB + k * kBlock + t;
      if (i < n) element(i);
    }
  }
  if constexpr (UNPACK) {
    if (p.found_inf) flag_nonfinite(bad, p.found_inf);
  }
}

// Table in the kernel-argument segment.
template <typename T, typename G, int W, bool UNPACK>
__global__ void __launch_bounds__(kBlock) allreduce_kernel(PieceBatch b, ReduceParams p) {
  allreduce_body<T, T, G, W, UNPACK, false, false>(PieceArgView{b}, p);
}

// Table (plan) in device memory; the fused all-reduce + unpack only.
template <typename T, typename G, int W>
__global__ void __launch_bounds__(kBlock) allreduce_unpack_kernel_dev(DevTable t, ReduceParams p) {
  allreduce_body<T, T, G, W, true, false, false>(DevView{t}, p);
}

// Widening variants (fused all-reduce + unpack with pre-scale at the receiver).
template <typename In, typename T, typename G, int W>
__global__ void __launch_bounds__(kBlock) allreduce_wide_kernel(PieceBatch b, ReduceParams p) {
  allreduce_body<In, T, G, W, true, true, false>(PieceArgView{b}, p);
}

template <typename In, typename T, typename G, int W>
__global__ void __launch_bounds__(kBlock) allreduce_wide_kernel_dev(DevTable t, ReduceParams p) {
  allreduce_body<In, T, G, W, true, true, false>(DevView{t}, p);
}

// Pack fused into the all-reduce + unpack: gradients of the wire dtype In,
// bucket dtype T (T != In: widening, pre-scaled at the receiver).
template <typename In, typename T, int W>
__global__ void __launch_bounds__(kBlock) allreduce_pack_kernel(PieceBatch b, ReduceParams p) {
  allreduce_body<In, T, In, W, true, (sizeof(In) != sizeof(T)), true>(PieceArgView{b}, p);
}

template <typename In, typename T, int W>
__global__ void __launch_bounds__(kBlock) allreduce_pack_kernel_dev(DevTable t, ReduceParams p) {
  allreduce_body<In, T, In, W, true, (sizeof(In) != sizeof(T)), true>(DevView{t}, p);
}

template <typename T, typename G, bool UNPACK>
struct ArgAllreduce {
  const PieceBatch& b;
  template <int W>
  hipError_t go(const ReduceParams& p, hipStream_t stream) const {
    const int blocks = b.first_block[b.count];
    hipLaunchKernelGGL((allreduce_kernel<T, G, W, UNPACK>), dim3(blocks), dim3(kBlock),
                       reduce_lds(blocks, sizeof(T), sizeof(T), W), stream, b, p);
    return hipGetLastError();
  }
};

template <typename T, typename G>
struct DevAllreduceUnpack {
  const DevTable& t;
  int blocks;
  template <int W>
  hipError_t go(const ReduceParams& p, hipStream_t stream) const {
    return launch_plan_slices(t, blocks, [&](const DevTable& slice, int grid) {
      hipLaunchKernelGGL((allreduce_unpack_kernel_dev<T, G, W>), dim3(grid), dim3(kBlock),
                         reduce_lds(grid, sizeof(T), sizeof(T), W), stream, slice, p);
    });
  }
};

template <typename In, typename T, typename G>
struct ArgWide {
  const PieceBatch& b;
  template <int W>
  hipError_t go(const ReduceParams& p, hipStream_t stream) const {
    const int blocks = b.first_block[b.count];
    hipLaunchKernelGGL((allreduce_wide_kernel<In, T, G, W>), dim3(blocks), dim3(kBlock),
                       reduce_lds(blocks, sizeof(In), sizeof(T), W), stream, b, p);
    return hipGetLastError();
  }
};

template <typename In, typename T, typename G>
struct DevWide {
  const DevTable& t;
  int blocks;
  template <int W>
  hipError_t go(const ReduceParams& p, hipStream_t stream) const {
    return launch_plan_slices(t, blocks, [&](const DevTable& slice, int grid) {
      hipLaunchKernelGGL((allreduce_wide_kernel_dev<In, T, G, W>), dim3(grid), dim3(kBlock),
                         reduce_lds(grid, sizeof(In), sizeof(T), W), stream, slice, p);
    });
  }
};

template <typename In, typename T>
struct ArgPack {
  const PieceBatch& b;
  template <int W>
  hipError_t go(const ReduceParams& p, hipStream_t stream) const {
    const int blocks = b.first_block[b.count];
    hipLaunchKernelGGL((allreduce_pack_kernel<In, T, W>), dim3(blocks), dim3(kBlock),
                       reduce_lds(blocks, sizeof(In), sizeof(T), W), stream, b, p);
    return hipGetLastError();
  }
};

template <typename In, typename T>
struct DevPack {
  const DevTable& t;
  int blocks;
  template <int W>
  hipError_t go(const ReduceParams& p, hipStream_t stream) const {
    return launch_plan_slices(t, blocks, [&](const DevTable& slice, int grid) {
      hipLaunchKernelGGL((allreduce_pack_kernel_dev<In, T, W>), dim3(grid), dim3(kBlock),
                         reduce_lds(grid, sizeof(In), sizeof(T), W), stream, slice, p);
    });
  }
};

template <typename L>
hipError_t by_world(int world, const L& l, const ReduceParams& p, hipStream_t stream) {
  switch (world) {
    case 1: return l.template go<1>(p, stream);
    case 2: return l.template go<2>(p, stream);
    case 3: return l.template go<3>(p, stream);
    case 4: return l.template go<4>(p, stream);
    case 5: return l.template go<5>(p, stream);
    case 6: return l.template go<6>(p, stream);
    case 7: return l.template go<7>(p, stream);
    case 8: return l.template go<8>(p, stream);
    case 9: return l.template go<9>(p, stream);
    case 10: return l.template go<10>(p, stream);
    case 11: return l.template go<11>(p, stream);
    case 12: return l.template go<12>(p, stream);
    case 13: return l.template go<13>(p, stream);
    case 14: return l.template go<14>(p, stream);
    case 15: return l.template go<15>(p, stream);
    default: return l.template go<16>(p, stream);
  }
}

template <typename T, typename G, bool UNPACK>
hipError_t launch_allreduce(int world, const PieceBatch& b, const ReduceParams& p, hipStream_t stream) {
  return by_world(world, ArgAllreduce<T, G, UNPACK>{b}, p, stream);
}

template <typename T, typename G>
hipError_t launch_allreduce_unpack_dev(int world, const DevTable& t, int blocks, const ReduceParams& p,
                                       hipStream_t stream) {
  return by_world(world, DevAllreduceUnpack<T, G>{t, blocks}, p, stream);
}

template <typename In, typename T, typename G>
hipError_t launch_allreduce_wide(int world, const PieceBatch& b, const ReduceParams& p, hipStream_t stream) {
  return by_world(world, ArgWide<In, T, G>{b}, p, stream);
}

template <typename In, typename T, typename G>
hipError_t launch_allreduce_wide_dev(int world, const DevTable& t, int blocks, const ReduceParams& p,
                                     hipStream_t stream) {
  return by_world(world, DevWide<In, T, G>{t, blocks}, p, stream);
}

// Per-dtype instantiation sets, one call each from the instantiating
// translation units: T is the bucket dtype (plain SUM and fused unpack into
// any gradient dtype); In is the wire dtype of the widening variant.
template <typename T>
hipError_t launch_allreduce_for(int grad_dtype, bool unpack, int world, const PieceBatch& b,
                                const ReduceParams& p, hipStream_t stream) {
  if (!unpack) return launch_allreduce<T, T, false>(world, b, p, stream);
  if (grad_dtype == MDX_F32) return launch_allreduce<T, float, true>(world, b, p, stream);
  if (grad_dtype == MDX_BF16) return launch_allreduce<T, bf16, true>(world, b, p, stream);
  return launch_allreduce<T, f16, true>(world, b, p, stream);
}

template <typename T>
hipError_t launch_allreduce_dev_for(int grad_dtype, int world, const DevTable& t, int blocks,
                                    const ReduceParams& p, hipStream_t stream) {
  if (grad_dtype == MDX_F32) return launch_allreduce_unpack_dev<T, float>(world, t, blocks, p, stream);
  if (grad_dtype == MDX_BF16) return launch_allreduce_unpack_dev<T, bf16>(world, t, blocks, p, stream);
  return launch_allreduce_unpack_dev<T, f16>(world, t, blocks, p, stream);
}

template <typename In>
hipError_t launch_wide_for(int grad_dtype, int world, const PieceBatch& b, const ReduceParams& p,
                           hipStream_t stream) {
  if (grad_dtype == MDX_F32) return launch_allreduce_wide<In, float, float>(world, b, p, stream);
  if (grad_dtype == MDX_BF16) return launch_allreduce_wide<In, float, bf16>(world, b, p, stream);
  return launch_allreduce_wide<In, float, f16>(world, b, p, stream);
}

template <typename In>
hipError_t launch_wide_dev_for(int grad_dtype, int world, const DevTable& t, int blocks, const ReduceParams& p,
                               hipStream_t stream) {
  if (grad_dtype == MDX_F32) return launch_allreduce_wide_dev<In, float, float>(world, t, blocks, p, stream);
  if (grad_dtype == MDX_BF16) return launch_allreduce_wide_dev<In, float, bf16>(world, t, blocks, p, stream);
  return launch_allreduce_wide_dev<In, float, f16>(world, t, blocks, p, stream);
}

// The fused pack + all-reduce + unpack of one (wire, bucket) dtype pair.
template <typename In, typename T>
hipError_t launch_pack_for(int world, const PieceBatch& b, const ReduceParams& p, hipStream_t stream) {
  return by_world(world, ArgPack<In, T>{b}, p, stream);
}

template <typename In, typename T>
hipError_t launch_pack_dev_for(int world, const DevTable& t, int blocks, const ReduceParams& p,
                               hipStream_t stream) {
  return by_world(world, DevPack<In, T>{t, blocks}, p, stream);
}

// ---------------------------------------------------------------------------
// reduce-scatter share
// ---------------------------------------------------------------------------

enum : int { kPreNone = 0, kPreMul = 1, kPreDiv = 2 };

// E quotients x / w, correctly rounded, for w a whole number from 3 to 15 that is
// not a power of two and rw = 1 / w rounded.  One Newton step on x * rw, with the
// remainder exact in an fma, gives the rounded quotient, and the sign of x that of
// a zero: equal to the division on all 2^32 patterns of x for each of these w,
// checked on the device, except infinities and, for even w, |x| < 2^-124.  A wave
// that meets one of those, or an |x| under 2^-118, divides.  8 instructions an
// element instead of a division's 13 with a reciprocal of its own (shares of 100 MB
// a rank: bf16 sums 161.3 -> 131.8 us at W = 6 and 83.0 -> 68.1 at W = 3, fp32 sums
// of bf16 139.8 -> 123.9 at W = 6).
template <int E>
__device__ __forceinline__ void divide_by_world(float (&x)[E], float w, float rw) {
  float z[E];
  uint32_t most = 0, least = UINT32_MAX;  // of the magnitudes' bits; zeros do not count for `least`
#pragma unroll
  for (int k = 0; k < E; ++k) {
    const float q = x[k] * rw;
    z[k] = __builtin_copysignf(__builtin_fmaf(__builtin_fmaf(-q, w, x[k]), rw, q), x[k]);
    const uint32_t t = __float_as_uint(x[k]) & 0x7fffffffu;
    most = most > t ? most : t;
    least = least < t - 1 ? least : t - 1;
  }
  constexpr uint32_t kInf = 0x7f800000u, kSmall = 9u << 23;  // 2^-118
  if (most >= kInf || least < kSmall - 1) {
#pragma unroll
    for (int k = 0; k < E; ++k) x[k] = x[k] / w;
  } else {
#pragma unroll
    for (int k = 0; k < E; ++k) x[k] = z[k];
  }
}

// A fragment divided by the world size, each quotient rounded to T.
template <typename T, int E>
__device__ __forceinline__ void divide_fragment(T (&x)[E], float w, float rw) {
  if constexpr (sizeof(T) == 4) {
    divide_by_world(x, w, rw);
  } else {
    float f[E];
#pragma unroll
    for (int k = 0; k < E; ++k) f[k] = to_f32(x[k]);
    divide_by_world(f, w, rw);
#pragma unroll
    for (int k = 0; k < E; k += 2) {
      const uint32_t v = pack2<T>(f[k], f[k + 1]);
      __builtin_memcpy(&x[k], &v, 4);
    }
  }
}

template <typename In, typename Acc, typename Out, int WMAX, int PRE>
__device__ __forceinline__ void share_body(const PieceRun& run, const ReduceParams& p) {
  constexpr int E = reduce_frag_elems(int(sizeof(In)), int(sizeof(Out)), int(sizeof(Out)));
  constexpr int U = share_unroll(WMAX, E * int(sizeof(In)));
  constexpr int VPB = kBlock * U;
  constexpr int EPB = VPB * E;
  // 32-byte fragments of the shard dtype go out through vstore_wave8 (16-bit
  // contributions into an fp32 shard), as in allreduce_body.
  constexpr bool kWave = E * int(sizeof(Out)) == 32;
  static_assert(!kWave || E == 8, "wave-permuted stores take 8 four-byte elements per lane");

  const int c = run.c;
  const int nblk = run.nblk;
  const int64_t pos = run.pos;
  const int n = int(run.numel);  // at most kMaxRunElems
  const int h = run.head;
  const int world = p.world;
  const int rank = p.rank;
  const bool own_zero = (run.own == nullptr);
  const int t = int(threadIdx.x);
  const float pre = p.pre;
  const float rpre = PRE == kPreDiv ? 1.0f / pre : 1.0f;
  const bool accumulate = (p.flags & kRedAccumulate) != 0;
  const bool unscale = (p.flags & kRedUnscale) != 0;
  const float inv = p.inv_scale;

  const In* src[WMAX];
#pragma unroll
  for (int r = 0; r < WMAX; ++r) {
    src[r] = (r == rank) ? static_cast<const In*>(run.own) : static_cast<const In*>(p.peer[r]) + pos;
  }
  // A piece of a multi-unit share carries its own destination (each unit's
  // shard gradient is a tensor of its own); otherwise the shard is p.out.
  Out* out = run.grad ? static_cast<Out*>(run.grad) : static_cast<Out*>(p.out) + pos;
  bool bad = false;

  auto widen = [&](In x) -> Acc {
    Acc a = Cvt<In, Acc>::run(x);
    if constexpr (PRE == kPreMul) a = from_f32<Acc>(to_f32(a) * pre);
    if constexpr (PRE == kPreDiv) a = from_f32<Acc>(to_f32(a) / pre);
    return a;
  };
  auto element = [&](int i) {
    Acc acc = zero_of<Acc>();
    for (int r = 0; r < world; ++r) {
      const In* row = (r == rank) ? static_cast<const In*>(run.own) : static_cast<const In*>(p.peer[r]) + pos;
      const In x = (r == rank && own_zero) ? zero_of<In>() : row[i];
      const Acc a = widen(x);
      acc = (r == 0) ? a : from_f32<Acc>(to_f32(acc) + to_f32(a));
    }
    Out y = Cvt<Acc, Out>::run(acc);
    if (accumulate) y = from_f32<Out>(to_f32(out[i]) + to_f32(y));
    if (unscale) y = from_f32<Out>(to_f32(y) * inv);
    bad |= !is_finite(y);
    out[i] = y;
  };

  if (h >= 0) {
    const int nvec = (n - h) / E;
    In x[U][WMAX][E];
    Out prev[U][E];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v = c * VPB + u * kBlock + t;
      const uint32_t i = uint32_t(h + v * E);
      if constexpr (kWave) {
#pragma unroll
        for (int k = 0; k < E; ++k) {
#pragma unroll
          for (int r = 0; r < WMAX; ++r) x[u][r][k] = zero_of<In>();
          prev[u][k] = zero_of<Out>();
        }
      }
      if (v < nvec) {
#pragma unroll
        for (int r = 0; r < WMAX; ++r) {
          if (r < world) {
            if (r == rank && own_zero) {
#pragma unroll
              for (int k = 0; k < E; ++k) x[u][r][k] = zero_of<In>();
            } else {
              vload<In, E, true>(x[u][r], at(src[r], i));
            }
          }
        }
        if (accumulate) vload<Out, E, false>(prev[u], at(out, i));
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v0 = c * VPB + u * kBlock;  // the fragment of lane 0
      const int v = v0 + t;
      const bool active = v < nvec;
      const int limit = max_size(0, min_size(nvec - v0, kBlock)) * E;
      if (kWave || active) {
        // rank 0's values, widened, pre-scaled; then every next rank's added
        RankSum<Acc, E> sum;
        Acc a[E];
#pragma unroll
        for (int r = 0; r < WMAX; ++r) {
          if (r < world) {
            convert_fragment(x[u][r], a);
            if constexpr (PRE == kPreMul) scale_fragment(a, pre);
            if constexpr (PRE == kPreDiv) divide_fragment(a, pre, rpre);
            if (r == 0) sum.first(a);
            else sum.add(a);
          }
        }
        // (a world of one hands its values on as they are, NaN payloads too)
        if (world > 1) sum.get(a);
        Out y[E];
        convert_fragment(a, y);
        if (accumulate) {
          if constexpr (sizeof(Out) == 4) {
#pragma unroll
            for (int k = 0; k < E; ++k) y[k] = prev[u][k] + y[k];
          } else {
            RankSum<Out, E> total;
            total.first(prev[u]);
            total.add(y);
            total.get(y);
          }
        }
        if (unscale) scale_fragment(y, inv);
        bad |= any_nonfinite(y);
        if constexpr (kWave) {
          vstore_wave8<Out>(out + uint32_t(h + v0 * E), y, t, limit);
        } else {
          vstore<Out, E, true>(at(out, uint32_t(h + v * E)), y);
        }
      }
    }
    if (c == 0 && t < h && t < n) element(t);
    const int tail0 = h + nvec * E;
    if (c == nblk - 1 && tail0 + t < n) element(tail0 + t);
  } else {
#pragma unroll 1
    for (int k = 0; k < U * E; ++k) {
      const int i = c * EPB + k * kBlock + t;
      if (i < n) element(i);
    }
  }
  if (p.found_inf) flag_nonfinite(bad, p.found_inf);
}

template <typename In, typename Acc, typename Out, int WMAX>
__device__ __forceinline__ void share_run(const PieceRun& run, const ReduceParams& p) {
  if (p.flags & kRedPreMul) share_body<In, Acc, Out, WMAX, kPreMul>(run, p);
  else if (p.flags & kRedPreDiv) share_body<In, Acc, Out, WMAX, kPreDiv>(run, p);
  else share_body<In, Acc, Out, WMAX, kPreNone>(run, p);
}

template <typename In, typename Acc, typename Out, int WMAX>
__global__ void __launch_bounds__(kBlock) share_kernel(PieceBatch b, ReduceParams p) {
  share_run<In, Acc, Out, WMAX>(PieceArgView{b}.piece_run(int(blockIdx.x)), p);
}

// One piece (an FSDP unit's shard) in the kernel-argument segment.
template <typename In, typename Acc, typename Out, int WMAX>
__global__ void __launch_bounds__(kBlock) share_kernel_one(PieceOne b, ReduceParams p) {
  share_run<In, Acc, Out, WMAX>(PieceOneView{b}.piece_run(int(blockIdx.x)), p);
}

// Up to kFewRuns pieces in the kernel-argument segment.
template <typename In, typename Acc, typename Out, int WMAX>
__global__ void __launch_bounds__(kBlock) share_kernel_few(PieceFew b, ReduceParams p) {
  share_run<In, Acc, Out, WMAX>(PieceFewView{b}.piece_run(int(blockIdx.x)), p);
}

// Pieces of a device plan: the shares of many FSDP units in one dispatch.
template <typename In, typename Acc, typename Out, int WMAX>
__global__ void __launch_bounds__(kBlock) share_kernel_dev(DevTable t, ReduceParams p) {
  const DevView v{t};
  share_run<In, Acc, Out, WMAX>(v.piece_run(v.block()), p);
}

// The share kernels' bound on waves per CU (see reduce_waves), GB/s at 32 / 18 /
// 12 / 9 waves:
//   bf16 -> fp32 sums, W = 8, 1.8 GB        6347 6438 6681 6871   (288 MB: 5761 5843 6215 6266)
//   bf16 -> bf16 sums -> fp32, W = 4, 630 MB  6310 6421 6574 6376
//   bf16 sums, W = 8, 1.9 GB                6241 6351 6769 5965
//   bf16 sums, W = 2, 630 MB                6532 6622 5500 4579
//   fp16 sums, W = 8, 940 MB                6244 6373 6567 6871
// A division per contribution (W not a power of two) takes more waves: fp32 sums
// of bf16, W = 6, 700 MB, 6475 6651 6409 5371 with 6772 at 14; fp16 sums, W = 5, 600 MB,
// 6305 6600 5690 4969 with 6782 at 16; bf16 sums, W = 6, lose with any bound.
template <typename Acc, typename Out>
int share_lds(int blocks, const ReduceParams& p) {
  if (blocks < 64 * kCus) return 0;
  const bool divides = (p.flags & kRedPreDiv) != 0;
  if constexpr (std::is_same_v<Acc, bf16>) {
    if (divides) return 0;
    return lds_for_waves(p.world <= 2 ? 18 : (p.world <= 8 ? 12 : 10));
  } else {
    if (divides) return lds_for_waves(sizeof(Acc) == 4 ? 14 : 16);
    return lds_for_waves(9);
  }
}

template <typename In, typename Acc, typename Out, int WMAX>
hipError_t launch_share_dev_w(const DevTable& t, int blocks, const ReduceParams& p, hipStream_t stream) {
  return launch_plan_slices(t, blocks, [&](const DevTable& slice, int grid) {
    const int lds = share_lds<Acc, Out>(grid, p);
    hipLaunchKernelGGL((share_kernel_dev<In, Acc, Out, WMAX>), dim3(grid), dim3(kBlock), lds, stream, slice, p);
  });
}

template <typename In, typename Acc, typename Out, int WMAX>
hipError_t launch_share_w(const PieceBatch& b, const ReduceParams& p, hipStream_t stream) {
  const int blocks = b.first_block[b.count], lds = share_lds<Acc, Out>(blocks, p);
  if (b.count == 1) {
    hipLaunchKernelGGL((share_kernel_one<In, Acc, Out, WMAX>), dim3(blocks), dim3(kBlock), lds, stream,
                       one_run_of(b), p);
  } else if (b.count <= kFewRuns) {
    hipLaunchKernelGGL((share_kernel_few<In, Acc, Out, WMAX>), dim3(blocks), dim3(kBlock), lds, stream,
                       few_runs_of(b), p);
  } else {
    hipLaunchKernelGGL((share_kernel<In, Acc, Out, WMAX>), dim3(blocks), dim3(kBlock), lds, stream, b, p);
  }
  return hipGetLastError();
}

// Every (Acc, Out) pair for contributions of type In, except (fp32, fp32), at the
// width classes of share_wmax.
template <typename In, typename Acc, typename Out>
hipError_t launch_share_width(int wmax, const PieceBatch& b, const ReduceParams& p, hipStream_t stream) {
  if (wmax == 4) return launch_share_w<In, Acc, Out, 4>(b, p, stream);
  if (wmax == 8) return launch_share_w<In, Acc, Out, 8>(b, p, stream);
  return launch_share_w<In, Acc, Out, 16>(b, p, stream);
}

template <typename In, typename Acc>
hipError_t launch_share_out(int out_dtype, int wmax, const PieceBatch& b, const ReduceParams& p, hipStream_t stream) {
  if (out_dtype == MDX_BF16) return launch_share_width<In, Acc, bf16>(wmax, b, p, stream);
  if (out_dtype == MDX_F16) return launch_share_width<In, Acc, f16>(wmax, b, p, stream);
  if constexpr (sizeof(Acc) == 4) {
    return hipErrorInvalidValue;  // (fp32, fp32) goes to launch_share_fast
  } else {
    return launch_share_width<In, Acc, float>(wmax, b, p, stream);
  }
}

template <typename In>
hipError_t launch_share_generic_for(int acc_dtype, int out_dtype, int wmax, const PieceBatch& b,
                                    const ReduceParams& p, hipStream_t stream) {
  if (acc_dtype == MDX_F32) return launch_share_out<In, float>(out_dtype, wmax, b, p, stream);
  if (acc_dtype == MDX_BF16) return launch_share_out<In, bf16>(out_dtype, wmax, b, p, stream);
  return launch_share_out<In, f16>(out_dtype, wmax, b, p, stream);
}

}  // namespace reduce_impl
}  // namespace mdx
