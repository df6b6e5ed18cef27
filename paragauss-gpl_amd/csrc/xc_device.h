// Device helpers shared by the kernels: memory access, the walk over work lists
// (XCD-aware order, queues), MFMA traits and result placement, the split into
// bf16 parts, and what the contractions have in common (a potential item's live
// blocks, sums over a result block's columns, the store of a block).
#pragma once
#include "pgxc_internal.h"

namespace pgxc {

// ------------------------------------------------------------------ helpers
// Global-memory access through pointers the compiler cannot place (they are
// read from descriptors): global_load / global_store instead of flat ones,
// which would also count against the LDS wait counter.
template <typename T>
__device__ __forceinline__ T gld(const T *p) {
  return *(const __attribute__((address_space(1))) T *)p;
}
template <typename T>
__device__ __forceinline__ void gst(T *p, T v) {
  *(__attribute__((address_space(1))) T *)p = v;
}
// Access at column p of a row whose address is the same for the whole wave: the
// instruction takes the scalar base and the lane's 32-bit byte offset (a unit has
// at most 2^24 points), no address arithmetic per lane.
template <typename T>
__device__ __forceinline__ void gst_row(T *row, unsigned p, T v) {
  auto *base = (__attribute__((address_space(1))) char *)row;
  unsigned off = p * (unsigned)sizeof(T);
  asm("" : "+v"(off));  // widened here, where the store's form is chosen
  *(__attribute__((address_space(1))) T *)(base + off) = v;
}

template <typename T>
__device__ __forceinline__ T gld_row(const T *row, unsigned p) {
  const auto *base = (const __attribute__((address_space(1))) char *)row;
  unsigned off = p * (unsigned)sizeof(T);
  asm("" : "+v"(off));
  return *(const __attribute__((address_space(1))) T *)(base + off);
}

// Unit whose items hold item `it` (base: the units' first items).
__device__ __forceinline__ int find_unit(const long *__restrict__ base, int nu, long it) {
  int lo = 0, hi = nu - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (base[mid] <= it) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Workgroups are dispatched round-robin over the 8 XCDs; give every XCD a
// contiguous range of tile ids so that tiles sharing an operand panel share
// that XCD's L2.
__device__ __forceinline__ int xcd_remap(int bid, int nblk) {
  const int per = nblk >> 3;
  if (bid >= (per << 3)) return bid;
  return (bid & 7) * per + (bid >> 3);
}

// A position of a queued list (the first wave calls it) from the queues after
// the workgroup's own (blockIdx.x % kQueues), from `first` on; total when all
// are drained.  The lanes look at all counters at once, so a workgroup at the
// end of the launch waits for one load, not for a claim on every queue in turn.
__device__ __forceinline__ long walk_claim_queue(const StageList &S, int first) {
  const int lane = threadIdx.x & 63, t = lane & (kQueues - 1);
  const int qq = (int)((blockIdx.x + t) % kQueues);
  const long beg = S.qbeg[qq], end = S.qbeg[qq + 1];
  const long seen = __hip_atomic_load(S.ctr + qq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  unsigned long long open = __ballot(lane < kQueues && lane >= first && beg + seen < end);
  while (open) {
    const int u = __builtin_ctzll(open);
    open &= open - 1;
    int c = 0;
    if (lane == u) c = atomicAdd(S.ctr + qq, 1);
    const long p = S.qbeg[(blockIdx.x + u) % kQueues] + __builtin_amdgcn_readlane(c, u);
    if (p < S.qbeg[(blockIdx.x + u) % kQueues + 1]) return p;
  }
  return S.total;
}

// Walk of a stage list's positions.  Static: blockIdx.x, + gridDim.x, ...
// With queues: the next position of the workgroup's own queue; once that is
// drained, of the next queue that is not; total when all are.  Every thread
// of the workgroup calls it.
__device__ __forceinline__ long walk_next(const StageList &S, long prev, long *slot) {
  if (!S.ctr) return prev < 0 ? (long)blockIdx.x : prev + (long)gridDim.x;
  if (threadIdx.x < 64) {
    const int q = (int)(blockIdx.x % kQueues);
    int raw = 0;
    if (threadIdx.x == 0) raw = atomicAdd(S.ctr + q, 1);
    long p = S.qbeg[q] + (long)__builtin_amdgcn_readfirstlane(raw);
    if (p >= S.qbeg[q + 1]) p = walk_claim_queue(S, 1);
    if (threadIdx.x == 0) *slot = p;
  }
  __syncthreads();
  const long p = *slot;
  __syncthreads();
  return p;
}

// The same walk with the next position claimed during the current item:
// walk_ahead (every thread, before the item's last phase) issues thread 0's
// claim on its own queue without waiting for it, and walk_take (every thread,
// after the item) checks it (falling back to the other queues) and hands it
// to the workgroup, so the claim's round trip overlaps the last phase.  The
// slot is written again only after the next item's barriers.
__device__ __forceinline__ int walk_ahead(const StageList &S) {
  int raw = 0;  // thread 0: the claim's counter value, still in flight here
  if (S.ctr && threadIdx.x == 0) raw = atomicAdd(S.ctr + blockIdx.x % kQueues, 1);
  return raw;
}
__device__ __forceinline__ long walk_take(const StageList &S, long cur, int raw, long *slot) {
  if (!S.ctr) return cur + (long)gridDim.x;
  // the claim's value is first read here: an empty asm that takes it keeps
  // the compiler from converting it (and so waiting for it) where it arrives
  asm volatile("" : "+v"(raw));
  if (threadIdx.x < 64) {
    const int q = (int)(blockIdx.x % kQueues);
    long p = S.qbeg[q] + (long)__builtin_amdgcn_readfirstlane(raw);
    if (p >= S.qbeg[q + 1]) p = walk_claim_queue(S, 1);
    if (threadIdx.x == 0) *slot = p;
  }
  __syncthreads();
  return *slot;
}

// item at a position: the schedule's order, else (static walk) the
// XCD-blocked order, else (queues) the natural order
__device__ __forceinline__ long walk_item(const StageList &S, long pos) {
  if (S.order) return (long)S.order[pos];
  return S.ctr ? pos : (long)xcd_remap((int)pos, (int)S.total);
}

// per-item time log (wall clock ticks of the workgroup)
__device__ __forceinline__ void item_log(const StageList &S, long it, uint64_t t0) {
  if (!S.tlog) return;
  __syncthreads();
  if (threadIdx.x == 0) S.tlog[it] = (uint32_t)(wall_clock64() - t0);
}

// x = hi + lo with hi = bf16(x), lo = bf16(x - hi)
__device__ __forceinline__ void split_bf16(float x, __bf16 &hi, __bf16 &lo) {
  // x stays a float: a conversion from FP64 before it must not be merged into
  // the one to bf16, which the hardware has only from FP32 (9 instructions more)
  asm("" : "+v"(x));
  hi = (__bf16)x;
  lo = (__bf16)(x - (float)hi);
}

template <typename T>
struct MF;
// 16x16x4 MFMA operand/result placement (wave64), both types:
//   A(i,k): lane = i + 16 k      B(k,j): lane = j + 16 k
// Result element r of lane l (measured on gfx950):
//   f64: D(i,j) with i = l / 16 + 4 r, j = l % 16
//   f32: D(i,j) with i = 4 (l / 16) + r, j = l % 16
template <>
struct MF<double> {
  typedef d4 acc;
  __device__ static __forceinline__ acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static constexpr bool kQuadRows = false;
  __device__ static __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <>
struct MF<float> {
  typedef f4 acc;
  __device__ static __forceinline__ acc mma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static constexpr bool kQuadRows = true;  // a lane's four results are consecutive rows
  __device__ static __forceinline__ int row(int lane, int r) { return ((lane >> 4) << 2) + r; }
};
__device__ __forceinline__ int mf_col(int lane) { return lane & 15; }


// K step and LDS stages of the contraction variants the layout can select
template <int V> struct Var;
template <> struct Var<0> { static constexpr int BK = 16, ST = 2; };
template <> struct Var<1> { static constexpr int BK = 32, ST = 1; };
template <> struct Var<2> { static constexpr int BK = 32, ST = 2; };

// ---------------------------------------------------------------- screening
// Copy n list entries into LDS (every thread calls it; ends with a barrier).
__device__ __forceinline__ void lds_list(const uint16_t *__restrict__ src, int n, uint16_t *dst) {
  for (int i = threadIdx.x; i < n; i += (int)blockDim.x) dst[i] = gld(src + i);
  __syncthreads();
}

// Potential item (row chunk x column chunk of a split's functions, both within
// BT): per 16-function block and 128-point tile of the split (at most 32)
// whether some function of the block is in the tile's list, as bits of rb[t]
// (rows) and cb[t] (columns), from the functions' tile masks rm and cm (nr and
// nc of them); and the tiles where both have one, ascending, in tl.  Returns
// their number; every thread of the workgroup calls it (rb, cb, tl, n in LDS).
template <int BT, int NT = kThreads>
__device__ __forceinline__ int potential_tiles(const uint32_t *__restrict__ rm, int nr,
                                               const uint32_t *__restrict__ cm, int nc,
                                               int (&rb)[32], int (&cb)[32], uint8_t (&tl)[32],
                                               int *n) {
  __syncthreads();  // the previous item's readers are done
  if (threadIdx.x < 32) rb[threadIdx.x] = cb[threadIdx.x] = 0;
  __syncthreads();
  // 16 lanes a block: each turns its function's mask into its tiles' bits
  for (int i = threadIdx.x; i < 2 * BT; i += NT) {
    const int f = i < BT ? i : i - BT;
    uint32_t m = i < BT ? (f < nr ? gld(rm + f) : 0u) : (f < nc ? gld(cm + f) : 0u);
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) m |= (uint32_t)__shfl_xor((int)m, o);
    // lane q of the block takes tiles q and q + 16
    int *d = i < BT ? rb : cb;
    const int q = f & 15, bit = 1 << (f >> 4);
    if ((m >> q) & 1u) atomicOr(d + q, bit);
    if ((m >> (q + 16)) & 1u) atomicOr(d + q + 16, bit);
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int t = threadIdx.x & 31;
    const unsigned long long live = __ballot(threadIdx.x < 32 && rb[t] != 0 && cb[t] != 0);
    if (threadIdx.x < 32 && ((live >> t) & 1ull)) tl[__popcll(live & ((1ull << t) - 1ull))] = (uint8_t)t;
    if (threadIdx.x == 0) *n = __popcll(live);
  }
  __syncthreads();
  return *n;
}

// Sums of 4 per-lane values over the 16 lanes of each lane group (the 16 columns
// of an MFMA result block) by recursive halving: at the first two exchanges a
// lane keeps half of the values it still holds and sends the other half, so they
// take 2 + 1 + 1 + 1 shuffles instead of 4 x 4.  Returns the total of value
// `index` in this lane (the groups of 4 lanes l & ~3 share index (l & 12) / 4).
// The addition order is fixed.
template <int O, int m>
struct GroupStep {  // one exchange with lane ^ O while m values are held
  __device__ static __forceinline__ void run(double (&v)[4], int lane, int &index) {
    if constexpr (m > 1) {
      const bool hi = (lane & O) != 0;
#pragma unroll
      for (int k = 0; k < m / 2; ++k) {
        const double send = hi ? v[k] : v[k + m / 2];
        const double keep = hi ? v[k + m / 2] : v[k];
        v[k] = keep + __shfl_xor(send, O);
      }
      if (hi) index += m / 2;
    } else {
      v[0] += __shfl_xor(v[0], O);
    }
    if constexpr (O > 1) GroupStep<O / 2, (m > 1 ? m / 2 : 1)>::run(v, lane, index);
  }
};
__device__ __forceinline__ double group_reduce(double (&v)[4], int lane, int &index) {
  index = 0;
  GroupStep<8, 4>::run(v, lane, index);
  return v[0];
}

// Columns of a share of a tile's nf functions: as many shares as `most` needs,
// their 16-column blocks dealt out evenly.
__device__ __forceinline__ int share_cols(int nf, int most) {
  const int n = (nf + most - 1) / most, nb = (nf + 15) / 16;
  return 16 * ((nb + n - 1) / n);
}

// Functions of a split, padded to whole 16-function blocks: the leading
// dimension of its potential partial.
__device__ __forceinline__ int split_ld(int n) { return (n + 15) & ~15; }

// Share of the nearest centre's Becke cell at or below which a centre's cell is
// left out: na of them are at most 2^-54, a quarter of an ulp of the cells' sum.
__device__ __forceinline__ double becke_negligible(int na) {
  return na <= 1024 ? 5.421010862427522e-20 /* 2^-64 */ : 5.551115123125783e-17 /* 2^-54 */ / na;
}

// One 16 x 16 block of H = W^T Phi into the split's partial.
template <typename T>
__device__ __forceinline__ void put_block(const typename MF<T>::acc &acc, double *H, int ld) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < 4; ++r) gst(H + (long)MF<T>::row(lane, r) * ld + mf_col(lane), (double)acc[r]);
}

}  // namespace pgxc
