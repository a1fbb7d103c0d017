// cpic_small_kernels.h -- the two particle passes of grids of few cells.
//
// The reference's 1D decks have some tens of cells.  With a lane per cell they
// are one wave, or 8 that share it, on one of 256 CUs: 42 us in pass 1 for 32
// cells of 64 particles in FP64, 26 in pass 2.  Here the roles are swapped: a
// wave owns one cell, its lanes the rows (pass 1) or the arrivals (pass 2) of
// that cell, so that a column of 64 particles takes one particle's time and
// the cells spread over the chip: 11.7 and 13.4 us.  The contributions meet in
// LDS and are added in row (arrival) order, so every result has the bits of
// the other kernels'.
#pragma once

#include "cpic_push_kernels.h"

namespace cpic {

constexpr int kSmallWaves = 4;      // cells per block: a 128-byte line of FP32 slots
constexpr int kSmallWords = 16;     // mask words whose taken rows k_arrive_cells notes in LDS
constexpr int kSmallCells = 4096;   // cells of a grid that uses them

// Contributions of up to 64 rows, padded against bank conflicts, and the sums
// of the cell: lane k < 12 of the wave holds sum k.
template <class R, bool K> struct CellSums {
  typedef R Rows[64][13];
  R s, c;
  __device__ __forceinline__ void zero() { s = c = 0; }
  // o: the lane's contributions (of rows n and more none are taken)
  __device__ __forceinline__ void add(Rows& rows, int lane, int n, const R o[12]) {
#pragma unroll
    for (int k = 0; k < 12; ++k) rows[lane][k] = o[k];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane < 12) {
      for (int r = 0; r < n; ++r) {
        const R v = rows[r][lane];
        if (K) {
          const R t = s + v;
          const R vv = t - s;
          c += (s - (t - vv)) + (v - vv);
          s = t;
        } else {
          s += v;
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  __device__ __forceinline__ void store(R* acc, size_t N, int v, int lane, bool onto) const {
    if (lane >= 12) return;
    R* p = acc + (size_t)lane * N + v;
    const R t = K ? s + c : s;
    *p = onto ? *p + t : t;
  }
};

// Pass 1 (as k_push_split), one wave per cell and one lane per row.
template <class R, bool K>
__global__ void __launch_bounds__(64 * kSmallWaves) k_push_cells(PushPass<R> a) {
  typedef typename Vec4T<R>::type V4;
  __shared__ typename CellSums<R, K>::Rows parts[kSmallWaves];
  __shared__ int movers[kSmallWaves];
  if (__builtin_amdgcn_readfirstlane(*a.err)) return;  // an earlier push failed
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int ci = blockIdx.x * kSmallWaves + wave;
  const int grp = ci >> 6;
  const size_t MP = a.cs.nc_pad;
  const int MW = a.cs.MW;
  int nmov = 0;
  if (ci < a.g.nc) {
    // words of the departure masks to write: those of the group's rows
    const int lens = min(a.cs.cnt_in[(grp << 6) + lane], a.cs.D);
    const int lmax = wave_max_int(lens);
    const int len = __shfl(lens, ci & 63, 64);
    const int nwords = (lmax + 63) >> 6;
    const int v = interior_to_voxel(a.g, ci);
    V4 e0, e1, e2, b0, b1;
    {
      PushPass<R> mine = a;
      if (lane != 0 && a.gather == kGatherStore) mine.gather = kGatherFields;
      cell_interpolator(mine, v, e0, e1, e2, b0, b1);
    }
    CellSums<R, K> sums;
    sums.zero();
    int hi = 0;
    for (int w = 0; w < nwords; ++w) {
      const int left = len - 64 * w;
      const unsigned long long m =
          left > 0 ? a.cs.mask_in[(size_t)w * MP + ci] & low_bits(left) : 0ull;
      const int row = 64 * w + lane;
      R o[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
      int d = -1;
      bool moved = false;
      if ((m >> lane) & 1ull) {
        const size_t slot = col_slot(ci, row, a.cs.D) * kSlotLen;
        const V4* src = reinterpret_cast<const V4*>(a.cs.in + slot);
        V4 o0, o1;
        moved = push_particle(a, e0, e1, e2, b0, b1, src[0], src[1], o, o0, o1, d);
        V4* dst = reinterpret_cast<V4*>(a.cs.out + slot);
        dst[0] = o0;
        dst[1] = o1;
      }
      nmov += __popcll(__ballot(moved));
      // lane k < 6 writes the departures through face k, 6 their union, 7 the
      // occupancy
      unsigned long long word = lane == 7 ? m : 0ull, any = 0;
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const unsigned long long gone = __ballot(d == k);
        any |= gone;
        if (lane == k) word = gone;
      }
      if (lane == 6) word = any;
      if (lane < 7)
        a.dep[dep_index(lane, w, MW, MP, ci)] = word;
      else if (lane == 7)
        a.cs.mask_out[(size_t)w * MP + ci] = word;
      if (m) {
        hi = 64 * (w + 1) - __clzll((long long)m);
        sums.add(parts[wave], lane, hi - 64 * w, o);
      }
    }
    for (int w = nwords + lane; w < MW; w += 64) a.cs.mask_out[(size_t)w * MP + ci] = 0ull;
    sums.store(a.acc, a.ncells, v, lane, a.accumulate);
    if (lane == 0) {
      a.cs.cnt_out[ci] = hi;
      // (the same values from each of the group's waves)
      a.grp_rows[grp] = lmax;
      a.dep_words[grp] = nwords;
    }
  }
  if (lane == 0) movers[wave] = nmov;
  __syncthreads();
  if (threadIdx.x == 0) {
    int all = 0;
#pragma unroll
    for (int u = 0; u < kSmallWaves; ++u) all += movers[u];
    a.grp_movers[blockIdx.x] = all;
  }
}

// Pass 2 (as k_arrive_split), one wave per cell and one lane per arrival.
template <class R, bool K>
__global__ void __launch_bounds__(64 * kSmallWaves) k_arrive_cells(ArrivePass<R> a) {
  typedef typename Vec4T<R>::type V4;
  __shared__ typename CellSums<R, K>::Rows parts[kSmallWaves];
  __shared__ unsigned long long taken[kSmallWaves][kSmallWords];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int ci = blockIdx.x * kSmallWaves + wave;
  if (ci >= a.g.nc) return;  // (no barrier below: a wave is on its own)
  if (__builtin_amdgcn_readfirstlane(*a.err)) return;  // this push already failed
  const size_t MP = a.cs.nc_pad;
  const int MW = a.cs.MW, D = a.cs.D;
  int v;
  int nb[6];
  face_neighbors6(a.g, ci, nb, v);
  // lane d < 6 looks after the arrivals through face d, which come from across
  // the opposite one
  const int src = sel6(lane < 6 ? lane : 0, nb[3], nb[4], nb[5], nb[0], nb[1], nb[2]);
  const int written = lane < 6 ? a.dep_words[src >> 6] : 0;
  const int nw = min(wave_max_int(written), MW);
  // rows handed out: in LDS, and for the words of columns that are deeper (a
  // grid of few particles has rows for all of them) in global memory, where
  // the lines of other cells' words are shared, so past the vector cache
  unsigned long long* const deep = a.taken + ci;
  for (int w = lane; w < MW; w += 64) {
    if (w < kSmallWords)
      taken[wave][w] = 0;
    else
      __hip_atomic_store(&deep[(size_t)w * MP], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (MW > kSmallWords) __threadfence();
  const unsigned long long* const occ = a.cs.mask_out + ci;
  int hw = 0;  // the first word with free rows that are still to be had, and those
  unsigned long long freeb = ~occ[0] & low_bits(D);
  int len = min(a.cs.cnt_out[ci], D);
  int kd[6] = {0, 0, 0, 0, 0, 0};
  CellSums<R, K> sums;
  sums.zero();
  bool any = false;
  // the n-th free row from (h, f) on, which move up to it; -1 if there is none
  auto free_row = [&](int& h, unsigned long long& f, int n) -> int {
    for (;;) {
      const int c = __popcll(f);
      if (n < c) break;
      n -= c;
      if ((h + 1) * 64 >= D) {
        f = 0;
        return -1;
      }
      ++h;
      f = ~occ[(size_t)h * MP] & low_bits(D - 64 * h);
    }
    for (; n > 0; --n) f &= f - 1;
    return 64 * h + __ffsll((long long)f) - 1;
  };
  for (int w = 0; w < nw; ++w) {
    const unsigned long long mine =
        lane < 6 && w < written ? a.dep[dep_index(lane, w, MW, MP, src)] : 0ull;
    int total = 0, p[6];
    unsigned long long went[6];
#pragma unroll
    for (int d = 0; d < 6; ++d) {
      went[d] = __shfl(mine, d, 64);
      p[d] = total;
      total += __popcll(went[d]);
    }
    if (total == 0) continue;
    any = true;
    for (int i0 = 0; i0 < total; i0 += 64) {
      const int i = i0 + lane;
      R pos[3], rem[3];
      R o[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
      V4 pa = {}, pb = {};
      int f = -1;  // -1 none, 0..5 face crossed, 6 stays
      if (i < total) {
        const int d = (i >= p[1]) + (i >= p[2]) + (i >= p[3]) + (i >= p[4]) + (i >= p[5]);
        unsigned long long bits = d == 0   ? went[0]
                                  : d == 1 ? went[1]
                                  : d == 2 ? went[2]
                                  : d == 3 ? went[3]
                                  : d == 4 ? went[4]
                                           : went[5];
        for (int n = i - sel6(d, p[0], p[1], p[2], p[3], p[4], p[5]); n > 0; --n) bits &= bits - 1;
        const int r = 64 * w + __ffsll((long long)bits) - 1;
        const int sc = sel6(d, nb[3], nb[4], nb[5], nb[0], nb[1], nb[2]);
        const V4* s = reinterpret_cast<const V4*>(a.cs.out + col_slot(sc, r, D) * kSlotLen);
        pa = s[0];
        pb = s[1];
        f = arrive_particle(a, pa, pb, o, pos, rem);
        if (f < 0) f = 6;
      }
      // rows and record slots in arrival order
      const unsigned long long below = (1ull << lane) - 1;
      const unsigned long long stays = __ballot(f == 6);
      int k = 0;
#pragma unroll
      for (int d = 0; d < 6; ++d) {
        const unsigned long long goes = __ballot(f == d);
        if (f == d) k = kd[d] + __popcll(goes & below);
        kd[d] += __popcll(goes);
      }
      int row = -1;
      if (f == 6) {
        int h = hw;
        unsigned long long fb = freeb;
        row = free_row(h, fb, __popcll(stays & below));
      }
      if (stays) {
        // past the rows just taken (none is left if the last of them was not
        // there either)
        if (free_row(hw, freeb, __popcll(stays) - 1) >= 0) freeb &= freeb - 1;
      }
      if (f == 6) {
        if (row >= 0) {
          store_particle(a.cs, ci, row, pos[0], pos[1], pos[2], pa.w, pb.x, pb.y, pb.z, pb.w);
          const unsigned long long bit = 1ull << (row & 63);
          if (row < 64 * kSmallWords)
            atomicOr(&taken[wave][row >> 6], bit);
          else
            atomicOr(&deep[(size_t)(row >> 6) * MP], bit);
        } else {
          atomicOr(a.err, kErrColumnFull);
        }
      } else if (f >= 0) {
        put_record(a.out, a.ovf, a.g, ci, f, k, pos, rem, pa.w, pb.x, pb.y, pb.z, pb.w, a.err);
      }
      len = max(len, wave_max_int(row + 1));
      sums.add(parts[wave], lane, min(64, total - i0), o);
    }
  }
  // the rows taken become occupied, those of the cell's own departures free
  const int own_words = min(a.dep_words[ci >> 6], MW);
  if (MW > kSmallWords) __threadfence();
  for (int w = lane; w < MW; w += 64) {
    const unsigned long long add =
        w < kSmallWords ? taken[wave][w]
                        : __hip_atomic_load(&deep[(size_t)w * MP], __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long own = w < own_words ? a.dep[dep_index(6, w, MW, MP, ci)] : 0ull;
    if (add | own) {
      unsigned long long* m = a.cs.mask_out + (size_t)w * MP + ci;
      *m = (*m | add) & ~own;
    }
  }
  if (any) sums.store(a.acc, a.ncells, v, lane, true);
  if (lane == 0) a.cs.cnt_out[ci] = len;
  if (lane < 6)
    a.out.cnt[(size_t)lane * a.g.nc + ci] = (unsigned char)min(
        sel6(lane, kd[0], kd[1], kd[2], kd[3], kd[4], kd[5]), a.out.M);
}

}  // namespace cpic
