// cpic_small_kernels.h -- the two particle passes of grids of few cells.
//
// The reference's 1D decks have some tens of cells.  With a lane per cell they
// are one wave, or 8 that share it, on one of 256 CUs: 42 us in pass 1 for 32
// cells of 64 particles in FP64, 26 in pass 2.  Here the roles are swapped: a
// wave owns one cell, its lanes the rows (pass 1) or the arrivals (pass 2) of
// that cell, so that a column of 64 particles takes one particle's time and
// the cells spread over the chip: 10.5 and 7.5 us.  The contributions meet in
// LDS and are added in row (arrival) order, so every result has the bits of
// the other kernels'.
#pragma once

#include "cpic_push_kernels.h"

namespace cpic {

constexpr int kSmallWaves = 4;      // cells per block: a 128-byte line of FP32 slots
constexpr int kSmallWords = 64;     // mask words whose taken rows k_arrive_cells notes in LDS
constexpr int kSmallCells = 4096;   // cells of a grid that uses them in any case

// Contributions of up to 64 rows, [12][rows], and the sums of the cell: lane
// k < 12 of the wave holds sum k.  The padding puts the lanes' reads of four
// rows in different banks.
template <class R, bool K> struct CellSums {
  typedef typename Vec4T<R>::type V4;
  struct alignas(sizeof(V4)) Rows {
    R v[12][64 + 4];
  };
  R s, c;
  __device__ __forceinline__ void zero() { s = c = 0; }
  // o: the lane's contributions (zeros in rows n and more).  The sum of rows in
  // order is a chain of additions; read one row at a time it was a chain of LDS
  // latencies too, so kAhead rows are read together (the zeros past row n
  // change no sum).
  static constexpr int kAhead = K ? 8 : 16;
  __device__ __forceinline__ void add(Rows& rows, int lane, int n, const R o[12]) {
#pragma unroll
    for (int k = 0; k < 12; ++k) rows.v[k][lane] = o[k];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane < 12) {
      for (int r0 = 0; r0 < n; r0 += kAhead) {
        V4 u[kAhead / 4];
#pragma unroll
        for (int r = 0; r < kAhead / 4; ++r)
          u[r] = *reinterpret_cast<const V4*>(&rows.v[lane][r0 + 4 * r]);
#pragma unroll
        for (int r = 0; r < kAhead / 4; ++r) {
          add1(u[r].x);
          add1(u[r].y);
          add1(u[r].z);
          add1(u[r].w);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  __device__ __forceinline__ void add1(R v) {
    if (K) {
      const R t = s + v;
      const R vv = t - s;
      c += (s - (t - vv)) + (v - vv);
      s = t;
    } else {
      s += v;
    }
  }
  // onto: whether the sums are to be added to what the accumulators hold, was
  __device__ __forceinline__ void store(R* acc, size_t N, int v, int lane, bool onto, R was) const {
    if (lane >= 12) return;
    const R t = K ? s + c : s;
    acc[(size_t)lane * N + v] = onto ? was + t : t;
  }
};

// Pass 1 (as k_push_split), one wave per cell and one lane per row.
//
// A cell's pass is a chain of dependent loads, 0.5 us and more each on a chip
// that is mostly idle.  The slots and masks of the first two words are there to
// be read whether or not the column reaches that far, and are requested with
// everything else.
template <class R, bool K>
__global__ void __launch_bounds__(64 * kSmallWaves) k_push_cells(PushPass<R> a) {
  typedef typename Vec4T<R>::type V4;
  __shared__ typename CellSums<R, K>::Rows parts[kSmallWaves];
  __shared__ int movers[kSmallWaves];
  const int failed = *a.err;  // an earlier push
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int ci = blockIdx.x * kSmallWaves + wave;
  const int grp = ci >> 6;
  const size_t MP = a.cs.nc_pad;
  const int MW = a.cs.MW, D = a.cs.D;
  int nmov = 0;
  if (ci < a.g.nc) {
    auto slot_of = [&](int row) {
      return reinterpret_cast<const V4*>(a.cs.in + col_slot(ci, min(row, D - 1), D) * kSlotLen);
    };
    V4 xa = slot_of(lane)[0], xb = slot_of(lane)[1];
    V4 ya = slot_of(64 + lane)[0], yb = slot_of(64 + lane)[1];
    unsigned long long m0 = a.cs.mask_in[ci];
    unsigned long long m1 = a.cs.mask_in[(size_t)min(1, MW - 1) * MP + ci];
    // words of the departure masks to write: those of the group's rows
    int lens = min(a.cs.cnt_in[(grp << 6) + lane], D);
    const int v = interior_to_voxel(a.g, ci);
    V4 e0, e1, e2, b0, b1;
    {
      PushPass<R> mine = a;
      if (lane != 0 && a.gather == kGatherStore) mine.gather = kGatherFields;
      cell_interpolator(mine, v, e0, e1, e2, b0, b1);
    }
    R was = a.accumulate ? a.acc[(size_t)min(lane, 11) * a.ncells + v] : 0;
    settle(xa);
    settle(xb);
    settle(ya);
    settle(yb);
    settle(m0);
    settle(m1);
    settle(lens);
    settle(was);
    if (__builtin_amdgcn_readfirstlane(failed)) return;  // (all waves of the block)
    const int lmax = wave_max_int(lens);
    const int len = __shfl(lens, ci & 63, 64);
    const int nwords = (lmax + 63) >> 6;
    CellSums<R, K> sums;
    sums.zero();
    int hi = 0;
    for (int w = 0; w < nwords; ++w) {
      if (w > 1) m0 = a.cs.mask_in[(size_t)w * MP + ci];
      const int left = len - 64 * w;
      const unsigned long long m = left > 0 ? m0 & low_bits(left) : 0ull;
      const int row = 64 * w + lane;
      R o[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
      int d = -1;
      bool moved = false;
      if ((m >> lane) & 1ull) {
        if (w > 1) {
          xa = slot_of(row)[0];
          xb = slot_of(row)[1];
        }
        V4 o0, o1;
        moved = push_particle(a, e0, e1, e2, b0, b1, xa, xb, o, o0, o1, d);
        V4* dst = reinterpret_cast<V4*>(a.cs.out + col_slot(ci, row, D) * kSlotLen);
        dst[0] = o0;
        dst[1] = o1;
      }
      xa = ya;
      xb = yb;
      m0 = m1;
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
    sums.store(a.acc, a.ncells, v, lane, a.accumulate, was);
    if (lane == 0) {
      a.cs.cnt_out[ci] = hi;
      // (the same values from each of the group's waves)
      a.grp_rows[grp] = lmax;
      a.dep_words[grp] = nwords;
    }
  }
  if (failed) return;
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
//
// Ten words of the six neighbours' departures at a time, a lane each: the
// arrivals of all are numbered by a scan over the lanes (words, then faces, then
// rows), and each lane lists its own in LDS, 64 arrivals at a time.
template <class R, bool K>
__global__ void __launch_bounds__(64 * kSmallWaves) k_arrive_cells(ArrivePass<R> a) {
  typedef typename Vec4T<R>::type V4;
  constexpr int kWordsAtOnce = 10;
  __shared__ typename CellSums<R, K>::Rows parts[kSmallWaves];
  __shared__ unsigned long long taken[kSmallWaves][kSmallWords];
  __shared__ unsigned long long arrivals[kSmallWaves][64];  // the slots they are in
  __shared__ int free_rows[kSmallWaves][64];
  const int failed = *a.err;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int ci = blockIdx.x * kSmallWaves + wave;
  if (ci >= a.g.nc) return;  // (no barrier below: a wave is on its own)
  const size_t MP = a.cs.nc_pad;
  const int MW = a.cs.MW, D = a.cs.D;
  int v;
  int nb[6];
  face_neighbors6(a.g, ci, nb, v);
  // the lane's face and word; arrivals through a face come from across the
  // opposite one
  const int face = lane % 6, word = lane / 6;
  const int src = sel6(face, nb[3], nb[4], nb[5], nb[0], nb[1], nb[2]);
  // all that does not depend on other loads is requested at once: the first
  // departure words, and what the end of the pass updates (word `lane` of the
  // cell's occupancy and own departures, sum `lane`)
  int written = min(a.dep_words[src >> 6], MW);
  unsigned long long gone = a.dep[dep_index(face, min(word, MW - 1), MW, MP, src)];
  const int wl = min(lane, MW - 1);
  unsigned long long occ = a.cs.mask_out[(size_t)wl * MP + ci];
  unsigned long long own = a.dep[dep_index(6, wl, MW, MP, ci)];
  int own_words = min(a.dep_words[ci >> 6], MW);
  R was = a.acc[(size_t)min(lane, 11) * a.ncells + v];
  int len = min(a.cs.cnt_out[ci], D);
  settle(written);
  settle(gone);
  settle(occ);
  settle(own);
  settle(own_words);
  settle(was);
  settle(len);
  if (__builtin_amdgcn_readfirstlane(failed)) return;  // this push already failed
  const int nw = wave_max_int(written);
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
  const unsigned long long below = (1ull << lane) - 1;
  // the first word with free rows that are still to be had, and those
  int hw = 0;
  unsigned long long freeb = ~__shfl(occ, 0, 64) & low_bits(D);
  int kd[6] = {0, 0, 0, 0, 0, 0};
  CellSums<R, K> sums;
  sums.zero();
  bool any = false;
  for (int w0 = 0; w0 < nw; w0 += kWordsAtOnce) {
    const int w = w0 + word;
    if (w0 > 0) gone = a.dep[dep_index(face, min(w, MW - 1), MW, MP, src)];
    unsigned long long bits = word < kWordsAtOnce && w < written ? gone : 0ull;
    const int mine = __popcll(bits);
    int end = mine;  // inclusive scan
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
      const int o = __shfl_up(end, s, 64);
      if (lane >= s) end += o;
    }
    const int total = __shfl(end, 63, 64);
    int next = end - mine;  // number of the lane's next arrival
    any |= total > 0;
    for (int i0 = 0; i0 < total; i0 += 64) {
      for (; bits && next < i0 + 64; ++next, bits &= bits - 1)
        arrivals[wave][next - i0] = col_slot(src, 64 * w + __ffsll((long long)bits) - 1, D);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      R pos[3], rem[3];
      R o[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
      V4 pa = {}, pb = {};
      int f = -1;  // -1 none, 0..5 face crossed, 6 stays
      if (i0 + lane < total) {
        const V4* s = reinterpret_cast<const V4*>(a.cs.out + arrivals[wave][lane] * kSlotLen);
        pa = s[0];
        pb = s[1];
        f = arrive_particle(a, pa, pb, o, pos, rem);
        if (f < 0) f = 6;
      }
      // rows and record slots in arrival order
      const unsigned long long stays = __ballot(f == 6);
      int k = 0;
#pragma unroll
      for (int d = 0; d < 6; ++d) {
        const unsigned long long goes = __ballot(f == d);
        if (f == d) k = kd[d] + __popcll(goes & below);
        kd[d] += __popcll(goes);
      }
      const int need = __popcll(stays);
      int have = 0;
      while (have < need) {
        // the lane's row of word hw, if free, is the place-th row handed out
        const int place = have + __popcll(freeb & below);
        const bool takes = ((freeb >> lane) & 1ull) && place < need;
        if (takes) free_rows[wave][place] = 64 * hw + lane;
        const unsigned long long took = __ballot(takes);
        if (took) {
          have += __popcll(took);
          freeb &= ~took;
          len = max(len, 64 * (hw + 1) - __clzll((long long)took));
          if (lane == 0) {
            if (hw < kSmallWords)
              taken[wave][hw] |= took;
            else
              atomicOr(&deep[(size_t)hw * MP], took);
          }
        }
        if (freeb == 0) {
          if ((hw + 1) * 64 >= D) break;
          ++hw;
          freeb = ~(hw < 64 ? __shfl(occ, hw, 64) : a.cs.mask_out[(size_t)hw * MP + ci]) &
                  low_bits(D - 64 * hw);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (f == 6) {
        const int place = __popcll(stays & below);
        if (place < have)
          store_particle(a.cs, ci, free_rows[wave][place], pos[0], pos[1], pos[2], pa.w, pb.x,
                         pb.y, pb.z, pb.w);
        else
          atomicOr(a.err, kErrColumnFull);
      } else if (f >= 0) {
        put_record(a.out, a.ovf, a.g, ci, f, k, pos, rem, pa.w, pb.x, pb.y, pb.z, pb.w, a.err);
      }
      sums.add(parts[wave], lane, min(64, total - i0), o);
    }
  }
  // the rows taken become occupied, those of the cell's own departures free
  if (MW > kSmallWords) __threadfence();
  for (int w = lane; w < MW; w += 64) {
    const unsigned long long add =
        w < kSmallWords ? taken[wave][w]
                        : __hip_atomic_load(&deep[(size_t)w * MP], __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
    if (w >= 64) {
      occ = a.cs.mask_out[(size_t)w * MP + ci];
      own = a.dep[dep_index(6, w, MW, MP, ci)];
    }
    const unsigned long long left = w < own_words ? own : 0ull;
    if (add | left) a.cs.mask_out[(size_t)w * MP + ci] = (occ | add) & ~left;
  }
  if (any) sums.store(a.acc, a.ncells, v, lane, true, was);
  if (lane == 0) a.cs.cnt_out[ci] = len;
  if (lane < 6)
    a.out.cnt[(size_t)lane * a.g.nc + ci] = (unsigned char)min(
        sel6(lane, kd[0], kd[1], kd[2], kd[3], kd[4], kd[5]), a.out.M);
}

}  // namespace cpic
