// cpic_split_kernels.h -- passes 1 and 2 of the push, a cell's rows and
// arrivals shared by several waves.
//
// One wave per 64 cells, walking their columns serially, needs some thousand
// groups of cells to fill the chip: 32^3 cells are 512 waves for 1024 SIMDs,
// and a 1D deck is one wave.  There the serial walk is all the time there is:
// one row costs a chain of square roots and divides, 1.3 us in FP32 and 2 us
// in FP64, whatever else the chip could do (62 + 39 us for the two passes at
// 32^3 x 32, 130 + 59 us for 32 cells x 64 in FP64).  Here a block of S waves
// owns one group: S rows (or arrivals) at a time, one to a wave.  Their
// contributions meet in LDS, and the waves add them to the cells' sums in row
// (arrival) order, four of the 12 sums to a wave, so the sums are those of the
// serial walk, bit for bit; so is everything else.  The price is 3 LDS writes
// and about 4 reads of 16 bytes per lane and row and a barrier every S rows
// (adding the waves' own sums in a tree at the end was 5 % faster, but changes
// the rounding, which is all the field there is in a quiet start).  On grids
// that fill the chip sharing still pays, with departure masks in LDS and
// per-group counts in place of atomics: 1343 + 770 us became 1281 + 724 us at
// 128^3 x 32, where pass 1 is bound by VALU issue and HBM together and pass 2
// by HBM's random-access rate.
#pragma once

#include "cpic_push_kernels.h"

namespace cpic {

constexpr int kSplitChunk = 2;  // mask words whose departures k_push_split gathers in LDS
constexpr int kTakenWords = 4;  // mask words whose taken rows k_arrive_split notes in LDS

// The contributions of S rows, [S][3][64] quads (jx, jy, jz), in LDS, and the
// sums of the quads that a wave looks after: quad wave, wave + S, ...  With
// two copies of the rows a barrier between writing and reading is enough;
// FP64 keeps one copy (LDS would limit the waves) and waits after reading too.
template <class R, bool K, int S> struct RowSums {
  typedef typename Vec4T<R>::type V4;
  static constexpr int kCopies = sizeof(R) == 4 ? 2 : 1;
  static constexpr int kQuads = (3 + S - 1) / S;
  typedef V4 Rows[kCopies][S][3][64];
  R s[kQuads][4];
  R c[K ? kQuads : 1][4];
  int copy;
  __device__ __forceinline__ void zero() {
    copy = 0;
#pragma unroll
    for (int q = 0; q < kQuads; ++q)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        s[q][k] = 0;
        if (K) c[K ? q : 0][k] = 0;
      }
  }
  __device__ __forceinline__ void add1(int q, int k, R v) {
    if (K) {
      // TwoSum, as LaneAcc
      const R t = s[q][k] + v;
      const R vv = t - s[q][k];
      const R e = (s[q][k] - (t - vv)) + (v - vv);
      c[K ? q : 0][k] += e;
      s[q][k] = t;
    } else {
      s[q][k] += v;
    }
  }
  // the wave's row; zeros (which change no sum) where the lane has none
  __device__ __forceinline__ void put(Rows& rows, int wave, int lane, const R o[12]) {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      V4 v;
      v.x = o[4 * q];
      v.y = o[4 * q + 1];
      v.z = o[4 * q + 2];
      v.w = o[4 * q + 3];
      rows[copy][wave][q][lane] = v;
    }
  }
  // after a barrier: the rows of all waves in order
  __device__ __forceinline__ void add(const Rows& rows, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < kQuads; ++i) {
      const int q = wave + i * S;
      if (q < 3) {
#pragma unroll
        for (int u = 0; u < S; ++u) {
          const V4 v = rows[copy][u][q][lane];
          add1(i, 0, v.x);
          add1(i, 1, v.y);
          add1(i, 2, v.z);
          add1(i, 3, v.w);
        }
      }
    }
    if (kCopies == 2)
      copy ^= 1;
    else
      __syncthreads();
  }
  // the accumulators of voxel v that the wave's sums go to
  __device__ __forceinline__ void fetch(const R* acc, size_t N, int v, int wave,
                                        R (&was)[kQuads][4]) const {
#pragma unroll
    for (int i = 0; i < kQuads; ++i) {
      const int q = wave + i * S;
#pragma unroll
      for (int k = 0; k < 4; ++k) was[i][k] = q < 3 ? acc[(size_t)(4 * q + k) * N + v] : 0;
    }
  }
  // the sums to the accumulators, or onto what they hold, was
  __device__ __forceinline__ void store(R* acc, size_t N, int v, int wave, bool onto,
                                        const R (&was)[kQuads][4]) const {
#pragma unroll
    for (int i = 0; i < kQuads; ++i) {
      const int q = wave + i * S;
      if (q < 3) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const R t = K ? s[i][k] + c[K ? i : 0][k] : s[i][k];
          acc[(size_t)(4 * q + k) * N + v] = onto ? was[i][k] + t : t;
        }
      }
    }
  }
};

// Pass 1 in place (every push but the packing ones), the arithmetic of
// k_push_pass; blockIdx is the group of 64 cells.
//
// Every row issues the same loads and stores on every lane: a lane without a
// particle in the row stores whatever it loaded when another lane of its
// 128-byte line holds one (the row is free in the output column, and arrivals
// overwrite it later), and otherwise its store is dropped by the buffer
// descriptor's range check, so memory only ever sees whole lines (a partly
// written line costs a read-modify-write), and rows past the ends of all the
// columns of a line cost nothing.  The loads of a wave's next row are issued
// before the stores of this one, and with a fixed number of instructions in
// between the wait for them does not wait for those stores.
template <class R, bool K, int S>
__global__ void __launch_bounds__(64 * S) k_push_split(PushPass<R> a) {
  typedef typename Vec4T<R>::type V4;
  typedef RowSums<R, K, S> Sums;
  __shared__ typename Sums::Rows parts;
  __shared__ unsigned long long sdep[kSplitChunk][6][64];
  __shared__ int movers[S];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // (no pass-1 wave raises a flag, so all waves of the block read the same)
  if (__builtin_amdgcn_readfirstlane(*a.err)) return;  // an earlier push failed
  const int grp = blockIdx.x;
  const int ci = grp * 64 + lane;  // < nc_pad
  const bool valid = ci < a.g.nc;
  const int len = valid ? min(a.cs.cnt_in[ci], a.cs.D) : 0;
  const int lmax = wave_max_int(len);
  const int v = valid ? interior_to_voxel(a.g, ci) : 0;
  V4 e0 = {}, e1 = {}, e2 = {}, b0 = {}, b1 = {};
  if (valid) {
    PushPass<R> mine = a;
    if (wave != 0 && a.gather == kGatherStore) mine.gather = kGatherFields;
    cell_interpolator(mine, v, e0, e1, e2, b0, b1);
  }
  Sums sums;
  sums.zero();
  int nmov = 0;
  const size_t MP = a.cs.nc_pad;
  const int MW = a.cs.MW;
  const int nwords = (lmax + 63) >> 6;
  const int gbytes = a.cs.D * 64 * kSlotLen * (int)sizeof(R);
  const __amdgpu_buffer_rsrc_t rows_out = __builtin_amdgcn_make_buffer_rsrc(
      a.cs.out + (size_t)grp * a.cs.D * 64 * kSlotLen, 0, gbytes, kBufferWord3);
  constexpr int kLine = 128 / (kSlotLen * (int)sizeof(R));  // lanes per line
  static_assert(kLine >= 1 && kLine < 64 && (kLine & (kLine - 1)) == 0, "line of slots");
  const int line0 = lane & ~(kLine - 1);
  const R* const dummy = a.cs.in;
  auto occ = [&](int w) -> unsigned long long {
    return (valid && w * 64 < len)
               ? a.cs.mask_in[(size_t)w * MP + ci] & low_bits(len - 64 * w)
               : 0ull;
  };

  for (int w0 = 0; w0 < nwords; w0 += kSplitChunk) {
    const int used = min(kSplitChunk, nwords - w0);
    __syncthreads();  // the previous chunk's words have been written out
    for (int i = threadIdx.x; i < used * 6 * 64; i += 64 * S) (&sdep[0][0][0])[i] = 0;
    __syncthreads();
    const int jend = min(lmax, (w0 + used) * 64);
    unsigned long long m_in = 0;
    int mword = -1;
    auto request = [&](int r, V4& x, V4& y) -> bool {
      if ((r >> 6) != mword && r < jend) {
        mword = r >> 6;
        m_in = occ(mword);
        settle(m_in);
      }
      const bool ok = r < jend && ((m_in >> (r & 63)) & 1ull);
      const V4* src = reinterpret_cast<const V4*>(ok ? a.cs.in + col_slot(ci, r, a.cs.D) * kSlotLen
                                                     : dummy);
      x = src[0];
      y = src[1];
      return ok;
    };
    V4 xa = {}, ya = {};
    bool ha = request(w0 * 64 + wave, xa, ya);
    for (int r0 = w0 * 64; r0 < jend; r0 += S) {
      const int j = r0 + wave;
      V4 xb = {}, yb = {};
      const bool hb = request(j + S, xb, yb);
      settle(xa);
      settle(ya);
      V4 o0 = xa, o1 = ya;
      R o[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
      if (ha) {
        int d;
        if (push_particle(a, e0, e1, e2, b0, b1, xa, ya, o, o0, o1, d)) ++nmov;
        if (d >= 0) atomicOr(&sdep[(j >> 6) - w0][d][lane], 1ull << (j & 63));
      }
      const unsigned long long in_row = __ballot(ha);
      const bool st = (in_row >> line0) & ((1ull << kLine) - 1);
      store_slot(rows_out, st ? (j * 64 + lane) * kSlotLen * (int)sizeof(R) : gbytes, o0, o1);
      sums.put(parts, wave, lane, o);
      __syncthreads();
      sums.add(parts, wave, lane);
      xa = xb;
      ya = yb;
      ha = hb;
    }
    // the chunk's departure words (complete since the last round's barrier),
    // their union, and the occupancy (every row that held a particle)
    for (int i = wave; i < used * 8; i += S) {
      const int u = i >> 3, k = i & 7, w = w0 + u;
      if (k < 6) {
        a.dep[dep_index(k, w, MW, MP, ci)] = sdep[u][k][lane];
      } else if (k == 6) {
        unsigned long long all = 0;
#pragma unroll
        for (int d = 0; d < 6; ++d) all |= sdep[u][d][lane];
        a.dep[dep_index(6, w, MW, MP, ci)] = all;
      } else {
        a.cs.mask_out[(size_t)w * MP + ci] = occ(w);
      }
    }
  }
  for (int w = nwords + wave; w < MW; w += S) a.cs.mask_out[(size_t)w * MP + ci] = 0ull;
  if (valid) {
    R was[Sums::kQuads][4] = {};
    if (a.accumulate) sums.fetch(a.acc, a.ncells, v, wave, was);
    sums.store(a.acc, a.ncells, v, wave, a.accumulate, was);
  }
  const int wm = wave_sum_int(nmov);
  if (lane == 0) movers[wave] = wm;
  __syncthreads();
  if (wave != 0) return;
  // rows in use: up to the last occupied one
  int hi = 0;
  for (int w = (len + 63) >> 6; w > 0 && hi == 0; --w) {
    const unsigned long long m = occ(w - 1);
    if (m) hi = 64 * w - __clzll((long long)m);
  }
  a.cs.cnt_out[ci] = hi;
  if (lane == 0) {
    int all = 0;
#pragma unroll
    for (int u = 0; u < S; ++u) all += movers[u];
    a.grp_movers[grp] = all;
    a.grp_rows[grp] = lmax;
    a.dep_words[grp] = nwords;
  }
}

// The zero bits of a column's occupancy words in ascending order (its holes,
// then the rows past its end), read as they were before any arrival: the rows
// taken are noted elsewhere until the block is done.
struct FreeRows {
  int hw;
  unsigned long long freeb;
  // w0: occupancy word 0
  __device__ __forceinline__ void start(unsigned long long w0, int D) {
    hw = 0;
    freeb = ~w0 & low_bits(D);
  }
  // the next free row below D, or -1; occ: the lane's words, stride apart
  __device__ __forceinline__ int next(int D, const unsigned long long* occ, size_t stride) {
    while (freeb == 0) {
      if ((hw + 1) * 64 >= D) return -1;
      ++hw;
      freeb = ~occ[(size_t)hw * stride] & low_bits(D - hw * 64);
    }
    const int b = __ffsll((long long)freeb) - 1;
    freeb &= freeb - 1;
    return hw * 64 + b;
  }
};

// Pass 2: every particle that left a cell in pass 1 continues in the cell
// across the face it crossed; blockIdx counts groups of 64 cells.  The owner
// of that cell finds it through the departure masks of its six neighbours,
// reads it from the neighbour's column, recomputes its displacement and first
// streak (the same operations as pass 1, without the deposit, which pass 1
// made), and runs the next streak.  Afterwards each cell releases the rows of
// its own departures.
//
// The arrivals of a cell that left rows of mask word w of their cells are
// numbered in face, then row order, and arrival i is taken by wave i % S.
// Where it is stored depends on the arrivals before it (the row of one that
// stays, the record slot of one that crosses again), so the waves tell each
// other what became of theirs, S arrivals at a time, and rows and record slots
// are handed out in arrival order.
template <class R, bool K, int S>
__global__ void __launch_bounds__(64 * S) k_arrive_split(ArrivePass<R> a) {
  typedef typename Vec4T<R>::type V4;
  typedef RowSums<R, K, S> Sums;
  __shared__ typename Sums::Rows parts;
  __shared__ unsigned long long went[6][64];  // the word of departures being taken in
  __shared__ int sources[6][64];              // the cells they left
  __shared__ int written[6][64];              // words that pass 1 wrote for those cells
  __shared__ unsigned long long taken[kTakenWords][64];  // rows handed out
  __shared__ signed char fate[Sums::kCopies][S][64];     // -1 none, 0..5 face crossed, 6 stays
  __shared__ int failed;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int MW = a.cs.MW;
  // groups in reverse order: the first blocks dispatched take the groups
  // pass 1 wrote last, whose lines the 256 MB Infinity Cache still holds, and
  // the last ones end at the groups the next pass 1 starts with
  const int grp = gridDim.x - 1 - blockIdx.x;
  const int ci = grp * 64 + lane;  // < nc_pad
  const bool valid = ci < a.g.nc;
  const size_t MP = a.cs.nc_pad;
  const size_t NC = a.g.nc;
  // everything the arrivals' addresses depend on is requested at once: the
  // pass is a chain of dependent loads, and word 0 is there to be read
  // whether or not pass 1 wrote it (it is dropped if not).  Wave d % S looks
  // after the arrivals through face d; they come from across the opposite one.
  int v = 0;
  {
    int nb[6] = {0, 0, 0, 0, 0, 0};
    if (valid) face_neighbors6(a.g, ci, nb, v);
#pragma unroll
    for (int d = 0; d < 6; ++d) {
      if (d % S != wave) continue;
      const int src = nb[d < 3 ? d + 3 : d - 3];
      const int n = a.dep_words[src >> 6];
      const unsigned long long bits = a.dep[dep_index(d, 0, MW, MP, src)];
      sources[d][lane] = src;
      written[d][lane] = valid ? n : 0;
      went[d][lane] = valid && n > 0 ? bits : 0;
    }
  }
  const unsigned long long* const occ = a.cs.mask_out + ci;
  const unsigned long long occ0 = *occ;
  int len = min(a.cs.cnt_out[ci], a.cs.D);  // rows in use (kept by wave 0)
  // and what the end of the pass updates: the wave's first word, and its sums
  // (where two waves share a group they are six quads a lane, whose registers
  // would cost FP64 a third of the waves, on grids that hide the latency anyway)
  constexpr bool kFetchEarly = S > 2;
  Sums sums;
  R was[Sums::kQuads][4];
  if (kFetchEarly) sums.fetch(a.acc, a.ncells, v, wave, was);
  const int w1 = min(wave, MW - 1);
  const unsigned long long occ1 = occ[(size_t)w1 * MP];
  const unsigned long long own1 = a.dep[dep_index(6, w1, MW, MP, ci)];
  const int own_words = min(a.dep_words[grp], MW);
  // one look at the flags for the block: a wave of this launch may raise one
  // meanwhile, and all waves must reach the same barriers
  if (threadIdx.x == 0) failed = *a.err;
  unsigned long long* const deep = a.taken + ci;  // the words past kTakenWords
  for (int w = wave; w < MW; w += S) {
    if (w < kTakenWords)
      taken[w][lane] = 0;
    else
      deep[(size_t)w * MP] = 0;
  }
  __syncthreads();
  if (failed) return;
  sums.zero();
  FreeRows rows;
  rows.start(occ0, a.cs.D);
  unsigned long long kd_lo = 0, kd_hi = 0;  // records per face, three 21-bit counts each
  auto records = [&](int d) {
    return (int)(((d < 3 ? kd_lo : kd_hi) >> (21 * (d < 3 ? d : d - 3))) & 0x1fffff);
  };
  bool any = false;
  int nw = 0;
#pragma unroll
  for (int d = 0; d < 6; ++d) nw = max(nw, written[d][lane]);
  nw = min(wave_max_int(nw), MW);
  for (int w = 0; w < nw; ++w) {
    if (w > 0) {
      __syncthreads();  // the previous word has been taken in
#pragma unroll
      for (int d = 0; d < 6; ++d)
        if (d % S == wave)
          went[d][lane] =
              w < written[d][lane] ? a.dep[dep_index(d, w, MW, MP, sources[d][lane])] : 0;
      __syncthreads();
    }
    // arrivals through the faces before d, in bits 9 d ... 9 d + 8 (a word has
    // 64 rows, six words 384)
    unsigned long long before_face = 0;
    int total = 0;
#pragma unroll
    for (int d = 0; d < 6; ++d) {
      before_face |= (unsigned long long)total << (9 * d);
      total += __popcll(went[d][lane]);
    }
    any |= total > 0;
    const int tmax = wave_max_int(total);
    auto request = [&](int i, V4& x, V4& y) -> bool {
      const R* slot = a.cs.in;  // lanes without an arrival read one shared slot
      const bool ok = i < total;
      if (ok) {
        int d = 0, n = i;
#pragma unroll
        for (int e = 1; e < 6; ++e) {
          const int p = (int)(before_face >> (9 * e)) & 511;
          if (i >= p) d = e, n = i - p;
        }
        unsigned long long bits = went[d][lane];
        for (; n > 0; --n) bits &= bits - 1;
        const int r = 64 * w + __ffsll((long long)bits) - 1;
        slot = a.cs.out + col_slot(sources[d][lane], r, a.cs.D) * kSlotLen;
      }
      const V4* p = reinterpret_cast<const V4*>(slot);
      x = p[0];
      y = p[1];
      return ok;
    };
    V4 xa = {}, ya = {};
    bool ha = false;
    if (tmax > 0) ha = request(wave, xa, ya);
    for (int i0 = 0; i0 < tmax; i0 += S) {
      V4 xb = {}, yb = {};
      const bool hb = request(i0 + S + wave, xb, yb);
      settle(xa);
      settle(ya);
      R pos[3], rem[3];
      R o[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
      int f = -1;
      if (ha) {
        f = arrive_particle(a, xa, ya, o, pos, rem);
        if (f < 0) f = 6;
      }
      sums.put(parts, wave, lane, o);
      fate[sums.copy][wave][lane] = (signed char)f;
      __syncthreads();
      int before = 0, stay = 0;  // stayers of lower waves, of all waves
      int k = 0;                 // record slot of this wave's arrival
      if (f >= 0 && f < 6) k = records(f);
#pragma unroll
      for (int u = 0; u < S; ++u) {
        const int c = fate[sums.copy][u][lane];
        if (c == 6) {
          ++stay;
          before += u < wave ? 1 : 0;
        } else if (c >= 0) {
          k += (u < wave && c == f) ? 1 : 0;
          if (c < 3)
            kd_lo += 1ull << (21 * c);
          else
            kd_hi += 1ull << (21 * (c - 3));
        }
      }
      for (int u = 0; u < stay; ++u) {
        const int row = rows.next(a.cs.D, occ, MP);
        if (wave == 0 && row >= 0) {
          const unsigned long long bit = 1ull << (row & 63);
          if (row < 64 * kTakenWords)
            taken[row >> 6][lane] |= bit;
          else
            deep[(size_t)(row >> 6) * MP] |= bit;
          len = max(len, row + 1);
        }
        if (f == 6 && u == before) {
          if (row >= 0)
            store_particle(a.cs, ci, row, pos[0], pos[1], pos[2], xa.w, ya.x, ya.y, ya.z, ya.w);
          else
            atomicOr(a.err, kErrColumnFull);
        }
      }
      if (f >= 0 && f < 6)
        put_record(a.out, a.ovf, a.g, ci, f, k, pos, rem, xa.w, ya.x, ya.y, ya.z, ya.w, a.err);
      sums.add(parts, wave, lane);
      xa = xb;
      ya = yb;
      ha = hb;
    }
  }
  __syncthreads();
  if (!valid) return;
  // the rows taken become occupied and those of the cell's own departures
  // free: other lanes may still be reading those rows in this pass, but nobody
  // writes them before the next one, which is the first that can hand them out
  // again
  for (int w = wave; w < MW; w += S) {
    const unsigned long long add = w < kTakenWords ? taken[w][lane] : deep[(size_t)w * MP];
    const unsigned long long own =
        w >= own_words ? 0ull : w == wave ? own1 : a.dep[dep_index(6, w, MW, MP, ci)];
    if (add | own) {
      unsigned long long* m = a.cs.mask_out + (size_t)w * MP + ci;
      *m = ((w == wave ? occ1 : *m) | add) & ~own;
    }
  }
  if (any) {
    if (!kFetchEarly) sums.fetch(a.acc, a.ncells, v, wave, was);
    sums.store(a.acc, a.ncells, v, wave, true, was);
  }
  if (wave != 0) return;
  a.cs.cnt_out[ci] = len;
#pragma unroll
  for (int d = 0; d < 6; ++d)
    a.out.cnt[(size_t)d * NC + ci] = (unsigned char)min(records(d), a.out.M);
}

}  // namespace cpic
