// cpic_block_kernels.h -- the stages after the particle passes of grids of few
// cells, in one workgroup.
//
// Six launches follow the two particle passes of a step: two finish passes, the
// spill pass and three field stages, each a chain of a few dependent loads over
// at most a thread per cell.  On a 1D deck they took 21 of a step's 50 us: each
// launch starts with cold caches and drains before the next.  Up to
// kBlockThreads cells one workgroup runs them all, with barriers in the
// launches' places: 11 us for 32 cells, of the 30 us that a step of 32 cells x 64
// takes in FP64 now (the host, to which the push's status goes before the field
// stages, queues the next step meanwhile).  Every value is computed by the same
// operations, and every sum in the same order, as in the kernels that larger grids
// run.
//
// (The particle passes stay outside: with whole steps in one workgroup the same
// deck took 60 us a step, where separate launches took 50, bound by its CU's
// vector cache, to which the rows of a cell, a wave's lanes, are 64 lines.)
//
// Visibility: what passes from wave to wave here goes through one CU's
// write-through vector cache, where a barrier is enough.  What atomics change
// (the spill pass, the error flags, the overflow count) they change in the L2,
// and is read with atomic loads or after an agent-scope fence.
#pragma once

#include "cpic_small_kernels.h"

namespace cpic {

constexpr int kBlockThreads = 1024;
constexpr int kBlockWaves = kBlockThreads / 64;

template <class R> struct BlockFields {
  R* fields;
  const R* acc;
  Grid g;
  R cx, cy, cz;     // unload's scales
  R hpx, hpy, hpz;  // advance_b, half a step
  R px, py, pz, cj;
};

template <class R> struct BlockFinish {
  FinishPass<R> pass[2];
  SpillPass<R> spill;
};

// What a launch leaves to the host, as publish_push does.
struct BlockStatus {
  const int* grp_rows;
  int ngroups;  // at most 64
  int* err;
  unsigned* ovf_count;
  int seq;
  PushStatus* host;
};

__device__ __forceinline__ int load_flag(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The stages of a step after pass 2: finish and spill passes, the field
// stages, the energies (row, if not null) and the push's status.
template <class R> struct BlockTail {
  BlockFinish<R> finish;
  BlockFields<R> fields;
  BlockStatus status;
  double* row;
};

// The argument of k_block_tail, where it lies.  Each phase looks it up for
// itself: kept in registers from phase to phase (and the addresses that follow
// from it and from the thread's number, for which phase_thread does the same)
// it would spill.
template <class R> __device__ __forceinline__ const BlockTail<R>& phase_args() {
  auto p = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const BlockTail<R>*)p;
}
__device__ __forceinline__ int phase_thread() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// The finish passes and the spill pass; all threads call it after a barrier.
// crossed: LDS, zero.  grids of at most kBlockThreads cells, a thread per cell.
template <class R, bool K>
__device__ __forceinline__ void block_finish(int& crossed) {
#pragma unroll 1
  for (int pass = 0; pass < 2; ++pass) {
    const int t = phase_thread();
    const FinishPass<R>& f = phase_args<R>().finish.pass[pass];
    if ((t & ~63) < f.g.nc && finish_cell<R, K>(f, t, 0)) crossed = 1;
    __syncthreads();
    if (!__builtin_amdgcn_readfirstlane(crossed)) break;
  }
  const SpillPass<R>& sp = phase_args<R>().finish.spill;
  const unsigned n = __builtin_amdgcn_readfirstlane(
      __hip_atomic_load(sp.ovf.count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  __syncthreads();  // the count has been read
  if (n == 0) return;
  const int t = phase_thread();
  spill_records(sp, min(n, (unsigned)sp.ovf.cap), (unsigned)t, kBlockThreads);
  if (t == 0)
    __hip_atomic_store(sp.ovf.count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __threadfence();  // the atomics' results are what the next loads see
  __syncthreads();
}

// The field stages, a thread per interior voxel; returns after the ghost copies
// without a barrier.  sums: LDS, per wave the E^2 and B^2 of its voxels if
// energy.  Ghosts are read at the interior voxels that they copy, and written
// once, at the end, by a loop over the grid: the kernels of larger grids have
// each interior voxel write up to 26 of them, whose straight-line code took
// longer to fetch than this loop takes.
template <class R>
__device__ __forceinline__ void block_fields(bool energy, double (&sums)[kBlockWaves][2]) {
  {
    // unload, the J fold, advance_b
    const BlockFields<R>& f = phase_args<R>().fields;
    const Grid g = f.g;
    const int t = phase_thread();
    if (t < g.nx * g.ny * g.nz) {
      const int x = 1 + t % g.nx, y = 1 + (t / g.nx) % g.ny, z = 1 + t / (g.nx * g.ny);
      const int i = voxel(g, x, y, z);
      currents_at(f.fields, f.acc, g, x, y, z, i, f.cx, f.cy, f.cz);
      R eb[6];
      advance_b_at(f.fields, g, i, f.hpx, f.hpy, f.hpz, eb);
    }
  }
  __syncthreads();
  {
    // advance_e
    const BlockFields<R>& f = phase_args<R>().fields;
    const Grid g = f.g;
    const size_t N = g.ncells;
    R* ex = f.fields;
    R* ey = f.fields + N;
    R* ez = f.fields + 2 * N;
    const R* bx = f.fields + 3 * N;
    const R* by = f.fields + 4 * N;
    const R* bz = f.fields + 5 * N;
    const R* jx = f.fields + 6 * N;
    const R* jy = f.fields + 7 * N;
    const R* jz = f.fields + 8 * N;
    const int mx = g.nx + 1, my = g.ny + 1, mz = g.nz + 1;
    const R px = f.px, py = f.py, pz = f.pz, cj = f.cj;
    for (int u = phase_thread(); u < mx * my * mz; u += kBlockThreads) {
      const int x = 1 + u % mx, y = 1 + (u / mx) % my, z = 1 + u / (mx * my);
      const int i = voxel(g, x, y, z);
      const int xs = x > g.nx ? 1 : x, ys = y > g.ny ? 1 : y, zs = z > g.nz ? 1 : z;
      const int s = voxel(g, xs, ys, zs);
      const int sx = voxel(g, x == 1 ? g.nx : x - 1, ys, zs);
      const int sy = voxel(g, xs, y == 1 ? g.ny : y - 1, zs);
      const int sz = voxel(g, xs, ys, z == 1 ? g.nz : z - 1);
      const R b_x = bx[s], b_y = by[s], b_z = bz[s];
      ex[i] = ex[i] + (-cj * jx[s]) + (py * (b_z - bz[sy]) - pz * (b_y - by[sz]));
      ey[i] = ey[i] + (-cj * jy[s]) + (pz * (b_x - bx[sz]) - px * (b_z - bz[sx]));
      ez[i] = ez[i] + (-cj * jz[s]) + (px * (b_y - by[sx]) - py * (b_x - bx[sy]));
    }
  }
  __syncthreads();
  double v[2] = {0, 0};
  {
    const BlockFields<R>& f = phase_args<R>().fields;
    const Grid g = f.g;
    const int t = phase_thread();
    if (t < g.nx * g.ny * g.nz) {
      const int x = 1 + t % g.nx, y = 1 + (t / g.nx) % g.ny, z = 1 + t / (g.nx * g.ny);
      R eb[6];
      advance_b_at(f.fields, g, voxel(g, x, y, z), f.hpx, f.hpy, f.hpz, eb);
      const double e0 = eb[0], e1 = eb[1], e2 = eb[2], b0 = eb[3], b1 = eb[4], b2 = eb[5];
      v[0] = e0 * e0 + e1 * e1 + e2 * e2;
      v[1] = b0 * b0 + b1 * b1 + b2 * b2;
    }
  }
  __syncthreads();
  const BlockFields<R>& f = phase_args<R>().fields;
  const Grid g = f.g;
  const int t = phase_thread();
  const int X = g.sy, Y = g.sz / g.sy;
  for (int u = t; u < g.ncells; u += kBlockThreads) {
    const int x = u % X, y = (u / X) % Y, z = u / g.sz;
    const int s = voxel(g, x == 0 ? g.nx : x > g.nx ? 1 : x, y == 0 ? g.ny : y > g.ny ? 1 : y,
                        z == 0 ? g.nz : z > g.nz ? 1 : z);
    if (s == u) continue;
    R c[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) c[k] = f.fields[(size_t)(3 + k) * g.ncells + s];
#pragma unroll
    for (int k = 0; k < 6; ++k) f.fields[(size_t)(3 + k) * g.ncells + u] = c[k];
  }
  if (!energy) return;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    v[q] = wave_sum(v[q]);
    if ((t & 63) == 0) sums[t >> 6][q] = v[q];
  }
}

// One thread, after a barrier: the energies of block_fields' sums, added as
// k_advance_b_energy's blocks of kBlock voxels and k_reduce_final add them.
__device__ __forceinline__ void block_energies(const double (&sums)[kBlockWaves][2],
                                               double* row) {
  constexpr int kPer = kBlock / 64;
  static_assert(kBlockWaves == 4 * kPer, "four blocks' sums");
  for (int q = 0; q < 2; ++q) {
    double p[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      p[b] = 0;
#pragma unroll
      for (int k = 0; k < kPer; ++k) p[b] += sums[kPer * b + k][q];
    }
    row[q] = 0.5 * ((p[0] + p[2]) + (p[1] + p[3]));
  }
}

// The calling wave.
__device__ __forceinline__ void block_publish(const BlockStatus& s, int lane) {
  const int m = wave_max_int(lane < s.ngroups ? s.grp_rows[lane] : 0);
  if (lane != 0) return;
  __hip_atomic_store(s.ovf_count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&s.host->err, load_flag(s.err), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&s.host->rows, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&s.host->seq, s.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <class R, bool K>
__global__ void __launch_bounds__(kBlockThreads) k_block_tail(BlockTail<R>) {
  __shared__ double sums[kBlockWaves][2];
  __shared__ int crossed, failed;
  const int* const err = phase_args<R>().status.err;
  if (threadIdx.x == 0) {
    crossed = 0;
    failed = load_flag(err);
  }
  __syncthreads();
  if (!__builtin_amdgcn_readfirstlane(failed)) block_finish<R, K>(crossed);
  // before the field stages: the host may be waiting for it to queue the next step
  const BlockStatus& status = phase_args<R>().status;
  if (threadIdx.x >= kBlockThreads - 64) block_publish(status, threadIdx.x & 63);
  const bool energy = phase_args<R>().row != nullptr;
  block_fields<R>(energy, sums);
  __syncthreads();
  double* const row = phase_args<R>().row;
  if (energy && threadIdx.x == 0) block_energies(sums, row);
}

}  // namespace cpic
