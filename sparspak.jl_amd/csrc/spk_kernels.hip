// Kernels of the numeric phase. See spk_kernels.h for the storage model.
#include "spk_kernels.h"

namespace spk {

// Index of the calling thread's wave in its workgroup, as a wave-uniform
// (scalar) value so that per-wave index arithmetic stays on the scalar unit.
__device__ inline int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x / 64); }

// Orders one wave's LDS accesses: every access before it is complete and
// visible to the wave's other lanes before any access after it. The
// wavefront-scope fences emit no instructions (one wave's LDS operations
// complete in issue order) but keep the compiler from moving LDS loads or
// stores across the barrier, which the barrier intrinsic alone does not.
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Column range of piece p (0-based supernode): first column (0-based) and
// width.
__device__ inline void piece_cols(const DevSym& s, int64_t p, int64_t& c0,
                                  int64_t& w) {
  c0 = s.xsuper[p] - 1;
  w = s.xsuper[p + 1] - s.xsuper[p];
}

// First (front-local) column of the piece holding own column c.
__device__ inline int piece_start_of_col(const DevSym& s, int64_t fc0, int c) {
  return (int)(s.xsuper[s.snode[fc0 + c] - 1] - 1 - fc0);
}

template <typename T>
__global__ void fill_kernel(T* __restrict__ a, int64_t len, T v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < len; i += stride) a[i] = v;
}

// Every entry of A (its slot map: lnz slot, -2 - unz slot, or -1) in its
// front: the slot's column (lnz) or row (unz) is an own column of the front.
// Without `out` counts the entries of every front column (cnt, index fvec[f]
// + c); with it takes cnt as the columns' next free positions. SPD entries
// below the diagonal appear at both positions. Once per pattern; the slots'
// columns are found by bisection.
__global__ void front_entries_kernel(DevSym s, const int64_t* __restrict__ amap, int64_t nnz,
                                     int64_t* __restrict__ cnt, AEnt* __restrict__ out) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  // last i in [0, m) with v[i] <= x
  auto last_le = [](const auto* v, int64_t m, int64_t x) {
    int64_t lo = 0, hi = m - 1;
    while (lo < hi) {
      const int64_t mid = (lo + hi + 1) >> 1;
      if (v[mid] <= x)
        lo = mid;
      else
        hi = mid - 1;
    }
    return lo;
  };
  for (; k < nnz; k += stride) {
    const int64_t a = amap[k];
    if (a == -1) continue;
    const int64_t slot = a >= 0 ? a : -a - 2;
    const int64_t g = last_le(a >= 0 ? s.xlnz : s.xunz, s.n, slot + 1);
    const int f = (int)last_le(s.fc0, s.nfront, g);
    const int own = (int)(g - s.fc0[f]);
    const int other = (int)(slot - (a >= 0 ? s.lcol[g] : s.ucol[g]));
    auto put = [&](int r, int c) {
      const unsigned long long at = atomicAdd(
          reinterpret_cast<unsigned long long*>(cnt + s.fvec[f] + c), 1ull);
      if (out) out[at] = AEnt{k, r, c};
    };
    put(a >= 0 ? other : own, a >= 0 ? own : other);
    if (s.sym && other != own) put(own, other);
  }
}

// Exclusive sums of cnt[0 .. n) in place, cnt[n] their total, and a copy of
// them (the columns' next free positions), in three launches: workgroup b's
// total of its kScan elements (PART 0), the totals' exclusive sums by one
// workgroup (1), the elements' (2). Once per pattern.
constexpr int kScan = 4096;
template <int PART>
__global__ void __launch_bounds__(kWG)
scan_kernel(int64_t* __restrict__ cnt, int64_t n, int64_t* __restrict__ part, int nb,
            int64_t* __restrict__ copy) {
  __shared__ int64_t sh[kWG];
  const int tid = threadIdx.x;
  // exclusive sums of v over the workgroup's threads; total: all of them
  auto scan = [&](int64_t v, int64_t& total) {
    sh[tid] = v;
    __syncthreads();
    for (int o = 1; o < kWG; o *= 2) {
      const int64_t x = tid >= o ? sh[tid - o] : 0;
      __syncthreads();
      sh[tid] += x;
      __syncthreads();
    }
    total = sh[kWG - 1];
    const int64_t r = sh[tid] - v;
    __syncthreads();
    return r;
  };
  int64_t total;
  if constexpr (PART == 1) {
    int64_t base = 0;
    for (int i0 = 0; i0 < nb; i0 += kWG) {
      const int i = i0 + tid;
      const int64_t v = i < nb ? part[i] : 0;
      const int64_t x = scan(v, total);
      if (i < nb) part[i] = base + x;
      base += total;
    }
    if (tid == 0) cnt[n] = copy[n] = base;
  } else {
    constexpr int E = kScan / kWG;
    const int64_t b0 = (int64_t)blockIdx.x * kScan + tid * E;
    int64_t v[E], sum = 0;
#pragma unroll
    for (int k = 0; k < E; ++k) {
      v[k] = b0 + k < n ? cnt[b0 + k] : 0;
      sum += v[k];
    }
    int64_t x = scan(sum, total);
    if constexpr (PART == 0) {
      if (tid == 0) part[blockIdx.x] = total;
    } else {
      x += part[blockIdx.x];
#pragma unroll
      for (int k = 0; k < E; ++k) {
        if (b0 + k < n) cnt[b0 + k] = copy[b0 + k] = x;
        x += v[k];
      }
    }
  }
}

// The assembly's items and the small fronts' entries from the columns'
// pointers (aptr, index fvec[f] + column).
__global__ void asm_items_kernel(const int32_t* __restrict__ front, const int32_t* __restrict__ col,
                                 int64_t n, const int32_t* __restrict__ fL,
                                 const int64_t* __restrict__ foff, const int64_t* __restrict__ fvec,
                                 const int64_t* __restrict__ aptr, AsmItem* __restrict__ out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) {
    const int f = front[i], j = col[i], L = fL[f];
    const int64_t a0 = aptr[fvec[f] + j];
    out[i] = AsmItem{foff[f] + (int64_t)j * L, a0, L, (int32_t)(aptr[fvec[f] + j + 1] - a0)};
  }
}
__global__ void small_entries_kernel(SmallDesc* __restrict__ d, int n,
                                     const int64_t* __restrict__ aptr) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  d[i].a0 = aptr[d[i].fvec];
  d[i].an = (int32_t)(aptr[d[i].fvec + d[i].L] - d[i].a0);
}

// ---------------------------------------------------------------------------
// Large fronts: the L x L work matrix lives in the arena.
// ---------------------------------------------------------------------------

// U part of a large front (rows of a piece, columns right of it) moves
// between unz (U12^T panels: a piece's U rows are its panel's columns) and
// the work matrix through 64-row x nq tiles transposed in LDS, so that both
// sides are read/written along their contiguous dimension. For SPD input the
// U entries are the transposed L entries (lnz panel rows below the block).
template <typename T, bool STORE>
__global__ void __launch_bounds__(kWG)
large_utile_kernel(DevSym s, const int32_t* __restrict__ it_front,
                   const int32_t* __restrict__ it_piece, const int32_t* __restrict__ it_r0,
                   T* __restrict__ lnz, T* __restrict__ unz, T* __restrict__ arena) {
  const int64_t vs = blockIdx.y;  // value set
  lnz += vs * s.vs_lnz;
  unz += vs * s.vs_unz;
  arena += vs * s.vs_arena;
  __shared__ T tile[64 * 97];
  const int f = it_front[blockIdx.x];
  const int p = it_piece[blockIdx.x];
  const int r0 = it_r0[blockIdx.x];
  const int L = s.fL[f];
  const int64_t fc0 = s.fc0[f];
  int64_t pc0, nq64;
  piece_cols(s, p, pc0, nq64);
  const int nq = (int)nq64;
  const int cq = (int)(pc0 - fc0);
  const int ul = L - cq - nq;
  const int nr = min(64, ul - r0);
  const int ld = nq + 1;
  T* F = arena + s.foff[f];
  const bool from_l = s.sym && !STORE;
  T* src = from_l ? lnz + (s.xlnz[pc0] - 1) + nq : unz + (s.xunz[pc0] - 1);
  const int64_t sld = from_l ? (int64_t)(L - cq) : (int64_t)ul;
  if (!STORE) {
    for (int idx = threadIdx.x; idx < 64 * nq; idx += kWG) {
      const int r = idx % 64, c = idx / 64;
      if (r < nr) tile[r * ld + c] = src[(r0 + r) + c * sld];
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < 64 * nq; idx += kWG) {
      const int c = idx % nq, r = idx / nq;
      if (r < nr) F[(cq + c) + (int64_t)(cq + nq + r0 + r) * L] = tile[r * ld + c];
    }
  } else {
    for (int idx = threadIdx.x; idx < 64 * nq; idx += kWG) {
      const int c = idx % nq, r = idx / nq;
      if (r < nr) tile[r * ld + c] = F[(cq + c) + (int64_t)(cq + nq + r0 + r) * L];
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < 64 * nq; idx += kWG) {
      const int r = idx % 64, c = idx / 64;
      if (r < nr) unz[(s.xunz[pc0] - 1) + (r0 + r) + (int64_t)c * ul] = tile[r * ld + c];
    }
  }
}

// Assembly from lnz/unz (the stateless drop-ins, whose arguments hold
// _inmatrix!'s output). One workgroup per (front, column j): the column's L part from lnz (rows
// from its piece's first row), zeros in the update block, then the
// children's update-matrix columns that map to j, one child after the other
// (rows of different children may coincide). Runs after large_utile_kernel
// has placed the U part. With staged set the column is assembled in LDS
// (dynamic, L elements): read once (the U part from the front, the rest from
// lnz or zero), the children's columns added there, written once; otherwise
// the children's entries are added in the front in place. The item and each
// child's entry come resolved (InitItem, EaItem); the next child's entry is
// read while the current child's column is added.
template <typename T>
__global__ void __launch_bounds__(kWG)
large_init_kernel(DevSym s, const InitItem* __restrict__ items,
                  const int64_t* __restrict__ it_ea, const EaItem* __restrict__ ea,
                  const T* __restrict__ lnz, T* __restrict__ arena, int staged) {
  const int64_t vs = blockIdx.y;  // value set
  lnz += vs * s.vs_lnz;
  arena += vs * s.vs_arena;
  extern __shared__ unsigned char smem_raw[];
  const int item = blockIdx.x;
  const InitItem m = items[item];
  const int L = m.L, W = m.W, j = m.j;
  T* F = arena + m.fcol;
  const int64_t e0 = it_ea[item], e1 = it_ea[item + 1];
  EaItem en = ea[e0 < e1 ? e0 : 0];
  if (staged && !s.sym) {
    T* Fs = reinterpret_cast<T*>(smem_raw);
    // rows below r1 come from lnz (own column) or are zero (update column);
    // rows above it are the U part already in the front
    const int r1 = m.r1;
    const T* lc = (m.lcb >= 0) ? lnz + m.lcb : nullptr;
    for (int r0 = threadIdx.x; r0 < L; r0 += 16 * kWG) {
      T v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int r = r0 + u * kWG;
        v[u] = (r >= L) ? T(0) : (r < r1) ? F[r] : (lc ? lc[r] : T(0));
      }
#pragma unroll
      for (int u = 0; u < 16; ++u)
        if (r0 + u * kWG < L) Fs[r0 + u * kWG] = v[u];
    }
    __syncthreads();
    for (int64_t e = e0; e < e1; ++e) {
      const EaItem ec = en;
      if (e + 1 < e1) en = ea[e + 1];
      const int Rc = ec.Rc;
      const int32_t* rel = s.relmap + ec.rel;
      const T* col = arena + ec.col;
      for (int tp0 = threadIdx.x; tp0 < Rc; tp0 += 8 * kWG) {
        int ri[8];
        T cv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int tp = tp0 + u * kWG;
          ri[u] = (tp < Rc) ? rel[tp] : 0;
          cv[u] = (tp < Rc) ? col[tp] : T(0);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (tp0 + u * kWG < Rc) Fs[ri[u]] += cv[u];
      }
      __syncthreads();
    }
    for (int r0 = threadIdx.x; r0 < L; r0 += 8 * kWG) {
      T v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = (r0 + u * kWG < L) ? Fs[r0 + u * kWG] : T(0);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (r0 + u * kWG < L) F[r0 + u * kWG] = v[u];
    }
    return;
  }
  if (j < W) {
    const int cp = m.r1;
    const T* lc = lnz + m.lcb;
    if (s.sym) {  // lower triangle only: the diagonal block's upper part is U
      for (int r = cp + threadIdx.x; r < L; r += kWG)
        if (r >= j) F[r] = lc[r];
        else F[r] = lnz[s.lcol[m.fc0 + r] + j];
    } else {
      // eight loads in flight per thread
      for (int r0 = cp + threadIdx.x; r0 < L; r0 += 8 * kWG) {
        T v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = (r0 + u * kWG < L) ? lc[r0 + u * kWG] : T(0);
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (r0 + u * kWG < L) F[r0 + u * kWG] = v[u];
      }
    }
  } else {
    for (int r = W + threadIdx.x; r < L; r += kWG) F[r] = T(0);
  }
  __syncthreads();
  for (int64_t e = e0; e < e1; ++e) {
    const EaItem ec = en;
    if (e + 1 < e1) en = ea[e + 1];
    const int Rc = ec.Rc;
    const int32_t* rel = s.relmap + ec.rel;
    const T* col = arena + ec.col;
    for (int tp0 = threadIdx.x; tp0 < Rc; tp0 += 4 * kWG) {
      int ri[4];
      T cv[4], fv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int tp = tp0 + u * kWG;
        ri[u] = (tp < Rc) ? rel[tp] : 0;
        cv[u] = (tp < Rc) ? col[tp] : T(0);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) fv[u] = F[ri[u]];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (tp0 + u * kWG < Rc) F[ri[u]] = fv[u] + cv[u];
    }
    __syncthreads();
  }
}

// One wave per front column, four per workgroup: the staged (LDS) assembly
// of large_init_kernel for LU levels whose longest column fits a quarter of
// the LDS budget, so that the many short columns of the lower levels take a
// quarter of the workgroups. A child's update rows are distinct, and one
// wave's LDS operations complete in issue order, so the children are added
// one after another without barriers, in the same order as there. Stateless
// LU factors (double) of 193 x 171, 32^3 and 44^3, three each: the assemblies
// of their 327 levels 8.60 ms with a workgroup per column throughout, 6.70 ms
// with this form where it fits (288 of them).
template <typename T>
__global__ void __launch_bounds__(kWG)
large_init_wave_kernel(DevSym s, const InitItem* __restrict__ items,
                       const int64_t* __restrict__ it_ea, const EaItem* __restrict__ ea,
                       const T* __restrict__ lnz, T* __restrict__ arena, int nitems, int maxL) {
  const int64_t vs = blockIdx.y;  // value set
  lnz += vs * s.vs_lnz;
  arena += vs * s.vs_arena;
  extern __shared__ unsigned char smem_raw[];
  const int lane = threadIdx.x % 64, wave = wave_id();
  const int item = blockIdx.x * 4 + wave;
  if (item >= nitems) return;  // no workgroup barrier below
  T* Fs = reinterpret_cast<T*>(smem_raw) + (size_t)wave * maxL;
  const InitItem m = items[item];
  const int L = m.L;
  T* F = arena + m.fcol;
  const int64_t e0 = it_ea[item], e1 = it_ea[item + 1];
  EaItem en = ea[e0 < e1 ? e0 : 0];
  const int r1 = m.r1;
  const T* lc = (m.lcb >= 0) ? lnz + m.lcb : nullptr;
  for (int r0 = lane; r0 < L; r0 += 8 * 64) {
    T v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int r = r0 + u * 64;
      v[u] = (r >= L) ? T(0) : (r < r1) ? F[r] : (lc ? lc[r] : T(0));
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (r0 + u * 64 < L) Fs[r0 + u * 64] = v[u];
  }
  wave_lds_sync();
  for (int64_t e = e0; e < e1; ++e) {
    const EaItem ec = en;
    if (e + 1 < e1) en = ea[e + 1];
    const int Rc = ec.Rc;
    const int32_t* rel = s.relmap + ec.rel;
    const T* col = arena + ec.col;
    for (int tp0 = lane; tp0 < Rc; tp0 += 8 * 64) {
      int ri[8];
      T cv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int tp = tp0 + u * 64;
        ri[u] = (tp < Rc) ? rel[tp] : 0;
        cv[u] = (tp < Rc) ? col[tp] : T(0);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (tp0 + u * 64 < Rc) Fs[ri[u]] += cv[u];
    }
    wave_lds_sync();
  }
  for (int r0 = lane; r0 < L; r0 += 8 * 64) {
    T v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = (r0 + u * 64 < L) ? Fs[r0 + u * 64] : T(0);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (r0 + u * 64 < L) F[r0 + u * 64] = v[u];
  }
}

// Assembly of a large front's column j from A's values: zero, A's entries
// of the column (distinct rows), then the children's update-matrix columns
// that map to j, one child after the other in a fixed order (rows of
// different children may coincide), summed in LDS and written once. G
// threads per column: a workgroup, or a wave (four columns per workgroup, no
// barriers: one wave's LDS operations complete in issue order) where the
// level's longest column fits 16 KB; columns longer than the LDS are summed
// in place (staged 0). The next batch of a child's rows (8 per thread, the
// next child's when this one ends) is requested before the current one is
// added. HBM-bound: L^2 entries written and the children's read. Reading
// the panels of a zeroed and scattered lnz/unz instead, transposing their U
// part into the front first, cost in the same pass at 64^3 (double) 0.43 ms
// of zeroing, 1.7 ms of transposition and the panels read once more: the
// factor and solve pass 81.0 -> 79.5 ms, elasticity 40^3 (float, SPD, whose
// columns were summed in place in HBM) 91.3 -> 80.7 ms, 32^3 double
// 9.57 -> 9.28 ms, 100^2 double 2.56 -> 2.46 ms.
template <typename T, int G>
__device__ __attribute__((always_inline)) void large_assemble_body(
    const DevSym& s, const AsmArgs& a, int b, const double* __restrict__ nzval,
    T* __restrict__ arena, unsigned char* smem_raw) {
  constexpr int U = 8;
  const int grp = (G == kWG) ? 0 : wave_id();
  const int gt = (G == kWG) ? (int)threadIdx.x : (int)threadIdx.x % 64;
  const int item = b * (kWG / G) + grp;
  if (item >= a.nitems) return;  // a whole wave (no workgroup barrier below) or workgroup
  auto gsync = [] {
    if constexpr (G == kWG)
      __syncthreads();
    else
      wave_lds_sync();
  };
  const AsmItem m = a.items[item];
  const int L = m.L;
  T* F = arena + m.fcol;
  T* Fs = a.staged ? reinterpret_cast<T*>(smem_raw) + (size_t)grp * a.maxL : F;
  int64_t e = a.it_ea[item];
  const int64_t e1 = a.it_ea[item + 1];
  // the batch in flight: rows t0 + gt + u G of child `cur`
  EaItem cur = a.ea[e < e1 ? e : 0];
  int t0 = 0;
  int ri[U];
  T cv[U];
  auto request = [&]() {
    const int32_t* rel = s.relmap + cur.rel;
    const T* col = arena + cur.col;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = t0 + gt + u * G;
      ri[u] = (t < cur.Rc) ? rel[t] : -1;
      cv[u] = (t < cur.Rc) ? col[t] : T(0);
    }
  };
  if (e < e1) request();
  for (int r = gt; r < L; r += G) Fs[r] = T(0);
  gsync();
  for (int i = gt; i < m.an; i += G) {
    const AEnt en = a.aent[m.a0 + i];
    Fs[en.r] = (T)nzval[en.k];
  }
  gsync();
  while (e < e1) {
    int rj[U];
    T cw[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      rj[u] = ri[u];
      cw[u] = cv[u];
    }
    t0 += U * G;
    const bool last = t0 >= cur.Rc;
    if (last) {
      t0 = 0;
      if (++e < e1) cur = a.ea[e];
    }
    if (e < e1) request();
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (rj[u] >= 0) Fs[rj[u]] += cw[u];
    if (last) gsync();
  }
  if (!a.staged) return;
  for (int r0 = gt; r0 < L; r0 += U * G) {
    T v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = (r0 + u * G < L) ? Fs[r0 + u * G] : T(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (r0 + u * G < L) F[r0 + u * G] = v[u];
  }
}

template <typename T, int G>
__global__ void __launch_bounds__(kWG)
large_assemble_kernel(DevSym s, AsmArgs a, const double* __restrict__ nzval, int64_t nnz,
                      T* __restrict__ arena) {
  const int64_t vs = blockIdx.y;  // value set
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  large_assemble_body<T, G>(s, a, blockIdx.x, nzval + vs * nnz, arena + vs * s.vs_arena, smem_raw);
}

// L part of the own columns back to lnz (contiguous per column).
template <typename T>
__global__ void __launch_bounds__(kWG)
large_writeback_kernel(DevSym s, const int32_t* __restrict__ it_front,
                       const int32_t* __restrict__ it_col,
                       T* __restrict__ lnz, T* __restrict__ unz,
                       const T* __restrict__ arena) {
  const int64_t vs = blockIdx.y;  // value set
  lnz += vs * s.vs_lnz;
  unz += vs * s.vs_unz;
  arena += vs * s.vs_arena;
  const int item = blockIdx.x;
  const int f = it_front[item];
  const int j = it_col[item];
  const int L = s.fL[f], W = s.fW[f];
  if (j >= W) return;
  const int64_t fc0 = s.fc0[f];
  const T* F = arena + s.foff[f] + (int64_t)j * L;
  const int cp = piece_start_of_col(s, fc0, j);
  T* lc = lnz + s.lcol[fc0 + j];
  for (int r0 = cp + threadIdx.x; r0 < L; r0 += 8 * kWG) {
    T v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = (r0 + u * kWG < L) ? F[r0 + u * kWG] : T(0);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (r0 + u * kWG < L) lc[r0 + u * kWG] = v[u];
  }
}

// Descriptor of workgroup b: the last one whose wg_begin <= b.
template <typename Desc>
__device__ inline int find_blk(const Desc* d, int nd, int b) {
  int lo = 0, hi = nd - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (d[mid].wg_begin <= b)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// ---------------------------------------------------------------------------
// Large fronts, blocked. The pieces of a front are taken in groups (blocks)
// of consecutive pieces spanning columns [c0, c1) (at most 128 columns).
// Each block takes three launches:
//
//  blk_diag_kernel     one workgroup per block factors the bw x bw diagonal
//                      region [c0, c1)^2 in LDS, piece by piece, exactly as
//                      the reference eliminates a supernode
//                      (SpkLUFactor.jl:230-240): LU with row interchanges
//                      inside the piece's nq x nq diagonal block, the
//                      interchanges applied to the piece's own columns and
//                      those right of it but never to earlier pieces' L
//                      columns, L21 = A21 U11^-1 for the region rows below,
//                      U12 = L11^-1 P A12 for the region columns right of
//                      it, then the update of the rest of the region.
//  blk_offdiag_kernel  rows below the block: X = A U_blk^-1 (U_blk = the
//                      upper triangle of the factored region, one piece at a
//                      time), and columns right of the block: per piece the
//                      earlier pieces' contribution, the piece's interchanges
//                      and its unit-lower solve — the left-looking order of
//                      the reference, so every entry is the reference's.
//  blk_gemm_kernel     trailing update A22 -= L21 U12. Blocks are taken in
//                      groups (8 by default): after each block but the last
//                      of a group only the border of the group's remaining
//                      blocks (their columns, and their rows right of them)
//                      is updated; after the last, the rest of the trailing
//                      matrix receives the whole group at once, with inner
//                      dimension up to 8 x 128 — an eighth of the
//                      read-modify-write traffic of one update per block.
// ---------------------------------------------------------------------------

// Copy of an nr x nc tile (nr <= 128) from a column-major HBM array (leading
// dimension lds) into LDS at dst[r * DR + c * DC]: lane = row (two halves),
// the four waves take interleaved columns, eight loads in flight per thread.
template <typename T, int DR, int DC>
__device__ inline void load_tile(const T* __restrict__ src, int64_t lds, int nr, int nc,
                                 T* __restrict__ dst) {
  const int w = threadIdx.x / 64;
  for (int r = threadIdx.x % 64; r < nr; r += 64) {
    for (int cb = w; cb < nc; cb += 32) {
      const T* sp = src + r + (int64_t)cb * lds;
      T v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = (cb + 4 * u < nc) ? sp[(int64_t)(4 * u) * lds] : T(0);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (cb + 4 * u < nc) dst[r * DR + (cb + 4 * u) * DC] = v[u];
    }
  }
}

// The reverse copy: dst[r + c * ldd] = src[r * DR + c * DC].
template <typename T, int DR, int DC>
__device__ inline void store_tile(T* __restrict__ dst, int64_t ldd, int nr, int nc,
                                  const T* __restrict__ src) {
  const int w = threadIdx.x / 64;
  for (int r = threadIdx.x % 64; r < nr; r += 64)
    for (int c = w; c < nc; c += 4) dst[r + (int64_t)c * ldd] = src[r * DR + c * DC];
}

// Cross-lane moves inside rows of 16 lanes (DPP): quad_perm [1,0,3,2],
// quad_perm [2,3,0,1], row_half_mirror, row_mirror.
template <int CTRL>
__device__ inline double dpp_mov(double v) {
  const long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(u & 0xffffffffll), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                          (unsigned long long)(unsigned)lo));
}
template <int CTRL>
__device__ inline float dpp_mov(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ inline double rdlane(double v, int l) {
  const long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(u & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane((int)(u >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                          (unsigned long long)(unsigned)lo));
}
__device__ inline float rdlane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// Wave-uniform maximum of v over the 64 lanes (all lanes active).
template <typename T>
__device__ inline T wave_max(T v) {
  v = fmax(v, dpp_mov<0xB1>(v));   // lanes ^1
  v = fmax(v, dpp_mov<0x4E>(v));   // lanes ^2
  v = fmax(v, dpp_mov<0x141>(v));  // mirror inside 8
  v = fmax(v, dpp_mov<0x140>(v));  // mirror inside 16
  return fmax(fmax(rdlane(v, 0), rdlane(v, 16)), fmax(rdlane(v, 32), rdlane(v, 48)));
}

// Wave-uniform minimum of v over the 64 lanes (all lanes active).
__device__ inline int wave_min(int v) {
  v = min(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, false));
  return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// Leading dimension of the diagonal region in LDS (blocks are at most 128
// columns wide); a compile-time stride turns every column offset into an
// immediate LDS offset.
constexpr int kRLD = 129;
// Most columns of one piece (the SPD limit 90, rounded up).
constexpr int kMaxNq = 96;

// One thread's triangular solve against a piece's diagonal block, in place
// in LDS: X[j XS] (j < nq) becomes
//   x_j = (a_j - sum_{k<j} x_k M(k, j)) * r_j,   M(k, j) = M[k MK + j MJ],
// r_j = 1 / M(j, j) (or rd[j] when given; 1 when UNIT). Columns go in
// blocks of eight: the earlier columns' contributions in a runtime loop over
// k with eight independent sums, then the block's own triangle in
// registers. Each x_j receives the same operations in the same order as the
// plain dot form (k ascending, then the scaling), so the result is the
// same, while the code stays a few hundred bytes (a fully unrolled solve is
// fetched from L2 once per piece and runs at instruction-fetch speed).
template <typename T, int XS, int MK, int MJ, bool UNIT>
__device__ inline void blk_trsv(T* X, const T* M, const T* rd, int nq) {
  for (int jb = 0; jb < nq; jb += 8) {
    int jc[8];  // columns of the block, clamped inside the piece
#pragma unroll
    for (int c = 0; c < 8; ++c) jc[c] = min(jb + c, nq - 1);
    T xb[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) xb[c] = X[jc[c] * XS];
#pragma unroll 2
    for (int kk = 0; kk < jb; ++kk) {
      const T xk = X[kk * XS];
#pragma unroll
      for (int c = 0; c < 8; ++c) xb[c] -= xk * M[kk * MK + jc[c] * MJ];
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
#pragma unroll
      for (int cp = 0; cp < c; ++cp) xb[c] -= xb[cp] * M[jc[cp] * MK + jc[c] * MJ];
      if (!UNIT) xb[c] = xb[c] * (rd ? rd[jc[c]] : T(1) / M[jc[c] * MK + jc[c] * MJ]);
    }
#pragma unroll
    for (int c = 0; c < 8; ++c)
      if (jb + c < nq) X[(jb + c) * XS] = xb[c];
  }
}

// Pivot of column k among the rows whose position is k or later (v: this
// lane's entry of the column, pos: its row's position): largest |v|, ties
// to the smallest position; a column without a comparable candidate (NaN)
// keeps the row at position k. Returns the lane of the pivot row.
template <typename T>
__device__ inline int pivot_lane(T v, int pos, bool mine, int k) {
  const bool cand = mine && pos >= k;
  const T a = cand ? fabs(v) : T(-1);
  const T m = wave_max(a);
  const bool tie = cand && a == m;
  const unsigned long long msk = __ballot(tie);
  int blane;
  if (msk == 0ull) {
    blane = __ffsll((long long)__ballot(mine && pos == k)) - 1;
  } else if (__popcll(msk) == 1) {
    blane = __ffsll((long long)msk) - 1;
  } else {
    const int mp = wave_min(tie ? pos : (1 << 20));
    blane = __ffsll((long long)__ballot(tie && pos == mp)) - 1;
  }
  return __builtin_amdgcn_readfirstlane(blane);
}

// Pivoted LU of the nq x nq block D (LDS, leading dimension LD, nq <= 64)
// with rows that never move during the elimination: lane i owns LDS row i of
// the block and tracks the position pos its row holds after the interchanges
// so far. Step k takes the row of smallest position among those holding the
// maximum |a| over positions >= k (the first maximum of ggetrf!,
// GenericBlasLapackFragments.jl:56-100; a zero maximum keeps row k and skips
// the scaling) and reads the pivot row where it lies. At the end every row
// moves to its position, together with the columns [nq, ncols) of D. piv[k]
// is the position swapped with k at step k, perm[p] the row now at position
// p, dinv[k] = 1 / U(k, k); *zero is set by a zero pivot. The whole
// workgroup, one barrier per step. Wave 0 updates
// the next pivot column first and runs the next step's pivot search on it
// (pivot_lane), publishing the pivot row and value through LDS (two slots,
// by step parity); waves 1-3 update the columns j = k + 2 + (wave - 1) + 3 i
// meanwhile. The multipliers of column k are written by wave 0 one step
// later, when no wave reads that column any more. Must be called by all
// threads of the workgroup.
template <typename T, int LD>
__device__ void wg_getrf(T* D, int nq, int ncols, int* piv, int* perm, T* dinv, int* zero) {
  __shared__ int s_blane[2];
  __shared__ T s_pv[2];
  const int lane = threadIdx.x % 64, wave = wave_id();
  const bool mine = lane < nq;
  int pos = lane;
  T lprev = T(0);
  bool wprev = false;
  if (wave == 0) {
    const T v = mine ? D[lane] : T(0);
    const int b = pivot_lane(v, pos, mine, 0);
    const T pv = rdlane(v, b);
    if (lane == 0) {
      s_blane[0] = b;
      s_pv[0] = pv;
    }
  }
  __syncthreads();
  for (int k = 0; k < nq; ++k) {
    const int par = k & 1;
    const int blane = s_blane[par];
    const T pv = s_pv[par];
    const T v = mine ? D[lane + k * LD] : T(0);
    if (wave == 0 && wprev) D[lane + (k - 1) * LD] = lprev;
    // the pivot row's position before this step's interchange
    const int kp = __builtin_amdgcn_readlane(pos, blane);
    const bool nonzero = pv != T(0);
    if (nonzero && kp != k) {
      if (mine && pos == k)
        pos = kp;
      else if (lane == blane)
        pos = k;
    }
    const T inv = T(1) / pv;
    if (threadIdx.x == 0) {
      piv[k] = kp;
      dinv[k] = inv;
      if (!nonzero) *zero = 1;
    }
    const bool below = mine && pos > k;
    const T l = nonzero ? v * inv : v;
    lprev = l;
    wprev = below && nonzero;
    if (wave == 0) {
      if (k + 1 < nq) {
        const int j = k + 1;
        const T u = D[blane + j * LD];
        T x = D[lane + j * LD];
        if (below) {
          x -= l * u;
          D[lane + j * LD] = x;
        }
        const int b = pivot_lane(x, pos, mine, j);
        const T pn = rdlane(x, b);
        if (lane == 0) {
          s_blane[par ^ 1] = b;
          s_pv[par ^ 1] = pn;
        }
      }
    } else {
      // columns j = k + 2 + (wave - 1) + 3 i in batches of eight: loads of a
      // batch are issued together (indices clamped inside the block), stores
      // guarded
      for (int jb = k + 1 + wave; jb < nq; jb += 24) {
        T u[8], x[8];
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
          const int j = min(jb + 3 * jj, nq - 1);
          u[jj] = D[blane + j * LD];
          x[jj] = D[lane + j * LD];
        }
        if (below) {
#pragma unroll
          for (int jj = 0; jj < 8; ++jj)
            if (jb + 3 * jj < nq) D[lane + (jb + 3 * jj) * LD] = x[jj] - l * u[jj];
        }
      }
    }
    __syncthreads();
  }
  if (wave == 0 && wprev) D[lane + (nq - 1) * LD] = lprev;
  if (wave == 0 && mine) perm[pos] = lane;
  __syncthreads();
  // rows to their positions (position p takes LDS row perm[p]), the waves
  // taking interleaved columns; all reads of a batch precede its writes
  const T* srow = D + (mine ? perm[lane] : 0);
  T* drow = D + lane;
  for (int c0 = 0; c0 < ncols; c0 += 32) {
    T x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = c0 + wave + 4 * u;
      x[u] = (c < ncols) ? srow[c * LD] : T(0);
    }
    __syncthreads();
    if (mine) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int c = c0 + wave + 4 * u;
        if (c < ncols) drow[c * LD] = x[u];
      }
    }
    __syncthreads();
  }
}

// The same factorisation without pivoting for SPD pieces of up to kMaxNq
// columns (lane = row, rows lane and lane + 64): a zero pivot sets *zero and
// skips the scaling; piv[k] = k.
template <typename T, int LD>
__device__ void nopiv_getrf(T* D, int nq, int* piv, T* dinv, int* zero) {
  const int lane = threadIdx.x % 64;
  for (int k = 0; k < nq; ++k) {
    const T pv = D[k + k * LD];
    const bool nonzero = pv != T(0);
    const T inv = T(1) / pv;
    if (lane == 0) {
      piv[k] = k;
      dinv[k] = inv;
      if (!nonzero) *zero = 1;
    }
    for (int i = k + 1 + lane; i < nq; i += 64) {
      T l = D[i + k * LD];
      if (nonzero) {
        l *= inv;
        D[i + k * LD] = l;
      }
      for (int j0 = k + 1; j0 < nq; j0 += 8) {
        T u[8], x[8];
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
          const int j = min(j0 + jj, nq - 1);
          u[jj] = D[k + j * LD];
          x[jj] = D[i + j * LD];
        }
#pragma unroll
        for (int jj = 0; jj < 8; ++jj)
          if (j0 + jj < nq) D[i + (j0 + jj) * LD] = x[jj] - l * u[jj];
      }
    }
    wave_lds_sync();
  }
}

// v_mfma_*_16x16x4: both forms take A(i, k) and B(k, j) from lane i + 16 k
// (j + 16 k); accumulator element v of lane l is D(i, l % 16) with i = 4
// (l / 16) + v for the f32 form and i = 4 v + l / 16 for the f64 form.
template <typename T>
struct Mfma16;
template <>
struct Mfma16<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ inline v4 op(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ inline int row(int lgrp, int v) { return 4 * v + lgrp; }
};
template <>
struct Mfma16<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ inline v4 op(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ inline int row(int lgrp, int v) { return 4 * lgrp + v; }
};

// Diagonal region of one block per workgroup (see the section comment);
// NQ bounds the piece width. Dynamic LDS: 128 * kRLD elements.
template <typename T, int NQ>
__global__ void __launch_bounds__(kWG)
blk_diag_kernel(DevSym s, const BlkDesc* __restrict__ desc, T* __restrict__ arena,
                int64_t* __restrict__ ipvt, int32_t* __restrict__ rperm,
                unsigned long long* __restrict__ first_fail) {
  const int64_t vs = blockIdx.y;  // value set
  arena += vs * s.vs_arena;
  ipvt += vs * s.n;
  rperm += vs * s.n;
  constexpr int LD = kRLD;
  extern __shared__ unsigned char smem_raw[];
  __shared__ int piv[NQ];
  __shared__ int perm[NQ];
  __shared__ T dinv[NQ];
  __shared__ int s_zero;
  // the row each position takes, and the position each row takes
  __shared__ unsigned char ssrc[128], spos[128];
  T* R = reinterpret_cast<T*>(smem_raw);
  const int tid = threadIdx.x, wave = wave_id();
  const BlkDesc d = desc[blockIdx.x];
  const int f = d.front;
  const int L = s.fL[f];
  const int64_t fc0 = s.fc0[f];
  const int c0 = d.c0, bw = d.c1 - d.c0;
  T* Fr = arena + s.foff[f] + c0 + (int64_t)c0 * L;
  load_tile<T, 1, LD>(Fr, L, bw, bw, R);
  __syncthreads();
  for (int pi = 0; pi < d.np; ++pi) {
    int64_t pc0, nq64;
    piece_cols(s, d.piece + pi, pc0, nq64);
    const int nq = (int)nq64;
    const int o = (int)(pc0 - fc0) - c0;  // piece offset inside the region
    const int rest = bw - o - nq;         // region rows below / columns right
    T* D = R + o + o * LD;
    if (tid == 0) s_zero = 0;
    __syncthreads();
    // interchanges reach the region columns right of the piece too
    if (s.pivot && nq <= 64) {
      wg_getrf<T, LD>(D, nq, nq + rest, piv, perm, dinv, &s_zero);
    } else if (wave == 0) {
      nopiv_getrf<T, LD>(D, nq, piv, dinv, &s_zero);
    }
    __syncthreads();
    if (tid < nq) {
      ipvt[pc0 + tid] = piv[tid] + 1;
      const int src = (s.pivot && nq <= 64) ? perm[tid] : tid;
      ssrc[o + tid] = (unsigned char)(o + src);
      spos[o + src] = (unsigned char)(o + tid);
    }
    if (tid == 0 && s_zero) atomicMin(first_fail, (unsigned long long)(d.piece + pi + 1));
    if (tid >= 128) {
      // U12 of the region (rows already interchanged): unit-lower solve,
      // u_i = a_i - sum_k<i L(i, k) u_k, one column per thread
      for (int c = tid - 128; c < rest; c += 128)
        blk_trsv<T, 1, LD, 1, true>(D + (nq + c) * LD, D, nullptr, nq);
    } else {
      // L21 of the region: x_j = (a_j - sum_k<j x_k U(k, j)) / U(j, j), one
      // row per thread
      for (int r = tid; r < rest; r += 128)
        blk_trsv<T, LD, 1, LD, false>(D + nq + r, D, dinv, nq);
    }
    __syncthreads();
    if (rest > 0) {
      // rest x rest update on the matrix cores: 16 x 16 tiles, every fourth
      // to a wave; per tile all operand reads are issued before the MFMAs
      // (k in steps of four, cut at nq); products summed from zero and
      // subtracted once, as in blk_gemm_kernel
      typedef typename Mfma16<T>::v4 v4;
      constexpr int KS = (NQ + 3) / 4;
      const int lane = tid % 64, l16 = lane % 16, lk = lane / 16;
      const int nt = (rest + 15) / 16;
      const T* Lb = D + nq;       // L21(i, k) = Lb[i + k LD]
      const T* Ub = D + nq * LD;  // U12(k, j) = Ub[k + j LD]
      T* C = D + nq + nq * LD;
      for (int t = wave; t < nt * nt; t += 4) {
        const int tr = (t % nt) * 16, tc = (t / nt) * 16;
        const int ri = tr + l16, cj = tc + l16;
        const bool rin = ri < rest, cin = cj < rest;
        T av[KS], bv[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int kk = 4 * ks + lk;
          const bool kin = kk < nq;
          av[ks] = (kin && cin) ? Ub[kk + cj * LD] : T(0);
          bv[ks] = (kin && rin) ? Lb[ri + kk * LD] : T(0);
        }
        v4 acc = v4{T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          if (4 * ks < nq) acc = Mfma16<T>::op(av[ks], bv[ks], acc);
        if (rin) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int j = tc + Mfma16<T>::row(lk, v);
            if (j < rest) C[ri + j * LD] -= acc[v];
          }
        }
      }
    }
    __syncthreads();
  }
  if (tid < bw) rperm[fc0 + c0 + tid] = ssrc[tid] | spos[tid] << 8;
  store_tile<T, 1, LD>(Fr, L, bw, bw, R);
}

// v, computed where it stands for every lane (keeps the compiler from
// turning a select of it into a branch around its computation).
__device__ inline double pin(double v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ inline float pin(float v) {
  asm volatile("" : "+v"(v));
  return v;
}

// 1 / v in every lane and the maximum of key over the 64 lanes (all lanes
// active): the two dependent chains, a division (about eleven operations)
// and four DPP maxima, are independent of each other, so each operation of
// one fills the other's latency; the scheduling barriers keep the compiler
// from placing one chain after the other (both one after the other: 250
// cycles). The division is the one that V_DIV_SCALE, V_DIV_FMAS and V_DIV_FIXUP are
// documented for in AMD's CDNA instruction set manuals: Newton steps on the
// reciprocal of the scaled operand, the quotient, one residual correction.
#define SPK_SB __builtin_amdgcn_sched_barrier(0)
template <int CTRL>
__device__ inline unsigned dpp_umax(unsigned v) {
  return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false));
}
__device__ inline unsigned row_umax(unsigned v) {  // v: the rows' own maxima
  const unsigned a = (unsigned)__builtin_amdgcn_readlane((int)v, 0);
  const unsigned b = (unsigned)__builtin_amdgcn_readlane((int)v, 16);
  const unsigned c = (unsigned)__builtin_amdgcn_readlane((int)v, 32);
  const unsigned d = (unsigned)__builtin_amdgcn_readlane((int)v, 48);
  return max(max(a, b), max(c, d));
}
__device__ inline double recip_and_max(double v, unsigned key, unsigned& mx) {
  bool f0, f1;
  const double d0 = __builtin_amdgcn_div_scale(1.0, v, false, &f0);
  unsigned m = dpp_umax<0xB1>(key);  // lanes ^1
  SPK_SB;
  const double r0 = __builtin_amdgcn_rcp(d0);
  const double n0 = __builtin_amdgcn_div_scale(1.0, v, true, &f1);
  SPK_SB;
  m = dpp_umax<0x4E>(m);  // lanes ^2
  SPK_SB;
  const double e0 = __builtin_fma(-d0, r0, 1.0);
  SPK_SB;
  m = dpp_umax<0x141>(m);  // mirror inside 8
  SPK_SB;
  const double r1 = __builtin_fma(r0, e0, r0);
  SPK_SB;
  m = dpp_umax<0x140>(m);  // mirror inside 16
  SPK_SB;
  const double e1 = __builtin_fma(-d0, r1, 1.0);
  SPK_SB;
  mx = row_umax(m);
  const double r2 = __builtin_fma(r1, e1, r1);
  const double q = n0 * r2;
  const double e2 = __builtin_fma(-d0, q, n0);
  return __builtin_amdgcn_div_fixup(__builtin_amdgcn_div_fmas(e2, r2, q, f1), v, 1.0);
}
__device__ inline float recip_and_max(float v, unsigned key, unsigned& mx) {
  bool f0, f1;
  const float d0 = __builtin_amdgcn_div_scalef(1.0f, v, false, &f0);
  unsigned m = dpp_umax<0xB1>(key);
  SPK_SB;
  const float r0 = __builtin_amdgcn_rcpf(d0);
  const float n0 = __builtin_amdgcn_div_scalef(1.0f, v, true, &f1);
  SPK_SB;
  m = dpp_umax<0x4E>(m);
  SPK_SB;
  const float e0 = __builtin_fmaf(-d0, r0, 1.0f);
  SPK_SB;
  m = dpp_umax<0x141>(m);
  SPK_SB;
  const float r1 = __builtin_fmaf(e0, r0, r0);
  SPK_SB;
  m = dpp_umax<0x140>(m);
  SPK_SB;
  const float q0 = n0 * r1;
  SPK_SB;
  mx = row_umax(m);
  const float e1 = __builtin_fmaf(-d0, q0, n0);
  const float q1 = __builtin_fmaf(e1, r1, q0);
  const float e2 = __builtin_fmaf(-d0, q1, n0);
  return __builtin_amdgcn_div_fixupf(__builtin_amdgcn_div_fmasf(e2, r1, q1, f1), v, 1.0f);
}

// The leading 32 bits of |v|, plus one, for a candidate that is a number;
// 0 otherwise. For floats all of |v|: the order of the keys is the order of
// the magnitudes, up to ties in the low half of a double.
__device__ inline unsigned pivot_key(double v, bool cand) {
  const unsigned hi = (unsigned)((unsigned long long)__double_as_longlong(v) >> 32) & 0x7fffffffu;
  return cand && v == v ? hi + 1u : 0u;
}
__device__ inline unsigned pivot_key(float v, bool cand) {
  return cand && v == v ? (__float_as_uint(v) & 0x7fffffffu) + 1u : 0u;
}

// ---------------------------------------------------------------------------
// Small fronts, whole, each by a group of G threads: a workgroup (G = 256)
// or one wave (G = 64).
// ---------------------------------------------------------------------------

// f(0), f(1), ... f(N - 1), each with its index a constant.
template <int N, int I = 0, typename F>
__device__ __attribute__((always_inline)) inline void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

// Static LDS of one workgroup: what one group of 256 threads or four waves
// of 64 need. Columns and rows are published in two slots by step parity.
template <typename T, int RMAX = 64>
struct SmallScratch {
  T col[2][RMAX];      // the step's pivot column
  T row[2][RMAX];      // the row at the step's position
  T prow[RMAX];        // the pivot row, where it is another one
  int64_t lc[RMAX], uc[RMAX];  // lnz and unz bases of the own columns / rows
  int cq[RMAX], ce[RMAX];      // column range of the own column's piece
  int piv[RMAX];
};

// One front: A's entries (aent; without them the panels of assembled
// lnz/unz) and the children's update matrices are summed in LDS (F, rows of
// odd stride LD, no bank conflicts along either direction), moved to
// registers, eliminated piece by piece exactly as the reference does
// (SpkLUFactor.jl:178-302: row interchanges inside the piece's diagonal
// block, applied to the piece's own columns and those right of it; rows
// below the block scaled always, rows inside it for a nonzero pivot), and
// written to lnz/unz/ipvt and the arena through LDS.
//
// The elimination is a chain of W column steps, so a step's latency is what
// bounds it: thread (ty, tx) of an NB x NB grid keeps the entries (ty + NB i,
// tx + NB j) in registers, and a step costs one publication of its column
// and of the row at its position, one pivot search that every wave makes
// alike (32-bit keys, with every lane's reciprocal computed meanwhile) and
// M x M updates per thread; only an interchange takes a second barrier
// (about 0.5 us a column of a 64-row front). With the front kept in LDS, the
// pivot searched by one thread and four barriers and an integer division per
// entry in each step, the small fronts of one pass took, before -> now:
// 193 x 171 grid 824 -> 450 us, 128 small SPD systems 1500 -> 895 us, 32
// value sets of 32^3 (float) 2310 -> 993 us. One wave per front of at most 32
// rows needs no barrier; its grid follows the front (8, 16 or 32 rows): with
// one grid of 64 rows for every front of a level above the small_wave_min
// knob the 128 systems took 1709 us, so that form is left to levels that
// have larger fronts.
template <typename T, int G, int M, typename Scratch>
__device__ __attribute__((always_inline)) void small_front_body(
    const DevSym& s, const SmallDesc& d, const SmallChild* __restrict__ child, T* F, int LD,
    Scratch& sh, const AEnt* __restrict__ aent, const double* __restrict__ nzval, T* __restrict__ lnz, T* __restrict__ unz,
    int64_t* __restrict__ ipvt, T* __restrict__ arena,
    unsigned long long* __restrict__ first_fail) {
  constexpr int NB = G == kWG ? 16 : 8;
  constexpr int RMAX = M * NB;  // rows a group can hold
  constexpr int RL = RMAX < 64 ? RMAX : 64;  // lanes along a column
  constexpr int NC = G / RL;    // columns a group takes at once
  const int gt = G == kWG ? (int)threadIdx.x : (int)threadIdx.x % 64;
  const int lane = (int)threadIdx.x % 64;
  const int cr = gt % RL, cc0 = gt / RL;  // (row, column) of the column-wise phases
  auto gsync = [] {
    if constexpr (G == kWG)
      __syncthreads();
    else
      wave_lds_sync();
  };
  const int L = d.L, W = d.W, R = L - W;
  const int64_t fc0 = d.fc0;
  // the first entries are read while F is cleared
  AEnt en{};
  double nv = 0.0;
  if (aent && gt < d.an) {
    en = aent[d.a0 + gt];
    nv = nzval[en.k];
  }
  if (gt < W) {
    const int64_t g = fc0 + gt;
    const int pc = s.pcol[g];
    sh.lc[gt] = s.lcol[g];
    sh.uc[gt] = s.ucol[g];
    sh.cq[gt] = pc & 0xffff;
    sh.ce[gt] = pc >> 16;
  }
  for (int i = gt; i < L * LD; i += G) F[i] = T(0);
  gsync();
  if (aent) {
    if (gt < d.an) F[en.r + en.c * LD] = (T)nv;
    for (int e = gt + G; e < d.an; e += G) {
      const AEnt x = aent[d.a0 + e];
      F[x.r + x.c * LD] = (T)nzval[x.k];
    }
  } else {
    for (int j = cc0; j < W; j += NC)
      if (cr < L) {
        if (cr >= (s.sym ? j : sh.cq[j])) F[cr + j * LD] = lnz[sh.lc[j] + cr];
        if (!s.sym && cr >= sh.ce[j]) F[j + cr * LD] = unz[sh.uc[j] + cr];
      }
    if (s.sym) {  // upper rows of the own columns from the lower triangle
      gsync();
      for (int j = cc0; j < W; j += NC)
        if (cr > j && cr < L) F[j + cr * LD] = F[cr + j * LD];
    }
  }
  gsync();
  // children's update matrices, one child at a time in a fixed order (rows
  // of different children may coincide)
  for (int ci = 0; ci < d.nch; ++ci) {
    const SmallChild ch = child[d.ch0 + ci];
    const int32_t* rel = s.relmap + ch.rel;
    const T* cb = arena + ch.cb;
    const bool in = cr < ch.R;
    const int rr = in ? rel[cr] : 0;
    for (int t0 = cc0; t0 < ch.R; t0 += 8 * NC) {
      T v[8];
      int rt[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int t = t0 + u * NC;
        v[u] = (in && t < ch.R) ? cb[cr + (int64_t)t * ch.ld] : T(0);
        rt[u] = t < ch.R ? rel[t] : 0;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (in && t0 + u * NC < ch.R) F[rr + rt[u] * LD] += v[u];
    }
    gsync();
  }
  const int ty = gt % NB, tx = gt / NB;
  T a[M][M];
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const int r = ty + NB * i, c = tx + NB * j;
      a[i][j] = (r < L && c < L) ? F[r + c * LD] : T(0);
    }
  const int srow = lane % RMAX;  // the row this lane looks at in a pivot search
  static_for<M>([&](auto jbc) __attribute__((always_inline)) {
    constexpr int jb = decltype(jbc)::value;
#pragma unroll 1
    for (int cc = 0; cc < NB && jb * NB + cc < W; ++cc) {
      const int k = jb * NB + cc, par = cc & 1;
      const int cq = sh.cq[k], ce = sh.ce[k];
      T* col = sh.col[par];
      T* row = sh.row[par];
      if (tx == cc) {
#pragma unroll
        for (int i = 0; i < M; ++i) col[ty + NB * i] = a[i][jb];
      }
      if (ty == cc) {
#pragma unroll
        for (int j = 0; j < M; ++j) row[tx + NB * j] = a[jb][j];
      }
      gsync();
      const T v = col[srow];
      T l[M], u[M];
#pragma unroll
      for (int i = jb; i < M; ++i) l[i] = col[ty + NB * i];
#pragma unroll
      for (int j = jb; j < M; ++j) u[j] = row[tx + NB * j];
      const bool cand = lane < RMAX && lane >= k && lane < ce;
      const unsigned key = pivot_key(v, cand);
      unsigned mx;
      const T rc = recip_and_max(v, key, mx);
      int kp = k;
      if (s.pivot) {
        const unsigned long long msk = __ballot(key == mx);
        kp = __builtin_amdgcn_readfirstlane(__ffsll((long long)msk) - 1);
        // ties of the leading bits, no number among the candidates, or none
        // in the first row (which then stays): the exact rule
        if (__builtin_expect(mx == 0u || (msk & (msk - 1ull)) != 0ull ||
                                 __builtin_amdgcn_readlane((int)key, k) == 0, 0)) {
          const bool keep = __builtin_amdgcn_readlane((int)key, k) == 0;
          kp = keep ? k : pivot_lane(v, lane, cand, k);
        }
      }
      const T pv = rdlane(v, kp), inv = rdlane(rc, kp);
      const bool nz = pv != T(0);
      if (gt == 0) {
        sh.piv[k] = kp - cq + 1;
        if (!nz) atomicMin(first_fail, (unsigned long long)s.snode[fc0 + k]);
      }
      if (kp != k && nz) {
        T* prow = sh.prow;
#pragma unroll
        for (int i = jb; i < M; ++i)
          if (ty + NB * i == kp) {
#pragma unroll
            for (int j = 0; j < M; ++j) prow[tx + NB * j] = a[i][j];
          }
        gsync();
#pragma unroll
        for (int j = 0; j < M; ++j) {
          const int c = tx + NB * j;
          const T x = row[c], y = prow[c];
#pragma unroll
          for (int i = jb; i < M; ++i)
            if (ty + NB * i == kp && c >= cq) a[i][j] = x;
          if (ty == cc && c >= cq) a[jb][j] = y;
          if (j >= jb) u[j] = y;
        }
        const T ck = col[k];
#pragma unroll
        for (int i = jb; i < M; ++i)
          if (ty + NB * i == kp) l[i] = ck;
      }
#pragma unroll
      for (int i = jb; i < M; ++i) {
        const int r = ty + NB * i;
        l[i] = (nz || r >= ce) ? l[i] * inv : l[i];
        const bool below = i > jb || r > k;
        if (tx == cc && below) a[i][jb] = l[i];
#pragma unroll
        for (int j = jb; j < M; ++j) {
          const T w = a[i][j] - l[i] * u[j];
          a[i][j] = (below && (j > jb || tx > cc)) ? w : a[i][j];
        }
      }
    }
  });
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const int r = ty + NB * i, c = tx + NB * j;
      if (r < L && c < L) F[r + c * LD] = a[i][j];
    }
  gsync();
  if (gt < W) ipvt[fc0 + gt] = sh.piv[gt];
  for (int j = cc0; j < W; j += NC)
    if (cr < L) {
      if (cr >= sh.cq[j]) lnz[sh.lc[j] + cr] = F[cr + j * LD];
      if (cr >= sh.ce[j]) unz[sh.uc[j] + cr] = F[j + cr * LD];
    }
  T* cb = arena + d.cb;
  if (cr < R)
    for (int t = cc0; t < R; t += NC) cb[cr + t * R] = F[(W + cr) + (W + t) * LD];
}

// The level's fronts of more than 32 rows (the first nbig of desc) one per
// workgroup, the others one per wave, four per workgroup; WAVE64: every
// front one per wave (levels of very many fronts). The grid of a wave's
// threads follows the front's rows. The workgroups behind the first wgs
// assemble the level's large fronts, which the small ones do not touch.
template <typename T, bool WAVE64>
__global__ void __launch_bounds__(kWG)
small_front_kernel(DevSym s, const SmallDesc* __restrict__ desc,
                   const SmallChild* __restrict__ child, int nbig, int cnt, int LD, int slot,
                   int wgs, AsmArgs asmb, const AEnt* __restrict__ aent,
                   const double* __restrict__ nzval, int64_t nnz, T* __restrict__ lnz, T* __restrict__ unz,
                   int64_t* __restrict__ ipvt, T* __restrict__ arena,
                   unsigned long long* __restrict__ first_fail) {
  const int64_t vs = blockIdx.y;  // value set
  nzval += vs * nnz;
  lnz += vs * s.vs_lnz;
  unz += vs * s.vs_unz;
  ipvt += vs * s.n;
  arena += vs * s.vs_arena;
  extern __shared__ unsigned char smem_raw[];
  if ((int)blockIdx.x >= wgs) {
    large_assemble_body<T, 64>(s, asmb, (int)blockIdx.x - wgs, nzval, arena, smem_raw);
    return;
  }
  T* F = reinterpret_cast<T*>(smem_raw);
  const int wave = wave_id();
  if constexpr (WAVE64) {
    __shared__ SmallScratch<T> sh[4];
    const int item = blockIdx.x * 4 + wave;
    if (item >= cnt) return;
    const SmallDesc d = desc[item];
    F += wave * slot;
    auto go = [&](auto m) __attribute__((always_inline)) {
      small_front_body<T, 64, decltype(m)::value>(s, d, child, F, LD, sh[wave], aent, nzval, lnz,
                                                  unz, ipvt, arena, first_fail);
    };
    if (d.L <= 16)
      go(std::integral_constant<int, 2>{});
    else if (d.L <= 32)
      go(std::integral_constant<int, 4>{});
    else
      go(std::integral_constant<int, 8>{});
  } else {
    __shared__ union U {
      SmallScratch<T> big;
      SmallScratch<T, 32> one[4];
      __device__ U() {}
    } sh;
    if ((int)blockIdx.x < nbig) {
      small_front_body<T, kWG, 4>(s, desc[blockIdx.x], child, F, LD, sh.big, aent, nzval, lnz, unz,
                                  ipvt, arena, first_fail);
      return;
    }
    const int item = nbig + ((int)blockIdx.x - nbig) * 4 + wave;
    if (item >= cnt) return;
    const SmallDesc d = desc[item];
    F += wave * slot;
    auto go = [&](auto m) __attribute__((always_inline)) {
      small_front_body<T, 64, decltype(m)::value>(s, d, child, F, min(LD, 33), sh.one[wave], aent,
                                                  nzval, lnz, unz, ipvt, arena, first_fail);
    };
    if (d.L <= 8)
      go(std::integral_constant<int, 1>{});
    else if (d.L <= 16)
      go(std::integral_constant<int, 2>{});
    else
      go(std::integral_constant<int, 4>{});
  }
}

// Diagonal region of one block of at most 64 columns per workgroup, held
// in registers in panels of eight columns: wave w keeps panels w and w + 4,
// one row per lane. The region is factored right-looking, one column at a time,
// with the reference's pivoting confined to each piece's rows (LU; an SPD
// front takes the row at position k, no interchanges)
// (SpkLUFactor.jl:230-240, GenericBlasLapackFragments.jl:56-100). Step k,
// a column of piece p, takes as pivot the row of p with the largest |a|
// among those whose position is k or later (ties: the smallest position; no
// comparable candidate: the row at position k), scales the rows below it by
// the reciprocal of the pivot (not when it is zero) and subtracts their
// multiple of the pivot row from the columns right of k. The rows below are
// p's rows at later positions and every row of the later pieces: for p's
// rows this is the piece's pivoted LU and, right of the piece, its
// unit-lower solve U12 = L11^-1 P A12; for the later pieces' rows it is
// L21 = A21 U11^-1 and the update of their part of the region. The
// triangular parts receive their terms one at a time in ascending k, in the
// order of the left-looking forms; the later pieces' part right of the
// piece sums the piece's products from zero and subtracts the sum once,
// as the reference's update of one supernode by another does (the sum is
// kept in the entry itself, the entry's value aside until the piece's last
// column). Rows never move while factoring: each lane tracks the position
// its row holds (positions of a piece stay inside the piece, so the rows
// below step k are those of a position past k, at any later time too). The
// wave owning column k updates the rest of its panel only, publishes the
// step (multipliers, pivot lane, pivot position) through LDS and goes on;
// the waves apply published steps to their other panels as they come,
// without barriers (a wave only ever waits for steps of columns left of its
// own, which are published without waiting on it). At the end each row is
// stored at its final position in the columns of its piece and right of it,
// and at its own row in the columns of earlier pieces, which the reference
// never interchanges.
// When d.fk1 > d.fk0 the region first takes the product of the previous
// block (columns [fk0, fk1)) with its own columns, summed from zero over
// those columns and subtracted once (the trailing update's form), so that
// the rest of that block's update can run beside this kernel; the product is
// formed by MFMA from LDS in steps of 32 columns.
// What bounds it: the chain pivot search -> reciprocal -> next column, once
// per column, on one wave (latency and issue: a readlane pair with its FMA
// costs 26 cycles, a DPP maximum 12, a taken branch 30). So the chain's wave
// touches eight columns only (alternating panels: sixteen columns in one
// wave cost 1 500 cycles per column), the search compares the leading 32
// bits of the magnitudes (only when they tie does the full search decide),
// and every lane forms its own entry's reciprocal beside the search. One
// 60-column block alone, two pieces: 42.8 -> 32.1 us in double and 38.3 ->
// 29.6 us in float, with a folded block 47.2 -> 36.1 and 41.6 -> 32.5 us
// (of these 4 us are the folded product, 2.6 us the launch). The LDS, 97 KB
// before, is 36 KB in double: other kernels' workgroups leave room for it
// (diagonal regions waited for the second stream's updates to drain: 175 us
// on average per launch in double at 64^3).
// lds: slab_elems(bw, first piece's width, folded) elements: the finished
// columns (bw x bw), the entries set aside (those of the later pieces), or
// the folded panels.
constexpr int kMaxBlkPieces = 8;  // most pieces in one block
constexpr int kFoldK = 32;        // folded columns per step
constexpr int kFoldMax = 2 * kFoldK;  // most folded columns (the plan merges no more)
__host__ __device__ constexpr int slab_elems(int bw, int w0, bool fold) {
  const int own = bw * bw + (bw - w0) * (bw - w0);
  return fold && own < 2 * kFoldK * 64 ? 2 * kFoldK * 64 : own;
}
template <typename T>
__device__ __attribute__((always_inline)) void blk_diag_slab_body(
    const DevSym& s, const BlkDesc& d, T* __restrict__ arena, int64_t* __restrict__ ipvt,
    int32_t* __restrict__ rperm, unsigned long long* __restrict__ first_fail,
    unsigned char* lds) {
  constexpr int PW = 8;                   // columns per panel
  // step k, once published (before: -1): pivot lane | position << 8 |
  // nonzero << 16
  __shared__ int smeta[64];
  __shared__ int spo[kMaxBlkPieces + 1];  // piece offsets in the region; spo[np] = bw
  __shared__ unsigned char scp[64];       // piece of each region column
  __shared__ unsigned char spos[64];      // final position of each row
  __shared__ unsigned char ssrc[64];      // the row each position takes
  const int lane = threadIdx.x % 64, w = wave_id();
  const int L = d.L;
  const int64_t fc0 = d.fc0;
  const int c0 = d.c0, bw = d.c1 - d.c0, np = d.np;
  const T* const Fb = arena + d.foff;
  T* R = arena + d.foff + c0 + (int64_t)c0 * L;
  // finished column k, rows in lane order, at sl[k bw + row]: multipliers of
  // the rows below the pivot, the others' values; and the entries set aside,
  // (row, column) from (n0, n0), n0 the first piece's width
  const int n0 = d.pw[0], nv = bw - n0;
  T* sl = reinterpret_cast<T*>(lds);
  T* ssv = sl + bw * bw;
  // this wave's panels: columns ca + i and cb + i. The front and the piece
  // widths come from the descriptor, so the region, the previous block's
  // panels and the widths are read in one batch
  const int ca = PW * w, cb = PW * w + 32;
  T a[PW], b[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    a[i] = (lane < bw && ca + i < bw) ? R[lane + (int64_t)(ca + i) * L] : T(0);
    b[i] = (lane < bw && cb + i < bw) ? R[lane + (int64_t)(cb + i) * L] : T(0);
  }
  const int fkw = d.fk1 - d.fk0;
  // L(c0 + r, fk0 + k) at Lp[64 k + (r ^ 16 (k % 4))], U(fk0 + k, c0 + c) at
  // Up[32 c + (k ^ usw(c))]: stores and operand reads without bank conflicts
  T* Lp = sl;
  T* Up = sl + kFoldK * 64;
  const int fk = lane % kFoldK, fc = 2 * w + lane / kFoldK;
  auto usw = [](int c) {
    return std::is_same<T, double>::value ? 2 * (c & 15) : 4 * ((c >> 1) & 7);
  };
  // both steps' panels (kFoldMax columns at most) from clamped addresses, in
  // flight with the region; what lies outside is zeroed below
  T pl[2][8], pu[2][8];
  if (fkw > 0) {
    const T* lrow = Fb + c0 + min(lane, bw - 1) + (int64_t)d.fk0 * L;
    const T* ucol = Fb + d.fk0 + (int64_t)c0 * L;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int k = kFoldK * h + w + 4 * u, c = fc + 8 * u;
        pl[h][u] = lrow[(int64_t)min(k, fkw - 1) * L];
        pu[h][u] = ucol[min(kFoldK * h + fk, fkw - 1) + (int64_t)min(c, bw - 1) * L];
      }
  }
  if ((int)threadIdx.x <= np) {
    int o = 0;  // spo[np] = bw: the pieces fill the block
    for (int q = 0; q < (int)threadIdx.x; ++q) o += d.pw[q];
    spo[threadIdx.x] = o;
  }
  if (threadIdx.x < 64) smeta[threadIdx.x] = -1;
  __syncthreads();
  if (threadIdx.x < 64) {
    int p = 0;
    while (p + 1 < np && (int)threadIdx.x >= spo[p + 1]) ++p;
    scp[threadIdx.x] = (unsigned char)p;
  }
  if (fkw > 0) {
    typedef typename Mfma16<T>::v4 v4;
    const int l16 = lane % 16, lk = lane / 16;
    // operand column l16 of the wave's sixteen: panel w, then panel w + 4
    const int mc = std::is_same<T, double>::value ? 4 * (l16 % 4) + l16 / 4 : l16;
    const int mcol = mc < PW ? ca + mc : cb + mc - PW;
    v4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = v4{T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k0 = kFoldK * h;
      if (k0 < fkw) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int k = w + 4 * u, c = fc + 8 * u;
          Lp[64 * k + (lane ^ (16 * (k & 3)))] = (lane < bw && k0 + k < fkw) ? pl[h][u] : T(0);
          Up[kFoldK * c + (fk ^ usw(c))] = (c < bw && k0 + fk < fkw) ? pu[h][u] : T(0);
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < kFoldK / 4; ++ks) {
          const int k = 4 * ks + lk;
          const T uv = Up[kFoldK * mcol + (k ^ usw(mcol))];
#pragma unroll
          for (int t = 0; t < 4; ++t)
            acc[t] = Mfma16<T>::op(uv, Lp[64 * k + ((16 * t + l16) ^ (16 * lk))], acc[t]);
        }
        __syncthreads();
      }
    }
    // lane l of tile t holds row 16 t + l % 16, columns 4 (l / 16) .. + 3:
    // through LDS to one row per lane
    T* Tw = sl + w * 2 * PW * 64;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) Tw[(4 * lk + v) * 64 + 16 * t + l16] = acc[t][v];
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      a[i] = a[i] - Tw[i * 64 + lane];
      b[i] = b[i] - Tw[(PW + i) * 64 + lane];
    }
  }
  __syncthreads();
  int pos = lane < bw ? lane : -1;
  // First step of a piece ending at cn, for the panel x of columns c, c + 1,
  // .. < cend: the later pieces' entries right of the piece are set aside and
  // the piece's products summed from zero in their place; last step: the
  // entries take the sum off. Called under wave-uniform branches that hold a
  // compiler barrier, so that they stay branches instead of selects executed
  // at every step.
  auto piece_begin = [&](T (&x)[PW], int cn, int c, int cend) {
    __asm__ volatile("" ::: "memory");
    if (pos >= cn) {
#pragma unroll
      for (int i = 0; i < PW; ++i)
        if (c + i >= cn && c + i < cend) {
          ssv[(c + i - n0) * nv + lane - n0] = x[i];
          x[i] = T(0);
        }
    }
  };
  auto piece_end = [&](T (&x)[PW], int cn, int c, int cend) {
    __asm__ volatile("" ::: "memory");
    if (pos >= cn) {
#pragma unroll
      for (int i = 0; i < PW; ++i)
        if (c + i >= cn && c + i < cend) x[i] = ssv[(c + i - n0) * nv + lane - n0] + x[i];
    }
  };
  // A panel's next step k and the piece [plo, phi) holding it
  struct At {
    int k, pk, plo, phi;
  };
  auto next_piece = [&](At& t) {
    t.pk += 1;
    t.plo = t.phi;
    t.phi = __builtin_amdgcn_readfirstlane(spo[t.pk + 1]);
  };
  auto published = [&](int k) {
    return __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(&smeta[k], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
  };
  int seen = 0;  // steps whose interchanges are in pos
  // published step t.k (its word meta) applied to the panel x of columns c ..
  auto apply = [&](T (&x)[PW], At& t, int c, int meta) {
    const int k = t.k;
    if (k == t.phi) next_piece(t);
    const T lv = sl[k * bw + min(lane, bw - 1)];
    const int bl = meta & 0xff;
    const int kp = (meta >> 8) & 0xff;
    if (k == seen) {
      if ((meta >> 16) & 1) {
        pos = pos == k ? kp : pos;
        pos = lane == bl ? k : pos;
      }
      ++seen;
    }
    if (k == t.plo) piece_begin(x, t.phi, c, min(c + PW, bw));
    // rows not below subtract 0 u, which leaves a finite entry unchanged
    const T lb = pos > k ? lv : T(0);
#pragma unroll
    for (int i = 0; i < PW; ++i) x[i] = x[i] - lb * rdlane(x[i], bl);
    if (k == t.phi - 1) piece_end(x, t.phi, c, min(c + PW, bw));
    t.k = k + 1;
  };
  // Panel a, then panel b. Until the panel's own columns come, published
  // steps are applied to it first, and to panel b while none is waiting.
  At ta{0, 0, 0, 0}, tb;
  ta.phi = __builtin_amdgcn_readfirstlane(spo[1]);
  tb = ta;
#pragma unroll 1
  for (int c = ca; c < bw; c += 32) {
    for (int it = 0; ta.k < c && it < (1 << 24); ++it) {
      const int meta = published(ta.k);
      if (meta >= 0)
        apply(a, ta, c, meta);
      else if (c == ca && tb.k < ta.k && cb < bw)
        apply(b, tb, cb, published(tb.k));
    }
    // The columns [c, cend): a[0] is the current column, the panel shifts
    // left by one with each step. Column k's pivot lane bl and every lane's
    // reciprocal of its entry rc are known when its step begins; the columns
    // of one piece run without looking at piece boundaries
    const int cend = min(c + PW, bw);
    int bl = 0;
    T rc = T(0);
    auto search = [&](int k, int hi) {
      // without pivoting (SPD) the pivot row is the one at position k: lane k
      const bool cand = pos >= k && pos < hi;
      const unsigned key = pivot_key(a[0], cand);
      unsigned mx;
      const T r = recip_and_max(a[0], key, mx);
      rc = pin(a[0] == T(0) ? T(1) : r);  // a zero pivot scales nothing
      bl = k;
      if (s.pivot) {
        const unsigned long long msk = __ballot(key == mx);
        bl = __builtin_amdgcn_readfirstlane(__ffsll((long long)msk) - 1);
        if (__builtin_expect(mx == 0u || (msk & (msk - 1ull)) != 0ull, 0))
          bl = pivot_lane(a[0], pos, cand, k);
      }
    };
    if (ta.k == ta.phi) next_piece(ta);
#pragma unroll 1
    for (int k = c; k < cend;) {
      const int phi = ta.phi, ke = min(cend, phi);
      if (k == ta.plo) piece_begin(a, phi, k, cend);
      search(k, phi);
      T* slk = sl + k * bw + lane;
#pragma unroll 1
      for (;;) {
        const T v = a[0];
        const T inv = rdlane(rc, bl);
        const int kp = __builtin_amdgcn_readlane(pos, bl);
        const bool nz = rdlane(v, bl) != T(0);
        const int meta = bl | (kp << 8) | ((int)nz << 16);
        pos = (nz && pos == k) ? kp : pos;
        pos = (nz && lane == bl) ? k : pos;
        const bool below = pos > k;
        const T l = v * inv;
        const T lb = below ? l : T(0);
        // (no global memory access until the end: a release would wait for it)
        if (lane < bw) *slk = below ? l : v;
        slk += bw;
#pragma unroll
        for (int i = 1; i < PW; ++i) a[i - 1] = a[i] - lb * rdlane(a[i], bl);
        a[PW - 1] = T(0);
        if (k + 1 < ke) search(k + 1, phi);
        // published after the next search, when the write above has long
        // completed (the release waits for nothing)
        __hip_atomic_store(&smeta[k], meta, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (++k >= ke) break;
      }
      if (k == phi) {
        piece_end(a, phi, k, cend);
        if (k < bw) next_piece(ta);
      }
    }
    seen = cend;
    // the second panel: its steps go on where they were left
#pragma unroll
    for (int i = 0; i < PW; ++i) a[i] = b[i];
    ta = tb;
  }
  // the wave of the last column has seen every interchange
  if (w == (bw - 1) / PW % 4 && lane < bw) {
    spos[lane] = (unsigned char)pos;
    ssrc[pos] = (unsigned char)lane;
  }
  __syncthreads();
  const int fpos = lane < bw ? spos[lane] : 0;
  const int pr = lane < bw ? scp[lane] : 0;  // the piece of row (column) `lane`
  const int rlo = spo[pr];
  if ((int)threadIdx.x < bw) {
    const int m = smeta[threadIdx.x];
    ipvt[fc0 + c0 + threadIdx.x] = ((m >> 8) & 0xff) - rlo + 1;
    rperm[fc0 + c0 + threadIdx.x] = ssrc[threadIdx.x] | fpos << 8;
    // a zero pivot: the first piece that met one
    if (!((m >> 16) & 1)) atomicMin(first_fail, (unsigned long long)(d.piece + pr + 1));
  }
  // row r of a column at its position in the columns of its piece and right
  // of it, at its own row in earlier pieces' columns
  if (lane < bw) {
    for (int c = w; c < bw; c += 4)
      R[(c >= rlo ? fpos : lane) + (int64_t)c * L] = sl[c * bw + lane];
  }
}

template <typename T>
__global__ void __launch_bounds__(kWG)
blk_diag_slab_kernel(DevSym s, const BlkDesc* __restrict__ desc, T* __restrict__ arena,
                     int64_t* __restrict__ ipvt, int32_t* __restrict__ rperm,
                     unsigned long long* __restrict__ first_fail) {
  const int64_t vs = blockIdx.y;  // value set
  arena += vs * s.vs_arena;
  ipvt += vs * s.n;
  rperm += vs * s.n;
  extern __shared__ __attribute__((aligned(32))) unsigned char smem_a32[];
  blk_diag_slab_body<T>(s, desc[blockIdx.x], arena, ipvt, rperm, first_fail, smem_a32);
}

// Element of the operand entry (m, k) of 16 x 16 sub-block sb in LDS: the
// sixteen m of a lane group and the four k = 4 (l / 16) + st of a step fall
// in different banks, in float and in double, also as they are staged.
__device__ inline int op16(int sb, int m, int k) {
  return sb * 256 + m * 16 + ((((k & 3) << 2) | (k >> 2)) ^ m);
}

// Off-diagonal parts of blocks of at most 64 columns on the matrix cores:
// workgroups b < d.nl take 64 rows below the block (X = A U^-1), the others
// 64 columns right of it (X = L^-1 P A), sixteen per wave. The block is
// solved in sub-blocks of 16 columns (rows), each in four steps of four:
// lane l holds entries 4 (l / 16) .. + 3 of its row (column) l % 16, which is
// an accumulator tile and, as it stands, the next product's operand, so X
// never leaves the registers. The earlier sub-blocks' contribution is summed
// from zero and subtracted once; inside a sub-block, step j solves the four
// entries held by lanes l / 16 = j by substitution in those lanes and
// subtracts their products from the entries right of them (four MFMAs whose
// other operand lanes are zero). This is substitution throughout: an
// explicit inverse per 16 columns costs the same and lost accuracy on small
// pivots (factor error 1.4e-12 of the largest entry against 1.6e-13, also
// with one correction step). U is the region's whole upper triangle, and the
// interchanges of every piece are applied to A's rows and to the earlier
// pieces' L rows first (rperm: row | position << 8 per column, from the
// diagonal kernel), which does the reference's operations on the same
// values.
// Latency-bound (2 .. 400 workgroups per launch): 11 .. 15 us per launch
// (events), against 20 .. 28 us for substitution by one wave, one row per
// lane, with the other three waves idle; the whole class 15.5 -> 8.5 ms in
// double and 11.6 -> 6.9 ms in split-bf16 at 64^3, 20.1 -> 9.5 ms on
// elasticity 40^3 (SPD, split-bf16).
template <typename T>
__global__ void __launch_bounds__(kWG)
blk_offdiag64_kernel(const BlkDesc* __restrict__ desc, int ndesc, T* __restrict__ arena,
                     const int32_t* __restrict__ rperm, int64_t vs_arena, int64_t vs_n) {
  const int64_t vs = blockIdx.y;  // value set
  arena += vs * vs_arena;
  rperm += vs * vs_n;
  typedef typename Mfma16<T>::v4 v4;
  // operand sub-blocks (s, q), q <= s, at s (s + 1) / 2 + q
  __shared__ __attribute__((aligned(16))) T S[10 * 256];
  __shared__ T srinv[64];
  __shared__ int ssrc[64];
  const int tid = threadIdx.x, lane = tid % 64, wave = wave_id();
  const int l16 = lane % 16, lk = lane / 16;
  const int mi = std::is_same<T, double>::value ? 4 * (l16 % 4) + l16 / 4 : l16;
  const int di = find_blk(desc, ndesc, blockIdx.x);
  const BlkDesc& d = desc[di];
  const int b = blockIdx.x - d.wg_begin;
  const int L = d.L, c0 = d.c0, bw = d.c1 - d.c0, nl = d.nl;
  const int ns = (bw + 15) / 16;
  T* F = arena + d.foff;
  const T* Fd = F + c0 + (int64_t)c0 * L;  // the diagonal region
  const bool below = b < nl;
  const int g0 = d.c1 + (below ? b : b - nl) * 64 + 16 * wave + l16;  // row or column
  const int g = min(g0, L - 1);
  int rp = lane | lane << 8;
  if (!below && lane < bw) rp = rperm[d.fc0 + c0 + lane];
  T rv[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int c = wave + 4 * u;
    rv[u] = (lane < bw && c < bw) ? Fd[lane + (int64_t)c * L] : T(0);
  }
  v4 X[4];
  if (below) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int c = 16 * q + 4 * lk + v;
        X[q][v] = c < bw ? F[g + (int64_t)(c0 + c) * L] : T(0);
      }
    T dv = T(1);  // U's diagonal (1 past the block)
#pragma unroll
    for (int u = 0; u < 16; ++u)
      if (wave + 4 * u == lane && lane < bw) dv = rv[u];
    if (lane % 4 == wave) srinv[lane] = T(1) / dv;
  } else {
    // the first row of the lane's piece, and where each row comes from
    int ps = 0;
    for (int q = 0, o = 0; q < d.np; ++q) {
      if (lane >= o) ps = o;
      o += d.pw[q];
    }
    if (wave == 0) {
      ssrc[lane] = rp & 0xff;
      srinv[lane] = T(1);
    }
    __syncthreads();
    const T* Fa = F + c0 + (int64_t)g * L;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = 16 * q + 4 * lk + v;
        X[q][v] = r < bw ? Fa[ssrc[r]] : T(0);
      }
    rp = (rp >> 8 & 0xff) | ps << 8;
  }
  // the region's strict triangle, sub-block by sub-block (zero elsewhere)
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int c = wave + 4 * u;
    if (below) {  // U(k, m): k = lane, m = c
      if (lane / 16 <= c / 16)
        S[op16((c / 16) * (c / 16 + 1) / 2 + lane / 16, c % 16, lane % 16)] =
            lane < c ? rv[u] : T(0);
    } else {  // L(m, k): k = c, m = the lane's row, moved in earlier pieces' columns
      const int m = c < (rp >> 8) ? (rp & 0xff) : lane;
      if (m / 16 >= c / 16)
        S[op16((m / 16) * (m / 16 + 1) / 2 + c / 16, m % 16, c % 16)] = m > c ? rv[u] : T(0);
    }
  }
  __syncthreads();
  // acc + sub-block sb times the tile x
  auto mul = [&](int sb, const v4& x, v4 acc) {
#pragma unroll
    for (int st = 0; st < 4; ++st) acc = Mfma16<T>::op(S[op16(sb, mi, 4 * lk + st)], x[st], acc);
    return acc;
  };
  const v4 zero = v4{T(0), T(0), T(0), T(0)};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q < ns) {
      const int sd = q * (q + 1) / 2 + q;
      // the lane's own four-column triangle and reciprocals
      T m01 = S[op16(sd, 4 * lk + 1, 4 * lk)], m02 = S[op16(sd, 4 * lk + 2, 4 * lk)];
      T m03 = S[op16(sd, 4 * lk + 3, 4 * lk)], m12 = S[op16(sd, 4 * lk + 2, 4 * lk + 1)];
      T m13 = S[op16(sd, 4 * lk + 3, 4 * lk + 1)], m23 = S[op16(sd, 4 * lk + 3, 4 * lk + 2)];
      T r0 = srinv[16 * q + 4 * lk], r1 = srinv[16 * q + 4 * lk + 1];
      T r2 = srinv[16 * q + 4 * lk + 2], r3 = srinv[16 * q + 4 * lk + 3];
      v4 t = X[q];
      if (q > 0) {
        v4 acc = zero;
#pragma unroll
        for (int p = 0; p < q; ++p) acc = mul(q * (q + 1) / 2 + p, X[p], acc);
        t = t - acc;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const T x0 = t[0] * r0;
        const T x1 = (t[1] - x0 * m01) * r1;
        const T x2 = ((t[2] - x0 * m02) - x1 * m12) * r2;
        const T x3 = (((t[3] - x0 * m03) - x1 * m13) - x2 * m23) * r3;
        const bool mine = lk == j;
        const v4 xj = mine ? v4{x0, x1, x2, x3} : zero;
        if (mine) X[q] = xj;
        if (j < 3) {
          const v4 acc = mul(sd, xj, zero);
          if (lk > j) t = t - acc;
        }
      }
    }
  }
  if (g0 < L) {
    if (below) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int c = 16 * q + 4 * lk + v;
          if (c < bw) F[g + (int64_t)(c0 + c) * L] = X[q][v];
        }
    } else {
      T* Fa = F + c0 + (int64_t)g * L;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int r = 16 * q + 4 * lk + v;
          if (r < bw) Fa[r] = X[q][v];
        }
    }
  }
}

// Off-diagonal parts of one block in steps that hold a block of more than 64
// columns, by substitution (see the section comment); NQ bounds the piece
// width. Workgroups b < d.nl take 64 rows below the block, the others 64
// columns right of it. Dynamic LDS: 64 * kRLD + 128 * NQ elements.
template <typename T, int NQ>
__global__ void __launch_bounds__(kWG)
blk_offdiag_kernel(DevSym s, const BlkDesc* __restrict__ desc, int ndesc,
                   T* __restrict__ arena, const int64_t* __restrict__ ipvt) {
  const int64_t vs = blockIdx.y;  // value set
  arena += vs * s.vs_arena;
  ipvt += vs * s.n;
  extern __shared__ unsigned char smem_raw[];
  __shared__ int spiv[NQ > 64 ? NQ : 64];
  T* S = reinterpret_cast<T*>(smem_raw);
  const int tid = threadIdx.x, lane = tid % 64, wave = wave_id();
  const int di = find_blk(desc, ndesc, blockIdx.x);
  const BlkDesc d = desc[di];
  const int b = blockIdx.x - d.wg_begin;
  const int f = d.front;
  const int L = s.fL[f];
  const int64_t fc0 = s.fc0[f];
  const int c0 = d.c0, c1 = d.c1, bw = c1 - c0;
  T* F = arena + s.foff[f];
  if (b < d.nl) {
    // rows [r0, r0 + nr): X(i, k) at X[i + 64 k]
    const int r0 = c1 + b * 64, nr = min(64, L - r0);
    T* X = S;
    T* Us = S + 64 * kRLD;  // strip of the piece's columns: Us[k * NQ + j]
    T* Fx = F + r0 + (int64_t)c0 * L;
    for (int idx = tid; idx < 64 * bw; idx += kWG) X[idx] = T(0);
    __syncthreads();
    load_tile<T, 1, 64>(Fx, L, nr, bw, X);
    for (int pi = 0; pi < d.np; ++pi) {
      int64_t pc0, nq64;
      piece_cols(s, d.piece + pi, pc0, nq64);
      const int nq = (int)nq64;
      const int o = (int)(pc0 - fc0) - c0;
      load_tile<T, NQ, 1>(F + c0 + (int64_t)(c0 + o) * L, L, o + nq, nq, Us);
      __syncthreads();
      if (o > 0) {  // earlier pieces of the block: X_q -= X_<q U_<q,q
        for (int cb = wave * 8; cb < nq; cb += 32) {
          T acc[8];
#pragma unroll
          for (int jj = 0; jj < 8; ++jj) acc[jj] = T(0);
          const T* xr = X + lane;
          const T* ur = Us + min(cb, nq - 8 >= 0 ? nq - 8 : 0);
          for (int k = 0; k < o; ++k) {
            const T xv = xr[k * 64];
#pragma unroll
            for (int jj = 0; jj < 8; ++jj) acc[jj] += xv * ur[k * NQ + jj];
          }
          const int cs = min(cb, nq - 8 >= 0 ? nq - 8 : 0);  // shifted start
#pragma unroll
          for (int jj = 0; jj < 8; ++jj) {
            const int j = cs + jj;
            if (j >= cb && j < nq) X[lane + (o + j) * 64] -= acc[jj];
          }
        }
        __syncthreads();
      }
      if (wave == 0)  // X_q U_qq^-1, one row per lane
        blk_trsv<T, 64, NQ, 1, false>(X + lane + o * 64, Us + o * NQ, nullptr, nq);
      __syncthreads();
    }
    store_tile<T, 1, 64>(Fx, L, nr, bw, X);
  } else {
    // columns [j0, j0 + nc): A(r, c) at A[r + c * kRLD]
    const int j0 = c1 + (b - d.nl) * 64, nc = min(64, L - j0);
    T* A = S;
    T* Ls = S + 64 * kRLD;  // the piece's rows of L: Ls[i + k * NQ], k < o + nq
    T* Fa = F + c0 + (int64_t)j0 * L;
    for (int idx = tid; idx < 64 * kRLD; idx += kWG) A[idx] = T(0);
    __syncthreads();
    load_tile<T, 1, kRLD>(Fa, L, bw, nc, A);
    for (int pi = 0; pi < d.np; ++pi) {
      int64_t pc0, nq64;
      piece_cols(s, d.piece + pi, pc0, nq64);
      const int nq = (int)nq64;
      const int o = (int)(pc0 - fc0) - c0;
      load_tile<T, 1, NQ>(F + c0 + o + (int64_t)c0 * L, L, nq, o + nq, Ls);
      if (tid < nq) spiv[tid] = (int)ipvt[pc0 + tid] - 1;
      __syncthreads();
      if (o > 0) {  // earlier pieces: A_q -= L_q,<q A_<q (rows not yet swapped)
        T* ac = A + lane * kRLD;
        for (int ib = wave * 8; ib < nq; ib += 32) {
          const int is = min(ib, nq - 8 >= 0 ? nq - 8 : 0);
          T acc[8];
#pragma unroll
          for (int ii = 0; ii < 8; ++ii) acc[ii] = T(0);
          for (int k = 0; k < o; ++k) {
            const T av = ac[k];
#pragma unroll
            for (int ii = 0; ii < 8; ++ii) acc[ii] += Ls[is + ii + k * NQ] * av;
          }
#pragma unroll
          for (int ii = 0; ii < 8; ++ii) {
            const int i = is + ii;
            if (i >= ib && i < nq) ac[o + i] -= acc[ii];
          }
        }
        __syncthreads();
      }
      if (wave == 0) {  // interchanges, then L_qq^-1, one column per lane
        T* a = A + lane * kRLD + o;
        for (int k = 0; k < nq; ++k) {
          const int kp = spiv[k];
          if (kp != k) {
            const T t = a[k];
            a[k] = a[kp];
            a[kp] = t;
          }
        }
        blk_trsv<T, 1, NQ, 1, true>(a, Ls + o * NQ, nullptr, nq);
      }
      __syncthreads();
    }
    store_tile<T, 1, kRLD>(Fa, L, bw, nc, A);
  }
}

// The trailing update on the matrix cores: 64 x 64 tiles, each of the four
// waves owns a 32 x 32 quadrant as 2 x 2 MFMA tiles. The operands are passed
// as (U^T, L^T) so that the accumulator holds the tile transposed: lane l
// keeps row l % 16 of four consecutive columns, and each group of 16 lanes
// writes 16 contiguous rows of the column-major front.
//
// What bounds it, and why 64 x 64: most launches hold few tiles or a short
// inner dimension (K = 60 .. 480), so the fixed cost of a workgroup (first
// loads, the read-modify-write of its tile) and the last, nearly empty wave
// of workgroups weigh as much as the products. Against 128 x 128 tiles with
// 64 x 64 per wave (two workgroups per CU), workgroups of a quarter of the
// size (five per CU in double, where LDS is the limit, four in float, where
// registers are) measured, in us for fp64 / fp32 / split-bf16 (R the order of
// the updated square, before -> now):
//   12 fronts, R 1500, K 178: 318 -> 237 / 180 -> 120 / 102 -> 85
//   40 fronts, R  800, K 120: 238 -> 158 / 127 ->  85 /  92 -> 71
//   1 front,   R 2000, K 480: 103 ->  83 /  64 ->  47 /  41 -> 30
//   1 front,   R 1200, K 480:  94 ->  45 /  60 ->  25 /  39 -> 21
//   1 front,   R  500, K 200:  46 ->  14 /  29 ->   9 /  21 -> 10
//   1 front,   R 4000, K 480: 340 -> 342 / 193 -> 166 /  95 -> 104
// (only the last, in split-bf16, reads its panels often enough for the
// larger tile to win). Loads are unconditional vectors of 16 bytes from
// clamped addresses: rows past the rectangle only reach accumulator rows
// that are not stored, the inner dimension's tail is zeroed as it is staged.

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 64;  // rows and columns of a trailing-update tile

// 16-byte vectors of the front's elements: as loaded (element alignment)
// and as staged in LDS (16-byte alignment).
template <typename T>
struct Vec16;
template <>
struct Vec16<double> {
  static constexpr int n = 2;
  typedef double load __attribute__((ext_vector_type(2), aligned(8)));
  typedef double lds __attribute__((ext_vector_type(2)));
};
template <>
struct Vec16<float> {
  static constexpr int n = 4;
  typedef f4u load;
  typedef float lds __attribute__((ext_vector_type(4)));
};

// Tile of workgroup bid among n: workgroups go to the eight XCDs in turn, so
// each XCD takes runs of up to kXcdRun consecutive tiles (which share the
// panels of one front in its L2) out of every 8 kXcdRun; the last n mod
// (8 run) tiles keep their order. Measured on 200 fronts of R 300, K 90:
// 131 -> 99 us (fp64), 77 -> 47 us (split-bf16); on one large front the
// same within 2 %. Runs are short so that fronts of unlike depth in one
// launch still spread over all XCDs.
constexpr int kXcdRun = 32;
__device__ inline int xcd_tile(int bid, int n) {
  const int run = min(kXcdRun, n / 8);
  if (run < 2) return bid;
  const int round = 8 * run;
  if (bid >= n / round * round) return bid;
  const int x = bid % 8, g = bid / 8;
  return (g / run) * round + x * run + g % run;
}

// four floats to bf16 (round to nearest even), two per v_cvt_pk_bf16_f32
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ inline uint2 pack_bf16(float a, float b, float c, float d) {
  const bf16x2 p = {(__bf16)a, (__bf16)b}, q = {(__bf16)c, (__bf16)d};
  return uint2{__builtin_bit_cast(unsigned, p), __builtin_bit_cast(unsigned, q)};
}
// the part of x below its bf16 rounding (exact: x and its rounding are floats
// within a factor of two of each other)
__device__ inline float bf_lo(float x) { return x - (float)(__bf16)x; }
__device__ inline uint2 pack_f16(float a, float b, float c, float d) {
  const f16x4 p = {(_Float16)a, (_Float16)b, (_Float16)c, (_Float16)d};
  return __builtin_bit_cast(uint2, p);
}

// One tile's products with 16-bit operands on the gfx950 matrix cores
// (v_mfma_f32_16x16x32_bf16 / _f16), K-chunks of 32, double-buffered in LDS:
// A(i, k) = L21 rows at part 0, row i, B(k, j) = U12 columns at part 1, row
// j; each lane reads its operand
// (eight consecutive k) with one 16-byte LDS read. lowp 1: bf16; lowp 3:
// split bf16, x = hi + lo (lo at parts 2 and 3), products lo_b hi_a +
// hi_b lo_a + hi_b hi_a; lowp 2: fp16 under diagonal scaling: A(i, k) times
// and B(k, j) divided by 2^e_k, the power of two nearest below |U(k, k)|
// (the product is unchanged; both stay in fp16 range when A is diagonally
// scaled). Waves 0-1 stage A (rows 4 ag .. 4 ag + 3, k = 4 q + u), waves
// 2-3 B (columns bc + 16 u, k = 4 q .. 4 q + 3). Row r of an array lies at
// row place 16 (r % 4) + r / 4 of 64 bytes, its 16-byte units exchanged by
// r % 4: the 32 lanes of a half-wave store rows 4 apart and the 16 lanes of
// an operand read take consecutive rows, both without bank conflicts and
// without padding (32 KB).
constexpr int kB16Part = kTile * 32;      // one operand array, halves
// k = 8 unit .. of row r
__device__ inline int at16(int r, int unit) {
  return ((r & 3) * 16 + (r >> 2)) * 32 + ((unit ^ (r & 3)) * 8);
}
template <int lowp>
__device__ __attribute__((always_inline)) inline void gemm16_tile(
    const float* __restrict__ F, int L, int k0, int bw, int r0, int rend, int j0, int cend,
    unsigned char* lds_raw, f32x4 (&acc)[2][2]) {
  constexpr int KC = 32;
  unsigned short* base = reinterpret_cast<unsigned short*>(lds_raw);
  auto part = [&](int buf, int which) { return base + (buf * 4 + which) * kB16Part; };
  const int tid = threadIdx.x, lane = tid % 64, wave = wave_id();
  const int wr = (wave % 2) * 32, wc = (wave / 2) * 32;
  const int l16 = lane % 16, lk = lane / 16;
  const bool isA = wave < 2;
  const int t7 = tid % 128, q = t7 % 8, ag = t7 / 8;
  const int bc = 4 * ((t7 / 8) % 4) + t7 / 32;
  // A: p[u] = row 4 ag of column k0 + 4 q + u; B: p[u] = k0 + 4 q of column
  // j0 + bc + 16 u
  const float* pA = F + min(r0 + 4 * ag, rend - 1) + (int64_t)k0 * L;
  const float* pB[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) pB[u] = F + k0 + (int64_t)min(j0 + bc + 16 * u, cend - 1) * L;
  f4u rg[4];
  float sc[4];
  // 2^e (A) or 2^-e (B) of the diagonal entry of front column k0 + k (1 when
  // the entry is zero, subnormal or not finite)
  auto pow2 = [&](int k) {
    const float dg = F[(int64_t)(k0 + min(k, bw - 1)) * (L + 1)];
    const unsigned be = (__float_as_uint(dg) >> 23) & 0xffu;
    if (be == 0u || be >= 254u) return 1.0f;
    return __uint_as_float((isA ? be : 254u - be) << 23);
  };
  auto gload = [&](int kc) {
    const int kq = kc + 4 * q;
    if (isA) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        rg[u] = *reinterpret_cast<const f4u*>(pA + (int64_t)min(kq + u, bw - 1) * L);
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) rg[u] = *reinterpret_cast<const f4u*>(pB[u] + min(kq, bw - 1));
    }
    if (lowp == 2)
#pragma unroll
      for (int u = 0; u < 4; ++u) sc[u] = pow2(kq + u);
  };
  auto lstore = [&](int buf, int kc) {
    const int kq = kc + 4 * q;
    // rg[u][e]: row e of k = kq + u (A), column u of k = kq + e (B)
    const bool tail = kc + KC > bw;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (lowp == 2) rg[u][e] *= isA ? sc[u] : sc[e];
        if (tail && kq + (isA ? u : e) >= bw) rg[u][e] = 0.0f;
      }
    if (isA) {
      unsigned short* P = part(buf, 0) + 4 * (q & 1);
      unsigned short* Q = part(buf, 2) + 4 * (q & 1);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x0 = rg[0][e], x1 = rg[1][e], x2 = rg[2][e], x3 = rg[3][e];
        *reinterpret_cast<uint2*>(P + at16(4 * ag + e, q / 2)) =
            lowp == 2 ? pack_f16(x0, x1, x2, x3) : pack_bf16(x0, x1, x2, x3);
        if (lowp == 3)
          *reinterpret_cast<uint2*>(Q + at16(4 * ag + e, q / 2)) =
              pack_bf16(bf_lo(x0), bf_lo(x1), bf_lo(x2), bf_lo(x3));
      }
    } else {
      unsigned short* P = part(buf, 1) + 4 * (q & 1);
      unsigned short* Q = part(buf, 3) + 4 * (q & 1);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float x0 = rg[u][0], x1 = rg[u][1], x2 = rg[u][2], x3 = rg[u][3];
        *reinterpret_cast<uint2*>(P + at16(bc + 16 * u, q / 2)) =
            lowp == 2 ? pack_f16(x0, x1, x2, x3) : pack_bf16(x0, x1, x2, x3);
        if (lowp == 3)
          *reinterpret_cast<uint2*>(Q + at16(bc + 16 * u, q / 2)) =
              pack_bf16(bf_lo(x0), bf_lo(x1), bf_lo(x2), bf_lo(x3));
      }
    }
  };
  const int nch = (bw + KC - 1) / KC;
  gload(0);
  lstore(0, 0);
  if (nch > 1) gload(KC);
  __syncthreads();
  for (int ch = 0; ch < nch; ++ch) {
    const int cur = ch & 1;
    // the next chunk goes to the other buffer (every wave left it at the
    // last barrier) and the one after is requested before the products
    if (ch + 1 < nch) {
      lstore(cur ^ 1, (ch + 1) * KC);
      if (ch + 2 < nch) gload((ch + 2) * KC);
    }
    auto frag = [&](int which, int row) {
      return *reinterpret_cast<const bf16x8*>(part(cur, which) + at16(row, lk));
    };
    bf16x8 ah[2], bh[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      ah[t] = frag(0, wr + t * 16 + l16);
      bh[t] = frag(1, wc + t * 16 + l16);
    }
    if (lowp == 3) {
      bf16x8 al[2], bl[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        al[t] = frag(2, wr + t * 16 + l16);
        bl[t] = frag(3, wc + t * 16 + l16);
      }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl[c], ah[a], acc[a][c], 0, 0, 0);
          acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[c], al[a], acc[a][c], 0, 0, 0);
          acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[c], ah[a], acc[a][c], 0, 0, 0);
        }
    } else if (lowp == 2) {
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              __builtin_bit_cast(f16x8, bh[c]), __builtin_bit_cast(f16x8, ah[a]), acc[a][c], 0, 0,
              0);
    } else {
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[c], ah[a], acc[a][c], 0, 0, 0);
    }
    __syncthreads();
  }
}

// The same tile in the front's own type (v_mfma_f64_16x16x4f64 /
// v_mfma_f32_16x16x4f32), K-chunks of 16, double-buffered in LDS:
// A(i, k) at As[64 k + (i ^ 16 (k % 4))], B(k, j) at Bs[16 j + (k ^ s(j))]
// with s(j) = 2 (j / 2 % 8) in double, 4 (j / 4 % 4) in float: the operand
// reads fall in different banks without padding. Column j of an accumulator tile is taken from U column
// mcol(j), chosen so that both types leave four consecutive columns
// 4 lk .. 4 lk + 3 in a lane (the f64 form puts row 4 v + lk in element v).
constexpr int kGK = 16;            // inner dimension per chunk
template <typename T>
constexpr int kGemmTLds = 4 * kGK * kTile * (int)sizeof(T);
template <typename T>
__device__ __attribute__((always_inline)) inline void gemmT_tile(
    const T* __restrict__ F, int L, int k0, int bw, int r0, int rend, int j0, int cend,
    unsigned char* lds_raw, typename Mfma16<T>::v4 (&acc)[2][2]) {
  constexpr int VE = Vec16<T>::n;
  constexpr int U = kTile * kGK / VE / kWG;  // vectors per thread and operand
  typedef typename Vec16<T>::load V;
  typedef typename Vec16<T>::lds VL;
  T (*As)[kGK * kTile] = reinterpret_cast<T (*)[kGK * kTile]>(lds_raw);
  T (*Bs)[kGK * kTile] = As + 2;
  auto swb = [](int j) {
    return std::is_same<T, double>::value ? 2 * ((j >> 1) & 7) : 4 * ((j >> 2) & 3);
  };
  const int tid = threadIdx.x, lane = tid % 64, wave = wave_id();
  const int wr = (wave % 2) * 32, wc = (wave / 2) * 32;
  const int l16 = lane % 16, lk = lane / 16;
  const int mcol = std::is_same<T, double>::value ? 4 * (l16 % 4) + l16 / 4 : l16;
  // vector v of a chunk: A rows VE (v % (64 / VE)) .. of k = v / (64 / VE);
  // B k = VE (v % (16 / VE)) .. of column v / (16 / VE)
  constexpr int RV = kTile / VE, KV = kGK / VE;
  const T* pA[U];
  const T* pB[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int v = tid + u * kWG;
    pA[u] = F + min(r0 + VE * (v % RV), rend - 1) + (int64_t)k0 * L;
    pB[u] = F + k0 + (int64_t)min(j0 + v / KV, cend - 1) * L;
  }
  V ra[U], rb[U];
  auto gload = [&](int kc) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v = tid + u * kWG;
      ra[u] = *reinterpret_cast<const V*>(pA[u] + (int64_t)min(kc + v / RV, bw - 1) * L);
      rb[u] = *reinterpret_cast<const V*>(pB[u] + min(kc + VE * (v % KV), bw - 1));
    }
  };
  auto lstore = [&](int buf, int kc) {
    if (kc + kGK > bw) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int v = tid + u * kWG;
        const bool in = kc + v / RV < bw;
#pragma unroll
        for (int e = 0; e < VE; ++e) {
          if (!in) ra[u][e] = T(0);
          if (kc + VE * (v % KV) + e >= bw) rb[u][e] = T(0);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v = tid + u * kWG;
      const int k = v / RV, j = v / KV;
      *reinterpret_cast<VL*>(&As[buf][k * kTile + ((VE * (v % RV)) ^ (16 * (k & 3)))]) = ra[u];
      *reinterpret_cast<VL*>(&Bs[buf][j * kGK + ((VE * (v % KV)) ^ swb(j))]) = rb[u];
    }
  };
  const int nch = (bw + kGK - 1) / kGK;
  gload(0);
  lstore(0, 0);
  if (nch > 1) gload(kGK);
  __syncthreads();
  for (int ch = 0; ch < nch; ++ch) {
    const int cur = ch & 1;
    if (ch + 1 < nch) {  // as in gemm16_tile
      lstore(cur ^ 1, (ch + 1) * kGK);
      if (ch + 2 < nch) gload((ch + 2) * kGK);
    }
#pragma unroll
    for (int ks = 0; ks < kGK / 4; ++ks) {
      const int kk = ks * 4 + lk;
      T av[2], bv[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int j = wc + t * 16 + mcol;
        av[t] = As[cur][kk * kTile + ((wr + t * 16 + l16) ^ (16 * lk))];
        bv[t] = Bs[cur][j * kGK + (kk ^ swb(j))];
      }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c) acc[a][c] = Mfma16<T>::op(bv[c], av[a], acc[a][c]);
    }
    __syncthreads();
  }
}

// LDS bytes of blk_gemm_body.
template <typename T>
constexpr int kGemmLds = (std::is_same<T, float>::value && 2 * 4 * kB16Part * 2 > kGemmTLds<T>)
                             ? 2 * 4 * kB16Part * 2
                             : kGemmTLds<T>;

// Tile t of a trailing-update launch over desc[0, ndesc); lds_raw:
// kGemmLds<T> bytes. With lowp set, a float update of a front wider than 256
// columns takes its L21 / U12 operands in 16 bits and accumulates in float
// (gemm16_tile); refinement in double recovers the accuracy.
template <typename T>
__device__ __attribute__((always_inline)) void blk_gemm_body(
    const DevSym& s, const GemmDesc* __restrict__ desc, int ndesc, T* __restrict__ arena,
    int lowp, int t, unsigned char* lds_raw) {
  typedef typename Mfma16<T>::v4 v4;
  const int lane = threadIdx.x % 64, wave = wave_id();
  const int di = find_blk(desc, ndesc, t);
  const GemmDesc d = desc[di];
  const int b = t - d.wg_begin;
  const int L = d.L;
  T* F = arena + d.foff;
  const int bw = d.k1 - d.k0;
  const int rend = d.r0 + d.nr, cend = d.j0 + d.nc;
  const int r0 = d.r0 + (b % d.ntr) * kTile, j0 = d.j0 + (b / d.ntr) * kTile;
  // symmetric fronts: an entry whose row lies past the tile's last column
  // also stands for its transpose, which no tile computes (a tile column's
  // own square, its first tile, is computed whole)
  const int mend = d.mirror ? min(j0 + kTile, cend) : (1 << 30);
  const int wr = (wave % 2) * 32, wc = (wave / 2) * 32;
  const int l16 = lane % 16, lk = lane / 16;
  // the products are summed from zero and subtracted from A22 once at the
  // end: starting the accumulators from A22 instead loses accuracy when
  // |A22| >> |L21 U12| (measured 8x larger backward error on the 3D
  // convection-diffusion operator)
  v4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int c = 0; c < 2; ++c) acc[a][c] = v4{T(0), T(0), T(0), T(0)};
  if constexpr (std::is_same<T, float>::value) {
    if (lowp == 1 && d.big)
      gemm16_tile<1>(F, L, d.k0, bw, r0, rend, j0, cend, lds_raw, acc);
    else if (lowp == 2 && d.big)
      gemm16_tile<2>(F, L, d.k0, bw, r0, rend, j0, cend, lds_raw, acc);
    else if (lowp == 3 && d.big)
      gemm16_tile<3>(F, L, d.k0, bw, r0, rend, j0, cend, lds_raw, acc);
    else
      gemmT_tile<T>(F, L, d.k0, bw, r0, rend, j0, cend, lds_raw, acc);
  } else {
    gemmT_tile<T>(F, L, d.k0, bw, r0, rend, j0, cend, lds_raw, acc);
  }
  // A22 -= the products: all 16 reads of a lane are issued before its writes
  // (one memory round trip)
  T cv[2][2][4];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int r = min(r0 + wr + a * 16 + l16, rend - 1);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        cv[a][c][v] = F[r + (int64_t)min(j0 + wc + c * 16 + 4 * lk + v, cend - 1) * L];
  }
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int r = r0 + wr + a * 16 + l16;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int col = j0 + wc + c * 16 + 4 * lk + v;
        if (r < rend && col < cend) {
          const T nv = cv[a][c][v] - acc[a][c][v];
          F[r + (int64_t)col * L] = nv;
          if (r >= mend) F[col + (int64_t)r * L] = nv;
        }
      }
  }
}

template <typename T>
__global__ void __launch_bounds__(kWG, 4)
blk_gemm_kernel(DevSym s, const GemmDesc* __restrict__ desc, int ndesc,
                T* __restrict__ arena, int lowp) {
  const int64_t vs = blockIdx.y;  // value set
  arena += vs * s.vs_arena;
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[kGemmLds<T>];
  blk_gemm_body<T>(s, desc, ndesc, arena, lowp, xcd_tile(blockIdx.x, gridDim.x), lds_raw);
}

// The diagonal regions of one block step (workgroups b < ndiag, with the
// previous block's product folded in) beside the rest of the previous
// block's update within its block group (the others): the two touch
// disjoint parts of each front, so one launch holds both and the update
// leaves the step's critical path.
template <typename T>
__global__ void __launch_bounds__(kWG)
blk_diag_border_kernel(DevSym s, const BlkDesc* __restrict__ ddesc, int ndiag,
                       const GemmDesc* __restrict__ gdesc, int ngemm, T* __restrict__ arena,
                       int64_t* __restrict__ ipvt, int32_t* __restrict__ rperm,
                       unsigned long long* __restrict__ first_fail, int lowp) {
  const int64_t vs = blockIdx.y;  // value set
  arena += vs * s.vs_arena;
  ipvt += vs * s.n;
  rperm += vs * s.n;
  // dynamic: the larger of the regions' slabs and kGemmLds<T>
  extern __shared__ __attribute__((aligned(32))) unsigned char smem_a32[];
  if ((int)blockIdx.x < ndiag)
    blk_diag_slab_body<T>(s, ddesc[blockIdx.x], arena, ipvt, rperm, first_fail, smem_a32);
  else
    blk_gemm_body<T>(s, gdesc, ngemm, arena, lowp,
                     xcd_tile((int)blockIdx.x - ndiag, (int)gridDim.x - ndiag), smem_a32);
}

// ---------------------------------------------------------------------------
// Triangular solves, one elimination-tree level at a time.
// Forward (_lulsolve!, SpkLUFactor.jl:269-323). A front's vector y (length
// L per right-hand side, in the vector arena) starts as the permuted rhs on
// its W own columns and zero on its R update rows, and receives the
// children's update vectors through the relative-index maps (the
// multifrontal form of the reference's scatter rhs[lindx] += temp). Then,
// block by block (the factor's blocks of pieces): a one-workgroup chain
// solves the block's pieces in LDS (interchanges, unit-lower block solve,
// rows below inside the block) and a many-workgroup GEMV updates every row
// below the block, y[c1:L] -= L[c1:L, c0:c1] y[c0:c1].
// Backward (_luusolve!, :325-377), blocks in reverse: t = U[c0:c1, c1:L]
// x[I[c1:L]] (a workgroup per row or eight), then the chain: y = x - t, per piece in
// reverse the in-block U12 part and the upper block solve.
// Small fronts (L <= kSmallLmax) do everything in one wave per block of
// right-hand sides.
// ---------------------------------------------------------------------------
// Large fronts, forward: y = [rhs on own columns; 0] + children, one thread
// per (front, row) item of the level (the factor's column items: a front's
// rows and columns share its index list). The children's entries come from
// the item's (child, row) list in ascending child order, so each entry is
// the same sum in the same order as a per-front gather; a level's fronts
// spread over many workgroups.
template <typename T>
__device__ inline void fwd_assemble_rows(const DevSym& s, const LevelRows& m, int b,
                                         const T* __restrict__ rhs, int64_t ldr, int nrhs,
                                         T* __restrict__ vec) {
  const int z = b / m.nb;
  const int item = (b - z * m.nb) * kWG + threadIdx.x;
  if (item >= m.n) return;
  const int f = m.front[item], r = m.row[item];
  const int L = s.fL[f], W = s.fW[f];
  const int64_t fc0 = s.fc0[f];
  const int64_t e0 = m.ea[item], e1 = m.ea[item + 1];
  for (int q = z; q < nrhs; q += m.qz) {
    T y = (r < W) ? rhs[(int64_t)q * ldr + fc0 + r] : T(0);
    for (int64_t e = e0; e < e1; ++e) {
      const int c = m.ea_child[e], t = m.ea_t[e];
      y += vec[s.fvec[c] * nrhs + (int64_t)q * s.fL[c] + s.fW[c] + t];
    }
    vec[s.fvec[f] * nrhs + (int64_t)q * L + r] = y;
  }
}

// Backward: the update rows of each large front's solve vector gathered
// from the solution by the front's index list, one thread per (front, row)
// item of the level.
template <typename T>
__device__ inline void bwd_gather_rows(const DevSym& s, const LevelRows& m, int b,
                                       const T* __restrict__ rhs, int64_t ldr, int nrhs,
                                       T* __restrict__ vec) {
  const int z = b / m.nb;
  const int item = (b - z * m.nb) * kWG + threadIdx.x;
  if (item >= m.n) return;
  const int f = m.front[item], j = m.row[item];
  const int L = s.fL[f], W = s.fW[f];
  if (j < W) return;
  const int g = s.lindx[s.xlindx[s.fsp0[f]] - 1 + j] - 1;
  for (int q = z; q < nrhs; q += m.qz)
    vec[s.fvec[f] * nrhs + (int64_t)q * L + j] = rhs[(int64_t)q * ldr + g];
}

// Per-block solve data, built once per factorisation and read by every
// solve (refinement solves many times). A block of bw columns is padded to
// bwp = 4 ng columns, ng = ceil(bw / 4), in ng panels of four columns.
//  - Lower part (8 ng (ng + 1) elements): panel g holds rows 4g .. bwp-1 of
//    columns 4g .. 4g+3 of the unit-lower factor, four values per row, at
//    lo_panel(g, ng); entries on or above the diagonal and padding are 0.
//    The rows of every piece carry that piece's interchanges also in the
//    columns of earlier pieces: the reference interchanges y's rows when it
//    reaches a piece, after earlier pieces have updated them; interchanging
//    y once at the start and the stored L rows instead does the same
//    operations on the same values.
//  - Upper part (8 ng (ng + 1) elements): panel g holds rows 0 .. 4g+3 of
//    columns 4g .. 4g+3 of U, at up_panel(g); entries below the diagonal are
//    0, padding columns are unit columns.
//  - The bwp reciprocals of U's diagonal (1 for padding).
// In all 16 ng (ng + 1) + 4 ng elements, from element 4 desc.aux. The
// integer part (kPrepInts per block, from desc.r0 kPrepInts) is the row each
// position takes after its piece's interchanges (composed, glaswp! order).
__device__ inline int lo_panel(int g, int ng) { return 4 * (4 * ng * g - 2 * g * (g - 1)); }
__device__ inline int up_panel(int g) { return 8 * g * (g + 1); }
constexpr int kPanelElems = 8 * 32 * 33;  // one part of a 128-column block

template <typename T>
struct Vec4;
template <>
struct Vec4<double> {
  typedef double __attribute__((ext_vector_type(4))) type;
  typedef double __attribute__((ext_vector_type(2))) half;
};
template <>
struct Vec4<float> {
  typedef float __attribute__((ext_vector_type(4))) type;
  typedef float __attribute__((ext_vector_type(2))) half;
};

// One workgroup per block.
template <typename T>
__global__ void __launch_bounds__(kWG)
solve_prep_kernel(DevSym s, const SolveDesc* __restrict__ desc, const T* __restrict__ lnz,
                  const T* __restrict__ unz, const int64_t* __restrict__ ipvt,
                  T* __restrict__ prep, int32_t* __restrict__ prepi) {
  const int64_t vs = blockIdx.y;  // value set
  lnz += vs * s.vs_lnz;
  unz += vs * s.vs_unz;
  ipvt += vs * s.n;
  prep += vs * s.vs_prep;
  prepi += vs * s.vs_prepi;
  __shared__ int spiv[128];
  __shared__ int sperm[128];
  __shared__ int pstart[128];
  __shared__ int pbeg[9];
  __shared__ int64_t lb[128], ub[128];
  const int tid = threadIdx.x, lane = tid % 64, wave = wave_id();
  const SolveDesc d = desc[blockIdx.x];
  const int64_t fc0 = s.fc0[d.front];
  const int c0 = d.c0, bw = d.c1 - d.c0;
  const int ng = (bw + 3) / 4, bwp = 4 * ng;
  const int64_t g0 = fc0 + c0;
  T* lo = prep + 4 * (int64_t)d.aux;
  T* up = lo + 8 * ng * (ng + 1);
  T* rinv = up + 8 * ng * (ng + 1);
  for (int i = tid; i < bw; i += kWG) {
    const int ps = piece_start_of_col(s, fc0, c0 + i) - c0;
    pstart[i] = ps;
    spiv[i] = ps + (int)ipvt[g0 + i] - 1;
    sperm[i] = i;
    lb[i] = s.lcol[g0 + i] + c0;
    ub[i] = s.ucol[g0 + i] + c0;
  }
  if (tid <= d.np) pbeg[tid] = (tid < d.np) ? (int)(s.xsuper[d.piece + tid] - 1 - g0) : bw;
  __syncthreads();
  if (wave == 0 && lane < d.np) {
    for (int k = pbeg[lane]; k < pbeg[lane + 1]; ++k) {
      const int kp = spiv[k];
      if (kp != k) {
        const int t = sperm[k];
        sperm[k] = sperm[kp];
        sperm[kp] = t;
      }
    }
  }
  __syncthreads();
  for (int g = wave; g < ng; g += 4) {
    T* P = lo + lo_panel(g, ng);
    const int ne = (bwp - 4 * g) * 4;
#pragma unroll 4
    for (int i = lane; i < ne; i += 64) {
      const int r = 4 * g + i / 4, c = 4 * g + i % 4;
      T v = T(0);
      if (r > c && r < bw && c < bw) v = lnz[lb[c] + (pstart[r] == pstart[c] ? r : sperm[r])];
      P[i] = v;
    }
  }
  for (int g = wave; g < ng; g += 4) {
    T* P = up + up_panel(g);
    const int ne = (4 * g + 4) * 4;
#pragma unroll 4
    for (int i = lane; i < ne; i += 64) {
      const int r = i / 4, c = 4 * g + i % 4;
      T v = T(0);
      if (r <= c) {
        if (c < bw)
          v = (r >= pstart[c]) ? lnz[lb[c] + r] : unz[ub[r] + c];
        else if (r == c)
          v = T(1);
      }
      P[i] = v;
    }
  }
  for (int c = tid; c < bwp; c += kWG) rinv[c] = (c < bw) ? T(1) / lnz[lb[c] + c] : T(1);
  int32_t* pi = prepi + (int64_t)d.r0 * kPrepInts;
  for (int i = tid; i < bw; i += kWG) pi[i] = sperm[i];
}

// Entry src (0 <= src < 128, per lane) of the same two-per-lane vector.
template <typename T>
__device__ inline T gather2(T y0, T y1, int src) {
  const T a = __shfl(y0, src & 63, 64), b = __shfl(y1, src & 63, 64);
  return src < 64 ? a : b;
}

// The solve data of a block (nv four-element vectors) into LDS, all loads in
// flight at once; at most kPrepV vectors per thread.
constexpr int kPrepV = 9;
template <typename V>
__device__ inline void load_panels(const V* __restrict__ src, V* dst, int nv) {
  V buf[kPrepV];
#pragma unroll
  for (int u = 0; u < kPrepV; ++u) {
    const int i = threadIdx.x + u * kWG;
    if (i < nv) buf[u] = src[i];
  }
#pragma unroll
  for (int u = 0; u < kPrepV; ++u) {
    const int i = threadIdx.x + u * kWG;
    if (i < nv) dst[i] = buf[u];
  }
}

// Forward chain of one block (one workgroup per front of the step). The
// block's lower panels come from the solve data in one coalesced load. Wave
// 0 holds y in registers, two entries per lane (rows lane, lane + 64),
// takes the block's interchanges at once (cross-lane shuffles) and
// eliminates four columns per step: the four new entries from a small
// unit-lower solve every lane does alike, then every row takes its four
// products in column order — the same operations, in the same order, as
// the reference's column-by-column piece solves and in-block L21 updates.
// A row at or above the step's first column reads the panel's zero row
// (its own four products are then exact no-ops), so the three rows below
// the first come out as the small solve's entries and no lane branches.
// The next step's panel values are read from LDS while the current step
// computes; once the first 64 rows are final only the second half updates.
template <typename T>
struct FwdStep {
  T t10, t32;                        // L(k+1, k), L(k+3, k+2)
  typename Vec4<T>::half t2, t3;     // L(k+2, k:k+2), L(k+3, k:k+2)
  typename Vec4<T>::type a, b;       // the lane's two rows
};

template <typename T>
__device__ __attribute__((always_inline)) void fwd_chain_body(
    const DevSym& s, const SolveDesc& d, const T* __restrict__ prep,
    const int32_t* __restrict__ prepi, T* __restrict__ rhs, int64_t ldr, int nrhs,
    T* __restrict__ vec, unsigned char* smem_a32) {
  using V = typename Vec4<T>::type;
  V* smem_v4 = reinterpret_cast<V*>(smem_a32);
  const T* R = reinterpret_cast<const T*>(smem_a32);
  const int tid = threadIdx.x, lane = tid % 64;
  // wave w takes right-hand sides w, w + 4, ..., spread over the z workgroups
  const int wave = wave_id() + 4 * (int)blockIdx.z, qstep = 4 * (int)gridDim.z;
  const int f = d.front;
  const int L = d.L;
  const int64_t fc0 = d.fc0;
  const int c0 = d.c0, bw = d.c1 - d.c0;
  const int ng = (bw + 3) / 4, bwp = 4 * ng;
  const bool in0 = lane < bw, in1 = lane + 64 < bw;
  const int32_t* pi = prepi + (int64_t)d.r0 * kPrepInts;
  // every wave: the permutation and its first right-hand side (wave w
  // takes right-hand sides w, w + 4, ...), in flight with the panels
  int s0 = lane, s1 = lane + 64;
  T y0r = T(0), y1r = T(0);
  const T* yv = vec + d.fvec * nrhs + (int64_t)wave * L;
  if (wave < nrhs) {
    if (in0) {
      s0 = pi[lane];
      y0r = yv[c0 + lane];
    }
    if (in1) {
      s1 = pi[lane + 64];
      y1r = yv[c0 + 64 + lane];
    }
  }
  load_panels(reinterpret_cast<const V*>(prep + 4 * (int64_t)d.aux), smem_v4,
              2 * ng * (ng + 1));
  __syncthreads();
  if (wave >= nrhs) return;
  const int gA = min(ng, 16);
  // panel values of step g (rows clamped into the panel)
  auto load = [&](int g, FwdStep<T>& o, bool both) {
    const int k = 4 * g;
    const T* P = R + lo_panel(g, ng);
    using H = typename Vec4<T>::half;
    o.t10 = P[4];
    o.t2 = *(const H*)(P + 8);
    o.t3 = *(const H*)(P + 12);
    o.t32 = P[14];
    if (both) o.a = *(const V*)(P + 4 * (min(max(lane, k), bwp - 1) - k));
    o.b = *(const V*)(P + 4 * (min(max(lane + 64, k), bwp - 1) - k));
  };
  for (int q = wave; q < nrhs; q += qstep) {
    T* yg = vec + d.fvec * nrhs + (int64_t)q * L;
    T* x = rhs + (int64_t)q * ldr;
    if (q > wave) {
      y0r = in0 ? yg[c0 + lane] : T(0);
      y1r = in1 ? yg[c0 + 64 + lane] : T(0);
    }
    T y0 = gather2(y0r, y1r, s0), y1 = gather2(y0r, y1r, s1);
    FwdStep<T> A, B;
    // pivots in rows 0..63: both halves update
    auto stepA = [&](int g, const FwdStep<T>& c, FwdStep<T>& n) {
      const int k = 4 * g;
      load(min(g + 1, ng - 1), n, true);
      const T b0 = rdlane(y0, k), b1 = rdlane(y0, k + 1);
      const T b2 = rdlane(y0, k + 2), b3 = rdlane(y0, k + 3);
      const T z0 = b0;
      const T z1 = b1 - c.t10 * z0;
      const T z2 = (b2 - c.t2.x * z0) - c.t2.y * z1;
      const T z3 = ((b3 - c.t3.x * z0) - c.t3.y * z1) - c.t32 * z2;
      y0 = (((y0 - c.a.x * z0) - c.a.y * z1) - c.a.z * z2) - c.a.w * z3;
      y1 = (((y1 - c.b.x * z0) - c.b.y * z1) - c.b.z * z2) - c.b.w * z3;
    };
    load(0, A, true);
    for (int g = 0; g < gA; g += 2) {
      stepA(g, A, B);
      if (g + 1 < gA) stepA(g + 1, B, A);
    }
    // pivots in rows 64..127: only the second half updates
    auto stepB = [&](int g, const FwdStep<T>& c, FwdStep<T>& n) {
      const int k = 4 * g - 64;
      load(min(g + 1, ng - 1), n, false);
      const T b0 = rdlane(y1, k), b1 = rdlane(y1, k + 1);
      const T b2 = rdlane(y1, k + 2), b3 = rdlane(y1, k + 3);
      const T z0 = b0;
      const T z1 = b1 - c.t10 * z0;
      const T z2 = (b2 - c.t2.x * z0) - c.t2.y * z1;
      const T z3 = ((b3 - c.t3.x * z0) - c.t3.y * z1) - c.t32 * z2;
      y1 = (((y1 - c.b.x * z0) - c.b.y * z1) - c.b.z * z2) - c.b.w * z3;
    };
    if (ng > 16) {
      load(16, A, false);
      for (int g = 16; g < ng; g += 2) {
        stepB(g, A, B);
        if (g + 1 < ng) stepB(g + 1, B, A);
      }
    }
    if (in0) {
      yg[c0 + lane] = y0;
      x[fc0 + c0 + lane] = y0;
    }
    if (in1) {
      yg[c0 + 64 + lane] = y1;
      x[fc0 + c0 + 64 + lane] = y1;
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(kWG)
fwd_chain_kernel(DevSym s, const SolveDesc* __restrict__ desc, const T* __restrict__ prep,
                 const int32_t* __restrict__ prepi, T* __restrict__ rhs, int64_t ldr, int nrhs,
                 T* __restrict__ vec) {
  const int64_t vs = blockIdx.y;  // value set
  prep += vs * s.vs_prep;
  prepi += vs * s.vs_prepi;
  rhs += vs * ldr * nrhs;
  vec += vs * s.vs_vec * nrhs;
  extern __shared__ __attribute__((aligned(32))) unsigned char smem_a32[];
  fwd_chain_body<T>(s, desc[blockIdx.x], prep, prepi, rhs, ldr, nrhs, vec, smem_a32);
}

// Forward: y[c1 + r0 + lane] -= L[., c0:c1] y[c0:c1]; wave w takes a
// quarter of the block's columns, partial sums added in a fixed order. The
// block's column offsets and y[c0:c1] are staged in LDS first, then every
// thread issues all of its L loads at once.
template <typename T, int QB>
__device__ __attribute__((always_inline)) void fwd_bgemv_body(
    const DevSym& s, const SolveDesc& d, const T* __restrict__ lnz, int nrhs,
    T* __restrict__ vec) {
  __shared__ T red[4][QB][64];
  __shared__ int64_t lc[128];
  __shared__ __attribute__((aligned(16))) T zs[QB][4][32];  // a quarter's entries, zeros behind
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int L = d.L;
  const int64_t fc0 = d.fc0;
  const int c0 = d.c0, c1 = d.c1, bw = c1 - c0;
  const int r = c1 + d.r0 + lane;
  const int cb = bw * wave / 4, ce = bw * (wave + 1) / 4;  // at most 32 columns
  // (quarter, entry) this thread stages of a right-hand side's y[c0:c1]
  const int zw = tid % 128 / 32, zj = tid % 32;
  const int zc = bw * zw / 4 + zj;
  const bool zin = zc < bw * (zw + 1) / 4;
  if (tid < bw) lc[tid] = s.lcol[fc0 + c0 + tid];
  __syncthreads();
  // the block's entries of this tile's rows, read once for every rhs
  T lv[32];
#pragma unroll
  for (int j = 0; j < 32; ++j) lv[j] = (r < L && cb + j < ce) ? lnz[lc[cb + j] + r] : T(0);
  for (int q0 = 0; q0 < nrhs; q0 += QB) {
    const int nq = min(QB, nrhs - q0);
    T* yv = vec + d.fvec * nrhs + (int64_t)q0 * L;
    if constexpr (QB == 1) {
      if (tid < 128) zs[0][zw][zj] = zin ? yv[c0 + zc] : T(0);
    } else {
#pragma unroll
      for (int i = 0; i < QB / 2; ++i) {
        const int q = 2 * i + tid / 128;
        if (q < nq) zs[q][zw][zj] = zin ? yv[(int64_t)q * L + c0 + zc] : T(0);
      }
    }
    // wave w ends right-hand sides w, w + 4, ...: this tile's rows of their y
    // (no other workgroup touches them)
    T yr[(QB + 3) / 4];
#pragma unroll
    for (int i = 0; i < (QB + 3) / 4; ++i)
      yr[i] = (wave + 4 * i < nq && r < L) ? yv[(int64_t)(wave + 4 * i) * L + r] : T(0);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < QB; ++q) {
      if (q < nq) {
        T acc = T(0);
#pragma unroll
        for (int j = 0; j < 32; ++j) acc += lv[j] * zs[q][wave][j];
        red[wave][q][lane] = acc;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (QB + 3) / 4; ++i) {
      const int q = wave + 4 * i;
      if (q < nq && r < L)
        yv[(int64_t)q * L + r] =
            yr[i] - (((red[0][q][lane] + red[1][q][lane]) + red[2][q][lane]) + red[3][q][lane]);
    }
    __syncthreads();
  }
}

// QB right-hand sides share the reads of the block and three barriers. The
// block's y is read as whole vectors from LDS (its quarters padded to 32
// entries): single reads were what bounded the launch. 56 x 48 x 41, one
// right-hand side, double: 6.7 -> 5.5 us a launch; 32 sets of 32^3, 16
// right-hand sides: 39 -> 23 us (33 us with the shared barriers alone).
template <typename T, int QB>
__global__ void __launch_bounds__(kWG)
fwd_bgemv_kernel(DevSym s, const SolveDesc* __restrict__ desc, const T* __restrict__ lnz,
                 int nrhs, T* __restrict__ vec) {
  const int64_t vs = blockIdx.y;  // value set
  lnz += vs * s.vs_lnz;
  vec += vs * s.vs_vec * nrhs;
  fwd_bgemv_body<T, QB>(s, desc[blockIdx.x], lnz, nrhs, vec);
}

// One level of a sum over the wave's lanes, lane l with lane l ^ OFF, of two
// values at once: the lanes whose bit OFF is clear get a's sum, the others
// b's (a = b: all get a's).
template <int OFF>
__device__ inline unsigned lane_xor_mov(unsigned v) {  // OFF 8, 4, 2, 1
  const int x = (int)v;
  if constexpr (OFF == 8) return (unsigned)__builtin_amdgcn_update_dpp(x, x, 0x128, 0xf, 0xf, false);
  if constexpr (OFF == 4) {
    const int up = __builtin_amdgcn_update_dpp(x, x, 0x104, 0xf, 0x5, false);  // row_shl:4
    return (unsigned)__builtin_amdgcn_update_dpp(up, x, 0x114, 0xf, 0xa, false);  // row_shr:4
  }
  return (unsigned)__builtin_amdgcn_update_dpp(x, x, OFF == 2 ? 0x4E : 0xB1, 0xf, 0xf, false);
}
template <int OFF>
__device__ inline float lane_xor(float v) {
  return __uint_as_float(lane_xor_mov<OFF>(__float_as_uint(v)));
}
template <int OFF>
__device__ inline double lane_xor(double v) {
  const unsigned long long x = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = lane_xor_mov<OFF>((unsigned)x), hi = lane_xor_mov<OFF>((unsigned)(x >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// a and b with a's upper half-wave (OFF 32) or odd rows of 16 (OFF 16)
// exchanged for b's lower half-wave or even rows
template <int OFF>
__device__ inline void swap_lanes(unsigned& a, unsigned& b) {
  if constexpr (OFF == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0], b = r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0], b = r[1];
  }
}
template <int OFF>
__device__ inline float tree_step(float a, float b, bool up) {
  if constexpr (OFF >= 16) {
    unsigned x = __float_as_uint(a), y = __float_as_uint(b);
    swap_lanes<OFF>(x, y);
    return __uint_as_float(x) + __uint_as_float(y);
  } else {
    return (up ? b : a) + lane_xor<OFF>(up ? a : b);
  }
}
template <int OFF>
__device__ inline double tree_step(double a, double b, bool up) {
  if constexpr (OFF >= 16) {
    const unsigned long long p = (unsigned long long)__double_as_longlong(a);
    const unsigned long long q = (unsigned long long)__double_as_longlong(b);
    unsigned x0 = (unsigned)p, y0 = (unsigned)q, x1 = (unsigned)(p >> 32), y1 = (unsigned)(q >> 32);
    swap_lanes<OFF>(x0, y0);
    swap_lanes<OFF>(x1, y1);
    return __longlong_as_double((long long)(((unsigned long long)x1 << 32) | x0)) +
           __longlong_as_double((long long)(((unsigned long long)y1 << 32) | y0));
  } else {
    return (up ? b : a) + lane_xor<OFF>(up ? a : b);
  }
}
// Sums over the wave of NV values (a power of two, at most 64): lane l
// returns value l NV / 64's, added in the order of a tree over the lanes 32,
// 16, ..., 1 apart. The values halve as the lanes of each sum do, about two
// operations per value; six ds_bpermute each were most of the backward GEMV
// of many right-hand sides (16, 32 sets of 32^3: 12.2 ms a pass, now 8.5).
template <int NV, int OFF = 32, typename T>
__device__ __attribute__((always_inline)) inline T wave_sums(T (&v)[NV], int lane) {
  const bool up = (lane & OFF) != 0;
  if constexpr (NV == 1) {
    v[0] = tree_step<OFF>(v[0], v[0], up);
    if constexpr (OFF == 1)
      return v[0];
    else
      return wave_sums<1, OFF / 2>(v, lane);
  } else {
    T w[NV / 2];
#pragma unroll
    for (int i = 0; i < NV / 2; ++i) w[i] = tree_step<OFF>(v[i], v[i + NV / 2], up);
    if constexpr (OFF == 1)
      return w[0];
    else
      return wave_sums<NV / 2, OFF / 2>(w, lane);
  }
}

// Backward: t[c] = U[c, c1:L] x[c1:L] for rows c = c0 + r0 of the block,
// stored in y[c]. x[c1:L] is read from the front's vector: its update rows
// from bwd_gather_rows, its own columns as the backward chains of the
// later blocks left them. R rows of one block (n of them wanted) share the
// loads of x, QB right-hand sides those of U: every thread takes columns c1 +
// tid + 256 m of all of them, its sums are added over the wave (wave_sums),
// then the four waves in order; a (row, right-hand side) sum does not depend
// on R, QB or n.
template <typename T, int R, int QB>
__device__ __attribute__((always_inline)) void bwd_bgemv_body(
    const SolveDesc* __restrict__ dr, int n, const T* __restrict__ unz, int nrhs,
    T* __restrict__ vec) {
  // columns per thread and pass: about 32 loads of U in flight
  constexpr int CH = R == 1 ? 16 : R * (int)sizeof(T) > 32 ? 2 : 4;
  constexpr int NV = R * QB;
  __shared__ T red[4][NV];
  const int tid = threadIdx.x, lane = tid % 64, wave = wave_id();
  const SolveDesc d = dr[0];
  const int L = d.L, c1 = d.c1;
  T* const yv = vec + d.fvec * nrhs;
  const T* u[R];
#pragma unroll
  for (int i = 0; i < R; ++i) u[i] = unz + dr[R == 1 ? 0 : min(i, n - 1)].ucol;
  for (int q0 = 0; q0 < nrhs; q0 += QB) {
    const int nq = min(QB, nrhs - q0);
    T acc[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = T(0);
    for (int j0 = c1 + tid; j0 < L; j0 += CH * kWG) {
      T uv[R][CH];
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int t = 0; t < CH; ++t) {
          const int j = j0 + kWG * t;
          uv[i][t] = (j < L) ? u[i][j] : T(0);
        }
#pragma unroll
      for (int qq = 0; qq < QB; ++qq) {
        if (qq < nq) {
          const T* yg = yv + (int64_t)(q0 + qq) * L;
          T xv[CH];
#pragma unroll
          for (int t = 0; t < CH; ++t) {
            const int j = j0 + kWG * t;
            xv[t] = (j < L) ? yg[j] : T(0);
          }
#pragma unroll
          for (int i = 0; i < R; ++i)
#pragma unroll
            for (int t = 0; t < CH; ++t) acc[i * QB + qq] += uv[i][t] * xv[t];
        }
      }
    }
    const T sum = wave_sums<NV>(acc, lane);
    if (lane % (64 / NV) == 0) red[wave][lane / (64 / NV)] = sum;
    __syncthreads();
    if (tid < NV) {
      const int i = tid / QB, qq = tid % QB;
      if (i < n && qq < nq)
        yv[(int64_t)(q0 + qq) * L + dr[i].c0 + dr[i].r0] =
            ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
    }
    __syncthreads();
  }
}

// R consecutive row descriptors per workgroup, in runs of rows of one block
template <typename T, int R, int QB>
__global__ void __launch_bounds__(kWG)
bwd_bgemv_kernel(DevSym s, const SolveDesc* __restrict__ desc, int ndesc,
                 const T* __restrict__ unz, int nrhs, T* __restrict__ vec) {
  const int64_t vs = blockIdx.y;  // value set
  unz += vs * s.vs_unz;
  vec += vs * s.vs_vec * nrhs;
  const int end = min((int)blockIdx.x * R + R, ndesc);
  for (int i = (int)blockIdx.x * R; i < end;) {
    int n = 1;
    while (i + n < end && desc[i + n].front == desc[i].front && desc[i + n].c0 == desc[i].c0) ++n;
    bwd_bgemv_body<T, R, QB>(desc + i, n, unz, nrhs, vec);
    i += n;
  }
}

// b / u from r = 1 / u (correctly rounded): q0 = b r, then one correction
// with the exact remainder b - q0 u (an FMA) gives the correctly rounded
// quotient b / u, as the division itself (Markstein's theorem), in three
// dependent operations. Where r or the quotient overflows (u subnormal or
// infinite, b infinite or NaN) the result is NaN or infinite: solves of small
// fronts that end with such an entry are done again with the division itself
// (quot<true>).
__device__ inline double div_r(double b, double u, double r) {
  const double q0 = b * r;
  return __builtin_fma(__builtin_fma(-q0, u, b), r, q0);
}
__device__ inline float div_r(float b, float u, float r) {
  const float q0 = b * r;
  return __builtin_fmaf(__builtin_fmaf(-q0, u, b), r, q0);
}
template <bool DIV, typename T>
__device__ inline T quot(T b, T u, T r) {
  if constexpr (DIV)
    return b / u;
  else
    return div_r(b, u, r);
}

// Small fronts, solves. A front's right-hand sides are taken by one wave, QB
// at a time, lane = row, every right-hand side's vector in a register: column
// j's entry of each is broadcast (readlane) and every row below (forward) or
// above (backward) subtracts its product: from its entry inside the column's
// piece, from a sum that starts at zero outside it, which joins the entry where
// the piece ends (forward) or the row's own begins (backward). So a row's
// products are summed before they meet its entry, as the reference sums them
// (a product alone can be less than the entry's last place; subtracted one by
// one from the entry they cost 6 % in the error of 128 small systems). Chains
// of W (L) such steps bound them, taken piece by piece so that the sums cost
// nothing per column; the columns' factor entries are read ahead (forward: eight
// columns from lnz, whose rows are contiguous; backward: the front's U rows
// staged in LDS by columns). Each right-hand side receives the same
// operations in the same order however many there are. Fronts of more than
// 32 rows have a workgroup, whose four waves share the right-hand sides (and
// the staging), those of 17 to 32 one wave, smaller ones a part of a wave per
// right-hand side (fwd_tiny, bwd_tiny).
// Before, everything went through LDS with integer divisions by the panel's
// sizes and a wave synchronisation per column: forward + backward of one
// pass, 24 x 17 grid 240 -> 178 us, 193 x 171 680 -> 400 us, 128 small
// systems with four right-hand sides 1985 -> 951 us. The launches have since
// taken the large fronts' rows in as well (now 175, 455 and 1010 us).

// Entry j of a 64-bit value held one per lane (j wave-uniform).
__device__ inline int64_t rdlane_i64(int64_t v, int j) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, j);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), j);
  return (int64_t)(((unsigned long long)hi << 32) | lo);
}

// Forward, one wave: right-hand sides q0, q0 + 1, ..., q0 + QB - 1, then
// those qstep further on. y starts as the own rows of x and zero update
// rows and receives the children's update vectors in a fixed child order in
// LDS (Y, QB x 64); then per piece the interchanges (glaswp!) and per column
// the unit-lower step (gtrsm! 'l','l','n','u') and the rows below. The update
// rows go to the vector arena (the parent reads nothing else), the own rows
// to x.
template <typename T, int QB>
__device__ __attribute__((always_inline)) void fwd_small_wave(
    const DevSym& s, const SmallDesc& d, const SmallChild* __restrict__ child, int q0, int qstep,
    T* Y, const T* __restrict__ lnz, const int64_t* __restrict__ ipvt, T* __restrict__ rhs,
    int64_t ldr, int nrhs, T* __restrict__ vec) {
  constexpr int CH = 8;  // columns read ahead
  const int lane = threadIdx.x % 64;
  const int L = d.L, W = d.W;
  const int64_t fc0 = d.fc0;
  const bool own = lane < W;
  const int64_t lcb = own ? s.lcol[fc0 + lane] : 0;
  const int pcol = own ? s.pcol[fc0 + lane] : 0;  // the column's piece
  const int cq = pcol & 0xffff, ce = pcol >> 16;
  const int kp = own ? (int)ipvt[fc0 + lane] - 1 + cq : lane;
  // columns whose step interchanges rows
  const unsigned long long swaps = __ballot(own && kp != lane);
  for (; q0 < nrhs; q0 += qstep) {
    const int nq = min(QB, nrhs - q0);
    T y[QB];
#pragma unroll
    for (int q = 0; q < QB; ++q) {
      y[q] = T(0);
      if (q < nq && own) y[q] = rhs[(int64_t)(q0 + q) * ldr + fc0 + lane];
    }
    if (d.nch > 0) {
#pragma unroll
      for (int q = 0; q < QB; ++q) Y[q * 64 + lane] = y[q];
      wave_lds_sync();
      // the next child's entries are requested before this one's are added
      int rr = 0, rows = 0;
      T v[QB];
      auto request = [&](int ci) {
        const SmallChild c = child[d.ch0 + ci];
        rows = c.R;
        const T* uc = vec + c.fvec * nrhs + (int64_t)q0 * c.L + (c.L - c.R);
        rr = lane < rows ? s.relmap[c.rel + lane] : 0;
#pragma unroll
        for (int q = 0; q < QB; ++q)
          v[q] = (q < nq && lane < rows) ? uc[(int64_t)q * c.L + lane] : T(0);
      };
      request(0);
      for (int ci = 0; ci < d.nch; ++ci) {
        const int r0 = rr;
        const bool in = lane < rows;
        T w[QB];
#pragma unroll
        for (int q = 0; q < QB; ++q) w[q] = v[q];
        if (ci + 1 < d.nch) request(ci + 1);
        if (in) {
#pragma unroll
          for (int q = 0; q < QB; ++q) Y[q * 64 + r0] += w[q];
        }
        wave_lds_sync();
      }
#pragma unroll
      for (int q = 0; q < QB; ++q) y[q] = Y[q * 64 + lane];
      wave_lds_sync();
    }
    int pe = 0;  // the end of the piece at hand; rows from there on: summed
    T base[QB];  // ... from zero in y, their entry here (zero for the others)
#pragma unroll
    for (int q = 0; q < QB; ++q) base[q] = T(0);
    T lv[CH];
    auto columns = [&](int j0) {
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int j = j0 + u;
        const T* c = lnz + rdlane_i64(lcb, min(j, 63));
        lv[u] = (j < W && lane > j && lane < L) ? c[lane] : T(0);
      }
    };
    columns(0);
    for (int j0 = 0; j0 < W;) {
      if (j0 == pe) {  // a piece begins
#pragma unroll
        for (int q = 0; q < QB; ++q) y[q] = base[q] + y[q];
        pe = __builtin_amdgcn_readlane(ce, j0);
        unsigned long long m = swaps & (~0ull << j0) & (pe < 64 ? (1ull << pe) - 1 : ~0ull);
        while (m) {
          const int k = __ffsll((long long)m) - 1, p = __builtin_amdgcn_readlane(kp, k);
          m &= m - 1;
#pragma unroll
          for (int q = 0; q < QB; ++q) {
            const T a = rdlane(y[q], k), b = rdlane(y[q], p);
            y[q] = lane == k ? b : lane == p ? a : y[q];
          }
        }
#pragma unroll
        for (int q = 0; q < QB; ++q) {
          base[q] = lane >= pe ? y[q] : T(0);
          y[q] = lane >= pe ? T(0) : y[q];
        }
      }
      const int jn = min(j0 + CH, pe);  // the columns read ahead end with the piece
      T l[CH];
#pragma unroll
      for (int u = 0; u < CH; ++u) l[u] = lv[u];
      if (jn < W) columns(jn);
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int j = j0 + u;
        if (j >= jn) break;
#pragma unroll
        for (int q = 0; q < QB; ++q) {
          if (q < nq) {
            const T yk = rdlane(y[q], j);
            // inside the block a zero entry is skipped, as the reference does
            const bool on = lane > j && (yk != T(0) || lane >= pe);
            const T t = y[q] - l[u] * yk;
            y[q] = on ? t : y[q];
          }
        }
      }
      j0 = jn;
    }
#pragma unroll
    for (int q = 0; q < QB; ++q) y[q] = base[q] + y[q];
    T* yg = vec + d.fvec * nrhs + (int64_t)q0 * L + lane;
#pragma unroll
    for (int q = 0; q < QB; ++q) {
      if (q < nq) {
        if (own)
          rhs[(int64_t)(q0 + q) * ldr + fc0 + lane] = y[q];
        else if (lane < L)
          yg[(int64_t)q * L] = y[q];
      }
    }
  }
}

// Entry J of each group of SW = 8 or 16 lanes in all of its lanes (DPP
// row_newbcast, one VALU operation per 32 bits and row of 16; ds_bpermute,
// through the LDS pipeline, was what bounded the tiny fronts of many systems).
template <int SW, int J>
__device__ inline int bcast(int v) {
  if constexpr (SW == 16) return __builtin_amdgcn_update_dpp(v, v, 0x150 + J, 0xf, 0xf, false);
  const int lo = __builtin_amdgcn_update_dpp(v, v, 0x150 + J % 8, 0xf, 0x3, false);
  return __builtin_amdgcn_update_dpp(lo, v, 0x158 + J % 8, 0xf, 0xc, false);
}
template <int SW, int J>
__device__ inline float bcast(float v) {
  return __int_as_float(bcast<SW, J>(__float_as_int(v)));
}
template <int SW, int J>
__device__ inline int64_t bcast(int64_t v) {
  const unsigned lo = (unsigned)bcast<SW, J>((int)(unsigned)v);
  const unsigned hi = (unsigned)bcast<SW, J>((int)(v >> 32));
  return (int64_t)(((unsigned long long)hi << 32) | lo);
}
template <int SW, int J>
__device__ inline double bcast(double v) {
  return __longlong_as_double(bcast<SW, J>((int64_t)__double_as_longlong(v)));
}

// Fronts of at most SW = 8 or 16 rows: groups of SW lanes take one front
// and right-hand side each (64 / SW at once in a wave, unit u = front nrhs +
// right-hand side), all of the front's entries in registers. The same
// operations in the same order as fwd_small_wave / bwd_small_wave, which
// leave most lanes idle on such fronts (128 small systems, four right-hand
// sides: 1172 us a pass, now 951).
template <typename T, int SW>
__device__ __attribute__((always_inline)) void fwd_tiny(
    const DevSym& s, const SmallDesc* __restrict__ desc, const SmallChild* __restrict__ child,
    int64_t u, int cnt, T* Y, const T* __restrict__ lnz, const int64_t* __restrict__ ipvt,
    T* __restrict__ rhs, int64_t ldr, int nrhs, T* __restrict__ vec) {
  const int lane = threadIdx.x % 64, g0 = lane - lane % SW, r = lane % SW;
  // u is the wave's first unit; its quotient by nrhs is scalar
  const int64_t f0 = u / nrhs;
  const unsigned qg = (unsigned)(u - f0 * nrhs) + lane / SW, dq = qg / (unsigned)nrhs;
  const int64_t fi = f0 + dq;
  const int q = (int)(qg - dq * (unsigned)nrhs);
  const bool on = fi < cnt;  // a whole group
  const SmallDesc d = desc[on ? fi : 0];
  const int L = on ? d.L : 0, W = on ? d.W : 0;
  const int64_t fc0 = d.fc0;
  const bool own = r < W;
  const int64_t lcb = own ? s.lcol[fc0 + r] : 0;
  const int pcol = own ? s.pcol[fc0 + r] : 0;
  const int cq = pcol & 0xffff, ce = pcol >> 16;
  const int kp = own ? (int)ipvt[fc0 + r] - 1 + cq : r;
  const bool swaps = __ballot(kp != r) != 0;  // in any of the wave's fronts
  const bool multi = __ballot(cq != 0) != 0;  // ... more than one piece
  T y = own ? rhs[(int64_t)q * ldr + fc0 + r] : T(0);
  const int wm = -wave_min(-W);
  T l[SW];
  static_for<SW>([&](auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    l[j] = T(0);
    if (j < wm) {
      const T* c = lnz + bcast<SW, j>(lcb);
      if (j < W && r > j && r < L) l[j] = c[r];
    }
  });
  Y[lane] = y;
  wave_lds_sync();
  for (int ci = 0; ci < (on ? d.nch : 0); ++ci) {
    const SmallChild c = child[d.ch0 + ci];
    if (r < c.R) {
      const T v = vec[c.fvec * nrhs + (int64_t)q * c.L + (c.L - c.R) + r];
      Y[g0 + s.relmap[c.rel + r]] += v;
    }
    wave_lds_sync();
  }
  y = Y[lane];
  wave_lds_sync();
  // as in fwd_small_wave; one piece: the rows from W on throughout
  T base = (multi || r < W) ? T(0) : y;
  if (!multi && r >= W) y = T(0);
  static_for<SW>([&](auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    if (j < wm) {
      const int jce = bcast<SW, j>(ce);
      const bool begins = multi && j < W && bcast<SW, j>(cq) == j;
      if (multi) y = begins ? base + y : y;
      if (swaps) {  // a piece's interchanges before its first column
        Y[lane] = y;
        wave_lds_sync();
        if (r == j && j < W && cq == j)
          for (int k = j; k < ce; ++k) {
            const int p = (int)ipvt[fc0 + k] - 1 + cq;
            const T t = Y[g0 + k];
            Y[g0 + k] = Y[g0 + p];
            Y[g0 + p] = t;
          }
        wave_lds_sync();
        y = Y[lane];
        wave_lds_sync();
      }
      if (multi) {
        base = !begins ? base : r >= jce ? y : T(0);
        y = begins && r >= jce ? T(0) : y;
      }
      const T yk = bcast<SW, j>(y);
      const bool act = j < W && r > j && (yk != T(0) || r >= jce);
      const T t = y - l[j] * yk;
      y = act ? t : y;
    }
  });
  y = base + y;
  if (own)
    rhs[(int64_t)q * ldr + fc0 + r] = y;
  else if (r < L)
    vec[d.fvec * nrhs + (int64_t)q * L + r] = y;
}

template <typename T, int SW>
__device__ __attribute__((always_inline)) void bwd_tiny(
    const DevSym& s, const SmallDesc* __restrict__ desc, int64_t u, int cnt,
    const T* __restrict__ lnz, const T* __restrict__ unz, T* __restrict__ rhs, int64_t ldr,
    int nrhs) {
  const int lane = threadIdx.x % 64, r = lane % SW;
  // u is the wave's first unit; its quotient by nrhs is scalar
  const int64_t f0 = u / nrhs;
  const unsigned qg = (unsigned)(u - f0 * nrhs) + lane / SW, dq = qg / (unsigned)nrhs;
  const int64_t fi = f0 + dq;
  const int q = (int)(qg - dq * (unsigned)nrhs);
  const bool on = fi < cnt;
  const SmallDesc d = desc[on ? fi : 0];
  const int L = on ? d.L : 0, W = on ? d.W : 0;
  const int64_t fc0 = d.fc0;
  const bool own = r < W;
  const int64_t idx = r < L ? (int64_t)s.lindx[d.ind + r] - 1 : 0;
  // the row's entries: in its piece from lnz (columns L - cq apart), right of
  // it from unz
  const int pcol = own ? s.pcol[fc0 + r] : 0;
  const int cq = pcol & 0xffff, ce = pcol >> 16, ldp = L - cq;
  const bool multi = __ballot(cq != 0) != 0;  // more than one piece in any of the fronts
  const T* pl = lnz + (own ? s.lcol[fc0 + r] + r - (int64_t)r * ldp : 0);
  const T* pu = unz + (own ? s.ucol[fc0 + r] : 0);
  const int wm = -wave_min(-W), lm = -wave_min(-L);
  const T b = r < L ? rhs[(int64_t)q * ldr + idx] : T(0);
  T v[SW], dg = T(1);
  static_for<SW>([&](auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    v[j] = T(0);
    if (j < lm) {
      const T* p = j >= ce ? pu + j : pl + (int64_t)(j * ldp);
      if (own && j < L && j >= r) v[j] = *p;
      if (j == r && own) dg = v[j];
    }
  });
  const T ri = T(1) / dg;
  auto sweep = [&](auto div) __attribute__((always_inline)) {
    // a row's products right of its piece are summed from zero, its entry
    // joins them at the piece's last column
    T y = own ? T(0) : b;
    static_for<SW>([&](auto jc) __attribute__((always_inline)) {
      constexpr int j = SW - 1 - decltype(jc)::value;
      if (j < lm) {
        if (multi) {
          const int jcq = bcast<SW, j>(cq), jce = bcast<SW, j>(ce);
          if (j < W && jce == j + 1 && r >= jcq && r <= j) y = b + y;
        } else if (j < wm) {
          y = j == W - 1 && own ? b + y : y;
        }
        const T yk = bcast<SW, j>(y);
        if (j >= wm) {  // an update column of every front of the wave
          const T t = y - v[j] * yk;
          y = own && j < L ? t : y;
        } else {
          const T xk = bcast<SW, j>(quot<decltype(div)::value>(y, dg, ri));
          const T t = y - v[j] * (j >= W ? yk : xk);
          if (j >= W)
            y = own && j < L ? t : y;
          else
            y = yk == T(0) ? y : r < j ? t : r == j ? xk : y;
        }
      }
    });
    return y;
  };
  T y = sweep(std::false_type{});
  if (__builtin_expect(__ballot(own && !__builtin_isfinite(y)) != 0, 0))
    y = sweep(std::true_type{});
  if (own) rhs[(int64_t)q * ldr + fc0 + r] = y;
}

// More than four right-hand sides: lanes (q, g) of QL right-hand sides and G
// = 64 / QL rows, rows g + G i of the vectors in register i, the front's L or
// U columns staged in LDS. A column's entry of every right-hand side is
// broadcast at once (one ds_bpermute where the form above reads one lane per
// right-hand side) and a division serves them all. Fronts of at most 32 rows
// take one wave (16 x 4), larger ones a workgroup whose waves take four
// right-hand sides each (4 x 16). The operations of each right-hand side are
// those of the form above in its order. 32 sets of 32^3 with 16 right-hand
// sides, forward and backward of one pass: 9.2 ms with the form above, 6.6
// with this one (gathers of the scattered right-hand sides bound it now; 11.4
// ms with the large fronts' rows, which the launches have taken in since).
template <typename T>
__device__ inline T bperm(T v, int src) {
  return __shfl(v, src, 64);
}

template <typename T, int QL, int NR>
__device__ __attribute__((always_inline)) void fwd_small_many(
    const DevSym& s, const SmallDesc& d, const SmallChild* __restrict__ child, int q0, int qstep,
    const T* S, int LDL, T* X, const int64_t* __restrict__ ipvt, T* __restrict__ rhs, int64_t ldr,
    int nrhs, T* __restrict__ vec) {
  constexpr int G = 64 / QL;
  const int lane = threadIdx.x % 64, ql = lane % QL, g = lane / QL;
  const int L = d.L, W = d.W;
  const int64_t fc0 = d.fc0;
  const bool own = lane < W;
  const int pcol = own ? s.pcol[fc0 + lane] : 0;
  const int cq = pcol & 0xffff, ce = pcol >> 16;
  const int kp = own ? (int)ipvt[fc0 + lane] - 1 + cq : lane;
  const unsigned long long swaps = __ballot(own && kp != lane);
  for (; q0 < nrhs; q0 += qstep) {
    const int q = q0 + ql;
    const bool on = q < nrhs;
    T y[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int r = g + G * i;
      y[i] = (on && r < W) ? rhs[(int64_t)q * ldr + fc0 + r] : T(0);
    }
    if (d.nch > 0) {
#pragma unroll
      for (int i = 0; i < NR; ++i) X[(g + G * i) * QL + ql] = y[i];
      wave_lds_sync();
      for (int ci = 0; ci < d.nch; ++ci) {
        const SmallChild c = child[d.ch0 + ci];
        const T* uc = vec + c.fvec * nrhs + (int64_t)q * c.L + (c.L - c.R);
        T v[NR];
        int rr[NR];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
          const int t = g + G * i;
          const bool in = on && t < c.R;
          v[i] = in ? uc[t] : T(0);
          rr[i] = in ? s.relmap[c.rel + t] : 0;
        }
#pragma unroll
        for (int i = 0; i < NR; ++i)
          if (on && g + G * i < c.R) X[rr[i] * QL + ql] += v[i];
        wave_lds_sync();
      }
#pragma unroll
      for (int i = 0; i < NR; ++i) y[i] = X[(g + G * i) * QL + ql];
      wave_lds_sync();
    }
    int pe = 0;  // as in fwd_small_wave
    T base[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) base[i] = T(0);
    static_for<NR>([&](auto jc) __attribute__((always_inline)) {
      constexpr int jb = decltype(jc)::value;
      const int ge = min(G, W - G * jb);
#pragma unroll 1
      for (int gg = 0; gg < ge;) {
        if (G * jb + gg == pe) {  // a piece begins
          const int j = pe;
#pragma unroll
          for (int i = 0; i < NR; ++i) y[i] = base[i] + y[i];
          pe = __builtin_amdgcn_readlane(ce, j);
          unsigned long long m = swaps & (~0ull << j) & (pe < 64 ? (1ull << pe) - 1 : ~0ull);
          if (m) {
#pragma unroll
            for (int i = 0; i < NR; ++i) X[(g + G * i) * QL + ql] = y[i];
            wave_lds_sync();
            while (m) {
              const int k = __ffsll((long long)m) - 1, p = __builtin_amdgcn_readlane(kp, k);
              m &= m - 1;
              if (g == 0) {
                const T t = X[k * QL + ql];
                X[k * QL + ql] = X[p * QL + ql];
                X[p * QL + ql] = t;
              }
              wave_lds_sync();
            }
#pragma unroll
            for (int i = 0; i < NR; ++i) y[i] = X[(g + G * i) * QL + ql];
            wave_lds_sync();
          }
#pragma unroll
          for (int i = 0; i < NR; ++i) {
            const bool below = g + G * i >= pe;
            base[i] = below ? y[i] : T(0);
            y[i] = below ? T(0) : y[i];
          }
        }
        const int gp = min(ge, pe - G * jb);
#pragma unroll 1
        for (; gg < gp; ++gg) {
          const int j = G * jb + gg;
          T l[NR];
#pragma unroll
          for (int i = jb; i < NR; ++i) l[i] = S[j * LDL + min(g + G * i, L - 1)];
          const T yk = bperm(y[jb], gg * QL + ql);
#pragma unroll
          for (int i = jb; i < NR; ++i) {
            const int r = g + G * i;
            const T t = y[i] - l[i] * yk;
            y[i] = (r > j && r < L && (yk != T(0) || r >= pe)) ? t : y[i];
          }
        }
      }
    });
#pragma unroll
    for (int i = 0; i < NR; ++i) y[i] = base[i] + y[i];
    T* yg = vec + d.fvec * nrhs + (int64_t)q * L;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int r = g + G * i;
      if (on && r < W)
        rhs[(int64_t)q * ldr + fc0 + r] = y[i];
      else if (on && r < L)
        yg[r] = y[i];
    }
  }
}

template <typename T, int QL, int NR>
__device__ __attribute__((always_inline)) void bwd_small_many(
    const DevSym& s, const SmallDesc& d, int q0, int qstep, const T* S, int LDW,
    T* __restrict__ rhs, int64_t ldr, int nrhs) {
  constexpr int G = 64 / QL;
  const int lane = threadIdx.x % 64, ql = lane % QL, g = lane / QL;
  const int L = d.L, W = d.W;
  const T dg = lane < W ? S[lane * LDW + lane] : T(1);
  const T ri = T(1) / dg;
  const int cq = lane < W ? s.pcol[d.fc0 + lane] & 0xffff : 0;
  for (; q0 < nrhs; q0 += qstep) {
    const int q = q0 + ql;
    const bool on = q < nrhs;
    T y[NR];
    auto sweep = [&](auto div) __attribute__((always_inline)) {
      // as in bwd_small_wave, the own rows' entries read when their piece's
      // columns come (kept in registers they cost a sixth of the waves in flight)
      int pa = W;
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int r = g + G * i;
        y[i] = (on && r >= W && r < L) ? rhs[(int64_t)q * ldr + s.lindx[d.ind + r] - 1] : T(0);
      }
      T u[NR], c[NR];  // the column's rows, read one column ahead
      auto column = [&](int j) {
#pragma unroll
        for (int i = 0; i < NR; ++i)
          u[i] = G * i < W ? S[max(j, 0) * LDW + min(g + G * i, W - 1)] : T(0);
      };
      column(L - 1);
      static_for<NR>([&](auto jc) __attribute__((always_inline)) {
        constexpr int jb = NR - 1 - decltype(jc)::value;
        int gg = min(G, L - G * jb) - 1;
        auto step = [&]() {
          const T yk = bperm(y[jb], gg * QL + ql);
#pragma unroll
          for (int i = 0; i <= jb; ++i) c[i] = u[i];
          column(G * jb + gg - 1);
          return yk;
        };
#pragma unroll 1
        for (; gg >= max(W - G * jb, 0); --gg) {  // update columns
          const T yk = step();
#pragma unroll
          for (int i = 0; i <= jb; ++i) {
            const T t = y[i] - c[i] * yk;
            y[i] = g + G * i < W ? t : y[i];
          }
        }
#pragma unroll 1
        while (gg >= 0) {  // own columns, piece by piece
          if (G * jb + gg == pa - 1) {
            const int pe = pa;
            pa = __builtin_amdgcn_readlane(cq, pe - 1);
#pragma unroll
            for (int i = 0; i <= jb; ++i) {
              const int r = g + G * i;
              if (on && r >= pa && r < pe) y[i] = rhs[(int64_t)q * ldr + d.fc0 + r] + y[i];
            }
          }
          const int gl = max(pa - G * jb, 0);
#pragma unroll 1
          for (; gg >= gl; --gg) {
            const int j = G * jb + gg;
            const T yk = step();
            const T xk = quot<decltype(div)::value>(yk, rdlane(dg, j), rdlane(ri, j));
            const bool nz = yk != T(0);  // a zero entry stays, as in the reference
#pragma unroll
            for (int i = 0; i <= jb; ++i) {
              const int r = g + G * i;
              const T t = y[i] - c[i] * xk;
              y[i] = nz && r < j ? t : nz && r == j ? xk : y[i];
            }
          }
        }
      });
      bool finite = true;
#pragma unroll
      for (int i = 0; i < NR; ++i) finite = finite && (g + G * i >= W || __builtin_isfinite(y[i]));
      return __ballot(!finite) == 0;
    };
    if (__builtin_expect(!sweep(std::false_type{}), 0)) sweep(std::true_type{});
#pragma unroll
    for (int i = 0; i < NR; ++i)
      if (on && g + G * i < W) rhs[(int64_t)q * ldr + d.fc0 + g + G * i] = y[i];
  }
}

// The front's L columns in LDS, S[j LDL + r] for r > j, by G threads.
template <typename T, int G>
__device__ __attribute__((always_inline)) void stage_small_l(const DevSym& s, const SmallDesc& d,
                                                             T* S, int LDL,
                                                             const T* __restrict__ lnz) {
  constexpr int NW = G / 64, CH = 8;
  const int lane = threadIdx.x % 64;
  const int w = G == kWG ? wave_id() : 0;
  const int64_t lcb = lane < d.W ? s.lcol[d.fc0 + lane] : 0;
  for (int i0 = w * CH; i0 < d.W; i0 += NW * CH) {
    T a[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int i = min(i0 + u, 63);
      const T* l = lnz + rdlane_i64(lcb, i);
      a[u] = (i0 + u < d.W && lane > i && lane < d.L) ? l[lane] : T(0);
    }
#pragma unroll
    for (int u = 0; u < CH; ++u)
      if (i0 + u < d.W && lane < d.L) S[(i0 + u) * LDL + lane] = a[u];
  }
}

template <typename T, int QW>
__global__ void __launch_bounds__(kWG)
fwd_small_kernel(DevSym s, const SmallDesc* __restrict__ desc,
                 const SmallChild* __restrict__ child, SmallClasses k, LevelRows m, int LDL, int slot,
                 const T* __restrict__ lnz, const int64_t* __restrict__ ipvt,
                 T* __restrict__ rhs, int64_t ldr, int nrhs, T* __restrict__ vec) {
  const int64_t vs = blockIdx.y;  // value set
  int b = blockIdx.x;
  lnz += vs * s.vs_lnz;
  ipvt += vs * s.n;
  rhs += vs * ldr * nrhs;
  vec += vs * s.vs_vec * nrhs;
  if (b >= k.wgs) {
    fwd_assemble_rows<T>(s, m, b - k.wgs, rhs, ldr, nrhs, vec);
    return;
  }
  const int wave = wave_id();
  if constexpr (QW > 4) {
    extern __shared__ unsigned char smem_raw[];
    T* S = reinterpret_cast<T*>(smem_raw);
    __shared__ T X[4][512];
    if (b < k.cnt[0]) {
      const SmallDesc d = desc[b];
      stage_small_l<T, kWG>(s, d, S, LDL, lnz);
      __syncthreads();
      fwd_small_many<T, 4, 4>(s, d, child, wave * 4, 16, S, LDL, X[wave], ipvt, rhs, ldr, nrhs,
                              vec);
      return;
    }
    const int item = (b - k.cnt[0]) * 4 + wave;
    if (item >= k.cnt[1]) return;
    const SmallDesc d = desc[k.cnt[0] + item];
    S += wave * slot;
    LDL = min(LDL, 33);
    stage_small_l<T, 64>(s, d, S, LDL, lnz);
    wave_lds_sync();
    fwd_small_many<T, 16, 8>(s, d, child, 0, 16, S, LDL, X[wave], ipvt, rhs, ldr, nrhs, vec);
  } else {
    __shared__ T Y[4][QW * 64];
    if (b < k.cnt[0]) {
      fwd_small_wave<T, 1>(s, desc[b], child, wave, 4, Y[wave], lnz, ipvt, rhs, ldr, nrhs, vec);
      return;
    }
    b -= k.cnt[0];
    desc += k.cnt[0];
    if (b < k.wg1) {
      const int item = b * 4 + wave;
      if (item < k.cnt[1])
        fwd_small_wave<T, QW>(s, desc[item], child, 0, QW, Y[wave], lnz, ipvt, rhs, ldr, nrhs, vec);
      return;
    }
    b -= k.wg1;
    desc += k.cnt[1];
    if (b < k.wg2) {
      fwd_tiny<T, 16>(s, desc, child, ((int64_t)b * 4 + wave) * 4, k.cnt[2], Y[wave], lnz, ipvt, rhs, ldr,
                      nrhs, vec);
      return;
    }
    b -= k.wg2;
    desc += k.cnt[2];
    fwd_tiny<T, 8>(s, desc, child, ((int64_t)b * 4 + wave) * 8, k.cnt[3], Y[wave], lnz, ipvt, rhs, ldr, nrhs,
                   vec);
  }
}

// The front's U rows by columns in LDS, S[j LDW + c] = U(c, j) for c <= j:
// the pieces' blocks from the packed LU in lnz (rows contiguous), the
// columns right of them from unz (columns contiguous), by G threads.
template <typename T, int G>
__device__ __attribute__((always_inline)) void stage_small_u(
    const DevSym& s, const SmallDesc& d, T* S, int LDW, const T* __restrict__ lnz,
    const T* __restrict__ unz) {
  constexpr int NW = G / 64, CH = 8;
  const int lane = threadIdx.x % 64;
  const int w = G == kWG ? wave_id() : 0;
  const int L = d.L, W = d.W;
  const int64_t fc0 = d.fc0;
  const bool own = lane < W;
  const int64_t lcb = own ? s.lcol[fc0 + lane] : 0;
  const int64_t ucb = own ? s.ucol[fc0 + lane] : 0;
  const int pcol = own ? s.pcol[fc0 + lane] : 0;
  for (int i0 = w * CH; i0 < W; i0 += NW * CH) {
    T a[CH], b[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int i = min(i0 + u, 63);
      const bool on = i0 + u < W;
      const int pc = __builtin_amdgcn_readlane(pcol, i);
      const T* l = lnz + rdlane_i64(lcb, i);  // column i, lane = row
      const T* r = unz + rdlane_i64(ucb, i);  // row i, lane = column
      a[u] = (on && lane >= (pc & 0xffff) && lane <= i) ? l[lane] : T(0);
      b[u] = (on && lane >= (pc >> 16) && lane < L) ? r[lane] : T(0);
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int i = min(i0 + u, 63);
      const bool on = i0 + u < W;
      const int pc = __builtin_amdgcn_readlane(pcol, i);
      if (on && lane >= (pc & 0xffff) && lane <= i) S[i * LDW + lane] = a[u];
      if (on && lane >= (pc >> 16) && lane < L) S[lane * LDW + i] = b[u];
    }
  }
}

// Backward, one wave (right-hand sides as in fwd_small_wave): x gathered
// through the index list, then the columns last to first: an own column's
// entry is divided by U(j, j) and the rows above subtract their products
// (gtrsm! 'l','u','n','n' and the U12 products by columns).
template <typename T, int QB>
__device__ __attribute__((always_inline)) void bwd_small_wave(
    const DevSym& s, const SmallDesc& d, int q0, int qstep, const T* S, int LDW,
    T* __restrict__ rhs, int64_t ldr, int nrhs) {
  const int lane = threadIdx.x % 64;
  const int L = d.L, W = d.W;
  const bool own = lane < W;
  const int64_t idx = lane < L ? (int64_t)s.lindx[d.ind + lane] - 1 : 0;
  const T dg = own ? S[lane * LDW + lane] : T(1);
  const T ri = T(1) / dg;
  const int cl = min(lane, W - 1);
  const int cq = own ? s.pcol[d.fc0 + lane] & 0xffff : 0;
  for (; q0 < nrhs; q0 += qstep) {
    const int nq = min(QB, nrhs - q0);
    T y[QB];
    auto sweep = [&](auto div) __attribute__((always_inline)) {
      // own rows are summed from zero in y until their piece's columns come,
      // their entry in base
      T base[QB];
#pragma unroll
      for (int q = 0; q < QB; ++q) {
        const T b = (q < nq && lane < L) ? rhs[(int64_t)(q0 + q) * ldr + idx] : T(0);
        base[q] = b;
        y[q] = own ? T(0) : b;
      }
      constexpr int CH = 4;  // columns read ahead
      T sv[CH];
      auto columns = [&](int j0) {
#pragma unroll
        for (int u = 0; u < CH; ++u) sv[u] = S[max(j0 - u, 0) * LDW + cl];
      };
      columns(L - 1);
      // the columns read ahead end at jn, where a piece begins at the latest
      T c[CH];
      auto next = [&](int jn) {
#pragma unroll
        for (int u = 0; u < CH; ++u) c[u] = sv[u];
        if (jn >= 0) columns(jn);
      };
      int j0 = L - 1;
      while (j0 >= W) {  // update columns
        const int jn = max(j0 - CH, W - 1);
        next(jn);
#pragma unroll
        for (int u = 0; u < CH; ++u) {
          if (j0 - u <= jn) break;
#pragma unroll
          for (int q = 0; q < QB; ++q)
            if (q < nq) {
              const T xk = rdlane(y[q], j0 - u);
              const T t = y[q] - c[u] * xk;
              y[q] = own ? t : y[q];
            }
        }
        j0 = jn;
      }
      int pa = W;  // own columns: the piece at hand begins at pa
      while (j0 >= 0) {
        if (j0 == pa - 1) {
          const int pe = pa;
          pa = __builtin_amdgcn_readlane(cq, j0);
          const bool in = lane >= pa && lane < pe;
#pragma unroll
          for (int q = 0; q < QB; ++q) y[q] = in ? base[q] + y[q] : y[q];
        }
        const int jn = max(j0 - CH, pa - 1);
        next(jn);
#pragma unroll
        for (int u = 0; u < CH; ++u) {
          const int j = j0 - u;
          if (j <= jn) break;
#pragma unroll
          for (int q = 0; q < QB; ++q)
            if (q < nq) {
              const T xq = quot<decltype(div)::value>(y[q], dg, ri);
              const T yk = rdlane(y[q], j), xk = rdlane(xq, j);
              if (yk != T(0)) {  // a zero entry stays, as in the reference
                const T t = y[q] - c[u] * xk;
                y[q] = lane < j ? t : lane == j ? xk : y[q];
              }
            }
        }
        j0 = jn;
      }
      bool finite = true;
#pragma unroll
      for (int q = 0; q < QB; ++q) finite = finite && __builtin_isfinite(y[q]);
      return __ballot(own && !finite) == 0;
    };
    if (__builtin_expect(!sweep(std::false_type{}), 0)) sweep(std::true_type{});
#pragma unroll
    for (int q = 0; q < QB; ++q)
      if (q < nq && own) rhs[(int64_t)(q0 + q) * ldr + d.fc0 + lane] = y[q];
  }
}

template <typename T, int QW>
__global__ void __launch_bounds__(kWG)
bwd_small_kernel(DevSym s, const SmallDesc* __restrict__ desc, SmallClasses k, LevelRows m,
                 int LDW, int slot, const T* __restrict__ lnz, const T* __restrict__ unz,
                 T* __restrict__ rhs, int64_t ldr, int nrhs, T* __restrict__ vec) {
  const int64_t vs = blockIdx.y;  // value set
  int b = blockIdx.x;
  lnz += vs * s.vs_lnz;
  unz += vs * s.vs_unz;
  rhs += vs * ldr * nrhs;
  if (b >= k.wgs) {
    bwd_gather_rows<T>(s, m, b - k.wgs, rhs, ldr, nrhs, vec + vs * s.vs_vec * nrhs);
    return;
  }
  extern __shared__ unsigned char smem_raw[];
  T* S = reinterpret_cast<T*>(smem_raw);
  const int wave = wave_id();
  if (b < k.cnt[0]) {
    const SmallDesc d = desc[b];
    stage_small_u<T, kWG>(s, d, S, LDW, lnz, unz);
    __syncthreads();
    if constexpr (QW > 4)
      bwd_small_many<T, 4, 4>(s, d, wave * 4, 16, S, LDW, rhs, ldr, nrhs);
    else
      bwd_small_wave<T, 1>(s, d, wave, 4, S, LDW, rhs, ldr, nrhs);
    return;
  }
  b -= k.cnt[0];
  desc += k.cnt[0];
  if (b < k.wg1) {
    const int item = b * 4 + wave;
    if (item >= k.cnt[1]) return;
    const SmallDesc d = desc[item];
    S += wave * slot;
    LDW = min(LDW, 33);
    stage_small_u<T, 64>(s, d, S, LDW, lnz, unz);
    wave_lds_sync();
    if constexpr (QW > 4)
      bwd_small_many<T, 16, 8>(s, d, 0, 16, S, LDW, rhs, ldr, nrhs);
    else
      bwd_small_wave<T, QW>(s, d, 0, QW, S, LDW, rhs, ldr, nrhs);
    return;
  }
  if constexpr (QW <= 4) {
    b -= k.wg1;
    desc += k.cnt[1];
    if (b < k.wg2) {
      bwd_tiny<T, 16>(s, desc, ((int64_t)b * 4 + wave) * 4, k.cnt[2], lnz, unz, rhs, ldr, nrhs);
      return;
    }
    b -= k.wg2;
    desc += k.cnt[2];
    bwd_tiny<T, 8>(s, desc, ((int64_t)b * 4 + wave) * 8, k.cnt[3], lnz, unz, rhs, ldr, nrhs);
  }
}

// Backward chain of one block. The block's upper panels and diagonal
// reciprocals come from the solve data in one coalesced load. With t =
// U[c0:c1, c1:L] x[c1:L] already in the vector arena (bwd_bgemv_kernel),
// wave 0 holds y = x - t in registers and back-substitutes, last column
// first, four columns per step: the four new entries x_k = (y_k - ...) /
// U(k, k) every lane computes alike, then each earlier row takes its four
// products in column order — the in-block U12 products and the upper block
// solves of the reference, by columns. The next step's panel values are
// read from LDS while the current step computes.
template <typename T>
struct BwdStep {
  typename Vec4<T>::type d0, ri, a, b;  // U(k, k:k+4), 1 / U(j, j), the lane's rows
  typename Vec4<T>::half d1, d2;        // U(k+1, k+2:k+4), U(k+2, k+2:k+4)
  T d11, d33;                           // U(k+1, k+1), U(k+3, k+3)
};

template <typename T>
__device__ __attribute__((always_inline)) void bwd_chain_body(
    const DevSym& s, const SolveDesc& d, const T* __restrict__ prep, T* __restrict__ rhs,
    int64_t ldr, int nrhs, T* __restrict__ vec, unsigned char* smem_a32) {
  using V = typename Vec4<T>::type;
  V* smem_v4 = reinterpret_cast<V*>(smem_a32);
  const T* R = reinterpret_cast<const T*>(smem_a32);
  const int tid = threadIdx.x, lane = tid % 64;
  // wave w takes right-hand sides w, w + 4, ..., spread over the z workgroups
  const int wave = wave_id() + 4 * (int)blockIdx.z, qstep = 4 * (int)gridDim.z;
  const int f = d.front;
  const int L = d.L;
  const int64_t fc0 = d.fc0;
  const int c0 = d.c0, c1 = d.c1, bw = c1 - c0;
  const int ng = (bw + 3) / 4;
  const bool in0 = lane < bw, in1 = lane + 64 < bw, sub = c1 < L;
  T x0r = T(0), x1r = T(0), t0r = T(0), t1r = T(0);
  // wave w takes right-hand sides w, w + 4, ...; its first one in flight
  // with the panels
  if (wave < nrhs) {
    const T* x = rhs + (int64_t)wave * ldr + fc0 + c0;
    const T* yg = vec + d.fvec * nrhs + (int64_t)wave * L + c0;
    if (in0) {
      x0r = x[lane];
      if (sub) t0r = yg[lane];
    }
    if (in1) {
      x1r = x[lane + 64];
      if (sub) t1r = yg[lane + 64];
    }
  }
  const int npan = 8 * ng * (ng + 1);
  load_panels(reinterpret_cast<const V*>(prep + 4 * (int64_t)d.aux + npan), smem_v4,
              2 * ng * (ng + 1) + ng);
  __syncthreads();
  if (wave >= nrhs) return;
  const T* Rinv = R + npan;
  const int gA = min(ng, 16);
  auto load = [&](int g, BwdStep<T>& o, bool both) {
    const int k = 4 * g;
    const T* P = R + up_panel(g);
    using H = typename Vec4<T>::half;
    o.d0 = *(const V*)(P + 4 * k);
    o.d11 = P[4 * k + 5];
    o.d1 = *(const H*)(P + 4 * k + 6);
    o.d2 = *(const H*)(P + 4 * k + 10);
    o.d33 = P[4 * k + 15];
    o.ri = *(const V*)(Rinv + k);
    o.a = *(const V*)(P + 4 * min(lane, k + 3));
    if (both) o.b = *(const V*)(P + 4 * min(lane + 64, k + 3));
  };
  for (int q = wave; q < nrhs; q += qstep) {
    T* yg = vec + d.fvec * nrhs + (int64_t)q * L;
    T* x = rhs + (int64_t)q * ldr;
    if (q > wave) {
      x0r = in0 ? x[fc0 + c0 + lane] : T(0);
      x1r = in1 ? x[fc0 + c0 + 64 + lane] : T(0);
      t0r = (in0 && sub) ? yg[c0 + lane] : T(0);
      t1r = (in1 && sub) ? yg[c0 + 64 + lane] : T(0);
    }
    T y0 = in0 ? x0r - t0r : T(0);
    T y1 = in1 ? x1r - t1r : T(0);
    BwdStep<T> A, B;
    // the step's four new entries from its pivot values b0..b3
    auto solve4 = [&](const BwdStep<T>& c, T b0, T b1, T b2, T b3, T& x0, T& x1, T& x2,
                      T& x3) {
      x3 = div_r(b3, c.d33, c.ri.w);
      x2 = div_r(b2 - c.d2.y * x3, c.d2.x, c.ri.z);
      x1 = div_r((b1 - c.d1.y * x3) - c.d1.x * x2, c.d11, c.ri.y);
      x0 = div_r(((b0 - c.d0.w * x3) - c.d0.z * x2) - c.d0.y * x1, c.d0.x, c.ri.x);
    };
    // row update of y at offset dl from the step's first column: rows above
    // take the four products, the step's rows their new entries
    auto upd = [&](T y, const V& a, int dl, T x0, T x1, T x2, T x3) {
      T r = pin((((y - a.w * x3) - a.z * x2) - a.y * x1) - a.x * x0);
      r = (dl == 0) ? x0 : r;
      r = (dl == 1) ? x1 : r;
      r = (dl == 2) ? x2 : r;
      r = (dl == 3) ? x3 : r;
      r = (dl >= 4) ? y : r;
      return r;
    };
    // pivots in rows 64..127: every row of the first half updates
    auto stepB = [&](int g, const BwdStep<T>& c, BwdStep<T>& n) {
      const int k = 4 * g;
      load(max(g - 1, 0), n, true);
      T x0, x1, x2, x3;
      solve4(c, rdlane(y1, k - 64), rdlane(y1, k - 63), rdlane(y1, k - 62), rdlane(y1, k - 61),
             x0, x1, x2, x3);
      y0 = (((y0 - c.a.w * x3) - c.a.z * x2) - c.a.y * x1) - c.a.x * x0;
      y1 = upd(y1, c.b, lane + 64 - k, x0, x1, x2, x3);
    };
    if (ng > 16) {
      load(ng - 1, A, true);
      for (int g = ng - 1; g >= 16; g -= 2) {
        stepB(g, A, B);
        if (g - 1 >= 16) stepB(g - 1, B, A);
      }
    }
    // pivots in rows 0..63: only the first half updates
    auto stepA = [&](int g, const BwdStep<T>& c, BwdStep<T>& n) {
      const int k = 4 * g;
      load(max(g - 1, 0), n, false);
      T x0, x1, x2, x3;
      solve4(c, rdlane(y0, k), rdlane(y0, k + 1), rdlane(y0, k + 2), rdlane(y0, k + 3), x0, x1,
             x2, x3);
      y0 = upd(y0, c.a, lane - k, x0, x1, x2, x3);
    };
    load(gA - 1, A, false);
    for (int g = gA - 1; g >= 0; g -= 2) {
      stepA(g, A, B);
      if (g - 1 >= 0) stepA(g - 1, B, A);
    }
    if (in0) {
      x[fc0 + c0 + lane] = y0;
      yg[c0 + lane] = y0;
    }
    if (in1) {
      x[fc0 + c0 + 64 + lane] = y1;
      yg[c0 + 64 + lane] = y1;
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(kWG)
bwd_chain_kernel(DevSym s, const SolveDesc* __restrict__ desc, const T* __restrict__ prep,
                 T* __restrict__ rhs, int64_t ldr, int nrhs, T* __restrict__ vec) {
  const int64_t vs = blockIdx.y;  // value set
  prep += vs * s.vs_prep;
  rhs += vs * ldr * nrhs;
  vec += vs * s.vs_vec * nrhs;
  extern __shared__ __attribute__((aligned(32))) unsigned char smem_a32[];
  bwd_chain_body<T>(s, desc[blockIdx.x], prep, rhs, ldr, nrhs, vec, smem_a32);
}

// ---------------------------------------------------------------------------
// Float solves with explicit inverses of the diagonal blocks. The chains are
// the solves' serial critical path (one column group after another); with
// ML = L11^-1 P and MU = U11^-1 formed once per factorisation, every block
// step becomes GEMV work that all workgroups of the step do in parallel, one
// launch per step instead of a chain launch and a GEMV launch. (The double
// factor keeps substitution, the reference's operation order.)
// ---------------------------------------------------------------------------

// ML and MU of one block (one workgroup per block), each bwp x bwp
// row-major and zero outside bw x bw. Column j of each inverse is the solve
// of e_j: threads 0..127 take ML's columns (column jj of ML is the solve of
// e_i, i the row that the interchanges bring to jj), threads 128..255 MU's,
// 32 rows at a time in registers: the terms of the rows already solved, read
// back from the output, then the 32 x 32 triangle, the panels read from LDS
// as broadcasts (four coefficients of a row at a time). Column j's entries
// receive the terms of c = j, j + 1, ... (ML) or c = j, j - 1, ... (MU) in
// that order; the others would meet a zero and are left out. Bound by about
// 8000 dependent-free products per thread; with the panels read from global
// memory and one workgroup barrier per eliminated column it took 700 us on
// the blocks of 31 x 23 x 17, now 73 us (64^3: 1240 -> 198 us).
constexpr int kInvPrepLds = (2 * kPanelElems + 128) * 4;  // float
__global__ void __launch_bounds__(kWG)
solve_inv_prep_kernel(const SolveDesc* __restrict__ desc, const float* __restrict__ prep,
                      const int32_t* __restrict__ prepi, float* __restrict__ inv,
                      int64_t vs_prep, int64_t vs_prepi, int64_t vs_inv) {
  const int64_t vs = blockIdx.y;  // value set
  prep += vs * vs_prep;
  prepi += vs * vs_prepi;
  inv += vs * vs_inv;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_inv[];
  float* lo = reinterpret_cast<float*>(smem_inv);
  float* up = lo + kPanelElems;
  float* rinv = up + kPanelElems;
  __shared__ int iperm[128];
  const SolveDesc d = desc[blockIdx.x];
  const int bw = d.c1 - d.c0, ng = (bw + 3) / 4, bwp = 4 * ng;
  const int tid = threadIdx.x;
  const int npan = 8 * ng * (ng + 1);
  {
    const f32x4* g = reinterpret_cast<const f32x4*>(prep + 4 * (int64_t)d.aux);
    for (int i = tid; i < npan / 4; i += kWG) {
      reinterpret_cast<f32x4*>(lo)[i] = g[i];
      reinterpret_cast<f32x4*>(up)[i] = g[npan / 4 + i];
    }
    if (tid < ng) reinterpret_cast<f32x4*>(rinv)[tid] = g[npan / 2 + tid];
  }
  const int32_t* pi = prepi + (int64_t)d.r0 * kPrepInts;
  if (tid < bw) iperm[pi[tid]] = tid;
  __syncthreads();
  float* ML = inv + d.inv;
  const int jj = tid & 127;
  if (jj >= bwp) return;
  if (tid < 128) {
    const int j = jj < bw ? iperm[jj] : 1 << 20;
    float* X = ML + jj;
    for (int r0 = 0; r0 < bwp; r0 += 32) {
      float x[32];
#pragma unroll
      for (int r = 0; r < 32; ++r) x[r] = r0 + r == j ? 1.0f : 0.0f;
      for (int c = 0; c < r0; c += 4) {
        float xc[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) xc[k] = X[(c + k) * bwp];
        const float* P = lo + lo_panel(c / 4, ng) + 4 * (r0 - c);
#pragma unroll
        for (int rr = 0; rr < 32; rr += 8) {
          f32x4 p[8];
#pragma unroll
          for (int r = 0; r < 8; ++r) p[r] = *reinterpret_cast<const f32x4*>(P + 4 * (rr + r));
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (c + k >= j) {
#pragma unroll
              for (int r = 0; r < 8; ++r) x[rr + r] -= p[r][k] * xc[k];
            }
        }
      }
      static_for<8>([&](auto gc) __attribute__((always_inline)) {
        constexpr int c = 4 * decltype(gc)::value;
        const float* P = lo + lo_panel((r0 + c) / 4, ng) - 4 * c;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (r0 + c < bwp && r0 + c + k >= j) {
#pragma unroll
            for (int r = c + k + 1; r < 32; ++r) x[r] -= P[4 * r + k] * x[c + k];
          }
      });
#pragma unroll
      for (int r = 0; r < 32; ++r)
        if (r0 + r < bwp) X[(r0 + r) * bwp] = r0 + r < bw ? x[r] : 0.0f;
    }
  } else {
    const int j = jj < bw ? jj : -1;
    float* X = ML + (int64_t)bwp * bwp + jj;
    for (int r0 = (bwp - 1) / 32 * 32; r0 >= 0; r0 -= 32) {
      float x[32];
#pragma unroll
      for (int r = 0; r < 32; ++r) x[r] = r0 + r == j ? 1.0f : 0.0f;
      for (int c = bwp - 4; c >= r0 + 32; c -= 4) {
        float xc[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) xc[k] = X[(c + k) * bwp];
        const float* P = up + up_panel(c / 4) + 4 * r0;
#pragma unroll
        for (int rr = 0; rr < 32; rr += 8) {
          f32x4 p[8];
#pragma unroll
          for (int r = 0; r < 8; ++r) p[r] = *reinterpret_cast<const f32x4*>(P + 4 * (rr + r));
#pragma unroll
          for (int k = 3; k >= 0; --k)
            if (c + k <= j) {
#pragma unroll
              for (int r = 0; r < 8; ++r) x[rr + r] -= p[r][k] * xc[k];
            }
        }
      }
      static_for<8>([&](auto gc) __attribute__((always_inline)) {
        constexpr int c = 28 - 4 * decltype(gc)::value;
        const float* P = up + up_panel((r0 + c) / 4) + 4 * r0;
#pragma unroll
        for (int k = 3; k >= 0; --k)
          if (r0 + c + k <= j) {
            x[c + k] *= rinv[r0 + c + k];
#pragma unroll
            for (int r = 0; r < c + k; ++r) x[r] -= P[4 * r + k] * x[c + k];
          }
      });
#pragma unroll
      for (int r = 0; r < 32; ++r)
        if (r0 + r < bwp) X[(r0 + r) * bwp] = r0 + r <= j ? x[r] : 0.0f;
    }
  }
}

// Row i of a block's inverse, columns 64h .. 64h+63, as 16 four-vectors
// (zero outside the block). The row's entries outside columns [jlo, jhi)
// are zeros of the inverse: four-vectors wholly outside are not read.
__device__ __attribute__((always_inline)) inline void load_inv_row(
    const float* __restrict__ M, int bw, int bwp, int i, int h, int jlo, int jhi,
    f32x4 (&mv)[16]) {
  const f32x4* R = reinterpret_cast<const f32x4*>(M + (int64_t)i * bwp);
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int j = 64 * h + 4 * k;
    mv[k] = (i < bw && j < bwp && j < jhi && j + 4 > jlo) ? R[j / 4]
                                                          : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
}

// v = M yb for a block of up to 128 entries: thread (i = tid % 128, h = tid /
// 128) sums its 64 columns in order, the two halves are added in order; yb
// (128 entries, zero past the block) in LDS, v to LDS.
__device__ __attribute__((always_inline)) inline void inv_apply(const f32x4 (&mv)[16],
                                                                const float* yb, float (*zp)[128],
                                                                float* v) {
  const int tid = threadIdx.x, i = tid & 127, h = tid >> 7;
  float acc = 0.0f;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const f32x4 y = *reinterpret_cast<const f32x4*>(yb + 64 * h + 4 * k);
    acc += mv[k].x * y.x;
    acc += mv[k].y * y.y;
    acc += mv[k].z * y.z;
    acc += mv[k].w * y.w;
  }
  zp[h][i] = acc;
  __syncthreads();
  if (tid < 128) v[tid] = zp[0][tid] + zp[1][tid];
  __syncthreads();
}

// Forward block step: every workgroup forms z = ML y[x0:x1] of its block;
// the one marked write stores z as the block's solution entries (rhs only:
// the front's vector keeps y, which the step's other workgroups read); a
// tile workgroup then updates its 64 rows, y[x1 + r0 + lane] -= L[., x0:x1]
// z, with fwd_bgemv_body's operations.
__global__ void __launch_bounds__(kWG)
fwd_inv_kernel(DevSym s, const InvItem* __restrict__ items, const float* __restrict__ inv,
               const float* __restrict__ lnz, float* __restrict__ rhs, int64_t ldr, int nrhs,
               float* __restrict__ vec) {
  const int64_t vs = blockIdx.y;  // value set
  inv += vs * s.vs_inv;
  lnz += vs * s.vs_lnz;
  rhs += vs * ldr * nrhs;
  vec += vs * s.vs_vec * nrhs;
  __shared__ __attribute__((aligned(16))) float yb[128];
  __shared__ float zp[2][128];
  __shared__ float zs[128];
  __shared__ __attribute__((aligned(16))) float zq[4][32];  // zs by quarters, zeros behind
  __shared__ float red[4][64];
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const InvItem* const ip = items + blockIdx.x;
  const InvItem it = *ip;
  const int L = it.L, c0 = it.x0, bw = it.x1 - it.x0, bwp = 4 * ((bw + 3) / 4);
  // row i of ML = L^-1 P is zero from the end of its piece on (the
  // interchanges stay inside the pieces)
  int pend = bw;
#pragma unroll
  for (int q = 1; q < 8; ++q) {
    const int ps = ip->pst[q];
    if (ps > (tid & 127) && ps < pend) pend = ps;
  }
  f32x4 mv[16];
  load_inv_row(inv + it.inv, bw, bwp, tid & 127, tid >> 7, 0, pend, mv);
  const bool tile = it.r0 >= 0;
  const int r = it.x1 + it.r0 + lane;
  const int cb = bw * wave / 4, ce = bw * (wave + 1) / 4;
  // the tile's L entries, in flight with the inverse: block column c's lnz
  // offset from the item's piece table (a piece's columns follow each other
  // at its row count; the column index is uniform in the wave)
  float lv[32];
  {
    int q = 0;
    while (q < 7 && ip->pst[q + 1] <= cb) ++q;
    int64_t str = L - c0 - ip->pst[q];
    int64_t lcc = ip->pbs[q] + (int64_t)(cb - ip->pst[q]) * str;
    int nxt = q < 7 ? ip->pst[q + 1] : (1 << 30);
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const int c = cb + j;
      if (c == nxt) {
        ++q;
        str = L - c0 - ip->pst[q];
        lcc = ip->pbs[q];
        nxt = q < 7 ? ip->pst[q + 1] : (1 << 30);
      }
      lv[j] = (tile && r < L && c < ce) ? lnz[lcc + r] : 0.0f;
      lcc += str;
    }
  }
  float* const yf = vec + it.fvec * nrhs;
  // the first right-hand side's y
  if (tid < 128) yb[tid] = (tid < bw) ? yf[c0 + tid] : 0.0f;
  float yr = (tile && wave == 0 && r < L) ? yf[r] : 0.0f;
  __syncthreads();
  for (int q = 0; q < nrhs; ++q) {
    float* yg = yf + (int64_t)q * L;
    if (q > 0) {
      if (tid < 128) yb[tid] = (tid < bw) ? yg[c0 + tid] : 0.0f;
      yr = (tile && wave == 0 && r < L) ? yg[r] : 0.0f;
      __syncthreads();
    }
    inv_apply(mv, yb, zp, zs);
    if ((it.flags & 1) && tid < bw) rhs[(int64_t)q * ldr + it.fc0 + c0 + tid] = zs[tid];
    if (!tile) continue;  // the whole workgroup
    if (lane < 32) zq[wave][lane] = cb + lane < ce ? zs[cb + lane] : 0.0f;  // its own wave's
    wave_lds_sync();
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < 32; ++j) acc += lv[j] * zq[wave][j];
    red[wave][lane] = acc;
    __syncthreads();
    if (tile && wave == 0 && r < L)
      yg[r] = yr - (((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane]);
    __syncthreads();
  }
}

// Backward block step. Before it, the right-hand side holds y = z - t for
// the rows whose t is done. A row workgroup first forms x of the block
// after its row's block, x = MU y[x0:x1], then its row's t = U[c, rc1:L]
// x[rc1:L] (x[x0:x1] from LDS, of later blocks from the front's vector, the
// update rows as gathered) with bwd_bgemv_body's operations, and leaves y_c
// = z_c - t_c in the right-hand side. The workgroup marked write stores x of
// that block in the front's vector (read by later steps only). A finishing
// workgroup (one per front) forms x of the front's first block into the
// right-hand side and copies the other blocks' x there.
__global__ void __launch_bounds__(kWG)
bwd_inv_kernel(DevSym s, const InvItem* __restrict__ items, const float* __restrict__ inv,
               const float* __restrict__ unz, float* __restrict__ rhs, int64_t ldr, int nrhs,
               float* __restrict__ vec) {
  const int64_t vs = blockIdx.y;  // value set
  inv += vs * s.vs_inv;
  unz += vs * s.vs_unz;
  rhs += vs * ldr * nrhs;
  vec += vs * s.vs_vec * nrhs;
  constexpr int QB = 4;   // right-hand sides sharing one read of the row
  constexpr int CH = 16;  // columns per thread and pass
  __shared__ __attribute__((aligned(16))) float yb[128];
  __shared__ float zp[2][128];
  __shared__ float xs[QB][128];
  __shared__ float red[QB][4];
  const int tid = threadIdx.x, lane = tid % 64, wave = wave_id();
  const InvItem it = items[blockIdx.x];
  const bool row = it.c >= 0, fin = (it.flags & 2) != 0;
  const int L = it.L;
  const int xlo = it.x0, xhi = it.x1, xbw = it.x1 - it.x0;  // x columns formed here
  const bool hasx = xbw > 0;
  const int bwp = 4 * ((xbw + 3) / 4);
  f32x4 mv[16];
  if (hasx)  // MU is upper triangular
    load_inv_row(inv + it.inv + (int64_t)bwp * bwp, xbw, bwp, tid & 127, tid >> 7, tid & 127,
                 xbw, mv);
  float* const yf = vec + it.fvec * nrhs;
  for (int q0 = 0; q0 < nrhs; q0 += QB) {
    const int nq = min(QB, nrhs - q0);
    if (hasx) {
      for (int qq = 0; qq < nq; ++qq) {
        const float* y = rhs + (int64_t)(q0 + qq) * ldr + it.fc0 + xlo;
        if (tid < 128) yb[tid] = (tid < xbw) ? y[tid] : 0.0f;
        __syncthreads();
        inv_apply(mv, yb, zp, xs[qq]);
      }
      if (it.flags & 3) {
        for (int qq = 0; qq < nq; ++qq)
          if (tid < xbw) {
            if (fin)
              rhs[(int64_t)(q0 + qq) * ldr + it.fc0 + xlo + tid] = xs[qq][tid];
            else
              yf[(int64_t)(q0 + qq) * L + xlo + tid] = xs[qq][tid];
          }
      }
      if (fin) {
        for (int qq = 0; qq < nq; ++qq)
          for (int j = xhi + tid; j < it.W; j += kWG)
            rhs[(int64_t)(q0 + qq) * ldr + it.fc0 + j] = yf[(int64_t)(q0 + qq) * L + j];
      }
    }
    if (row) {
      const float* u = unz + it.ucol;
      float acc[QB];
#pragma unroll
      for (int qq = 0; qq < QB; ++qq) acc[qq] = 0.0f;
      for (int j0 = it.rc1 + tid; j0 < L; j0 += CH * kWG) {
        float uv[CH];
#pragma unroll
        for (int t = 0; t < CH; ++t) {
          const int j = j0 + kWG * t;
          uv[t] = (j < L) ? u[j] : 0.0f;
        }
#pragma unroll
        for (int qq = 0; qq < QB; ++qq) {
          if (qq < nq) {
            const float* yg = yf + (int64_t)(q0 + qq) * L;
            float xv[CH];
#pragma unroll
            for (int t = 0; t < CH; ++t) {
              const int j = j0 + kWG * t;
              xv[t] = (j >= L) ? 0.0f : (j < xhi && j >= xlo) ? xs[qq][j - xlo] : yg[j];
            }
#pragma unroll
            for (int t = 0; t < CH; ++t) acc[qq] += uv[t] * xv[t];
          }
        }
      }
      const float sum = wave_sums<QB>(acc, lane);
      if (lane % (64 / QB) == 0) red[lane / (64 / QB)][wave] = sum;
      __syncthreads();
      if (tid < nq) {
        float* y = rhs + (int64_t)(q0 + tid) * ldr + it.fc0 + it.c;
        *y = *y - (((red[tid][0] + red[tid][1]) + red[tid][2]) + red[tid][3]);
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Permutation, residual and refinement helpers (double unless noted).
// pb[i] = b[perm[i]-1] (rhs = b[rperm], SpkSparseBase.jl:407) and
// x[j] = pb[invp[j]-1] (solution = rhs[rinvp], :413).
// ---------------------------------------------------------------------------
// value set blockIdx.y: in and out start ivs and ovs elements further
template <typename TI, typename TO>
__global__ void permute_kernel(const TI* __restrict__ in, int64_t ldi,
                               TO* __restrict__ out, int64_t ldo,
                               const int64_t* __restrict__ idx, int64_t n,
                               int nrhs, int64_t ivs, int64_t ovs) {
  in += (int64_t)blockIdx.y * ivs;
  out += (int64_t)blockIdx.y * ovs;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int64_t src = idx[i] - 1;
  for (int q = 0; q < nrhs; ++q) out[i + q * ldo] = (TO)in[src + q * ldi];
}

// r = b - A x with A in CSR (original numbering): G consecutive lanes per
// row, lane g summing the row's entries g, g + G, ... in order, the G
// partial sums then added pairwise (G = 1: one row per thread, the entries in
// order). Value set blockIdx.y: its values nnz further, its rows of x, b and
// r n further (the sets' systems stacked as one block-diagonal system).
template <int G>
__global__ void __launch_bounds__(kWG)
residual_kernel(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind,
                const double* __restrict__ val, const double* __restrict__ x, int64_t ldx,
                const double* __restrict__ b, int64_t ldb, double* __restrict__ r, int64_t ldr,
                int64_t n, int nrhs, int64_t nnz) {
  const int64_t vs = blockIdx.y;
  val += vs * nnz;
  x += vs * n;
  b += vs * n;
  r += vs * n;
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / G;
  const int g = (int)(threadIdx.x % G);
  if (i >= n) return;  // a row's G lanes leave together
  const int64_t k0 = rowptr[i], k1 = rowptr[i + 1];
  for (int q = 0; q < nrhs; ++q) {
    const double* xq = x + (int64_t)q * ldx;
    double acc = 0.0;
    for (int64_t k = k0 + g; k < k1; k += G) acc = fma(val[k], xq[colind[k]], acc);
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, G);
    if (g == 0) r[i + q * ldr] = b[i + q * ldb] - acc;
  }
}

__device__ inline double abs_nan_inf(double x) {
  const double a = fabs(x);
  return (a != a) ? __builtin_huge_val() : a;
}

// Row sums |A| for ||A||_inf (a NaN entry makes its row sum +inf); value set
// blockIdx.y as in residual_kernel.
__global__ void rowabs_kernel(const int64_t* __restrict__ rowptr,
                              const double* __restrict__ val,
                              double* __restrict__ out, int64_t n, int64_t nnz) {
  val += (int64_t)blockIdx.y * nnz;
  out += (int64_t)blockIdx.y * n;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double acc = 0.0;
  for (int64_t k = rowptr[i]; k < rowptr[i + 1]; ++k) acc += abs_nan_inf(val[k]);
  out[i] = acc;
}

// Max |v| over row chunks [clo[c], clo[c+1]) of each column, folded into the
// per-(segment, column) maxima out[cseg[c] + q * nseg] by an integer
// atomicMax on the bit patterns (a non-negative double orders as its bits,
// +inf above every finite value); out starts at +0.0. NaN entries count as
// +inf. One block per (chunk, column).
__global__ void segmax_chunk_kernel(const double* __restrict__ v, int64_t ld,
                                    const int64_t* __restrict__ clo,
                                    const int32_t* __restrict__ cseg, int nchunks, int nseg,
                                    unsigned long long* __restrict__ out) {
  __shared__ double red[kWG];
  const int c = blockIdx.x % nchunks, q = blockIdx.x / nchunks;
  const double* vq = v + (int64_t)q * ld;
  const int64_t lo = clo[c], hi = clo[c + 1];
  double m = 0.0;
  int64_t r = lo + threadIdx.x;
  for (; r + 7 * kWG < hi; r += 8 * kWG) {
    double a[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = abs_nan_inf(vq[r + u * kWG]);
#pragma unroll
    for (int u = 0; u < 8; ++u) m = fmax(m, a[u]);
  }
  for (; r < hi; r += kWG) m = fmax(m, abs_nan_inf(vq[r]));
  red[threadIdx.x] = m;
  __syncthreads();
  for (int off = kWG / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + off]);
    __syncthreads();
  }
  if (threadIdx.x == 0)
    atomicMax(out + cseg[c] + (int64_t)q * nseg, (unsigned long long)__double_as_longlong(red[0]));
}

// x += d (d in the factor precision, already in original numbering).
template <typename T>
__global__ void axpy_kernel(double* __restrict__ x, int64_t ldx,
                            const T* __restrict__ d, int64_t ldd, int64_t n,
                            int nrhs) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int q = 0; q < nrhs; ++q) x[i + q * ldx] += (double)d[i + q * ldd];
}

// ---------------------------------------------------------------------------
// The 1-norm estimate of A^-1 (Hager's method, the reference's commented
// sparsespdainverseonenorm, SpkSparseSpdSolver.jl:346-431): its vector steps.
// ---------------------------------------------------------------------------
// mode 0: x_i = 1/n; mode 1: the unit vector e_j; mode 2: x_i = (-1)^i (1 +
// i/(n-1)) (0-based i: the reference's altsgn vector).
__global__ void condest_fill_kernel(double* __restrict__ x, int64_t n, int mode, int64_t j) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double v;
  if (mode == 0)
    v = 1.0 / (double)n;
  else if (mode == 1)
    v = (i == j) ? 1.0 : 0.0;
  else
    v = ((i & 1) ? -1.0 : 1.0) * (1.0 + (double)i / (double)(n - 1));
  x[i] = v;
}

// Per-block partial results over [b chunk, (b+1) chunk): the sum of |x|
// (a fixed tree order), the largest |x| and its first index.
__global__ void condest_reduce_kernel(const double* __restrict__ x, int64_t n, int64_t chunk,
                                      double* __restrict__ psum, double* __restrict__ pmax,
                                      int64_t* __restrict__ pidx) {
  __shared__ double ss[kWG], sm[kWG];
  __shared__ int64_t si[kWG];
  const int64_t lo = (int64_t)blockIdx.x * chunk, hi = min(n, lo + chunk);
  double sum = 0.0, mx = -1.0;
  int64_t mi = lo;
  for (int64_t i = lo + threadIdx.x; i < hi; i += kWG) {
    const double a = fabs(x[i]);
    sum += a;
    if (a > mx) {
      mx = a;
      mi = i;
    }
  }
  ss[threadIdx.x] = sum;
  sm[threadIdx.x] = mx;
  si[threadIdx.x] = mi;
  __syncthreads();
  for (int off = kWG / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) {
      ss[threadIdx.x] += ss[threadIdx.x + off];
      const double m2 = sm[threadIdx.x + off];
      const int64_t i2 = si[threadIdx.x + off];
      if (m2 > sm[threadIdx.x] || (m2 == sm[threadIdx.x] && i2 < si[threadIdx.x])) {
        sm[threadIdx.x] = m2;
        si[threadIdx.x] = i2;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    psum[blockIdx.x] = ss[0];
    pmax[blockIdx.x] = sm[0];
    pidx[blockIdx.x] = si[0];
  }
}

// Signs s_i = sign(1, x_i) (+1 for x_i >= 0): compare mode counts the
// entries whose sign differs from isgn; otherwise x and isgn become the
// signs.
__global__ void condest_sign_kernel(double* __restrict__ x, int32_t* __restrict__ isgn,
                                    int64_t n, int compare,
                                    unsigned int* __restrict__ changed) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int sg = (x[i] < 0.0) ? -1 : 1;
  if (compare) {
    if (sg != isgn[i]) atomicAdd(changed, 1u);
  } else {
    x[i] = (double)sg;
    isgn[i] = sg;
  }
}

// Factor conversions for download.
template <typename TI, typename TO>
__global__ void convert_kernel(const TI* __restrict__ in, TO* __restrict__ out,
                               int64_t len) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < len; i += stride) out[i] = (TO)in[i];
}

}  // namespace spk
