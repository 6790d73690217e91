// Chebyshev smoothing of the Schur complement (pressure mass matrix, one viscosity
// per cell, degree 2) with several steps per launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>
#include <type_traits>
#include <vector>

#include "mfs_internal.h"

namespace mfs {

// Several Chebyshev steps of the Schur smoother per launch.  A workgroup keeps x
// of a region of nodes (with one ring around it) in LDS, and b, D^-1, d and 1/eta of its
// nodes in registers; every step updates the whole region, so that after k steps the
// nodes within k - 1 of a face inside the level lack updates of their neighbours, and
// the core away from them is written.  Beyond the level x, 1/eta and D^-1 are zero, so
// its faces need no such margin.  A thread owns RUN nodes of a column and sums per
// plane the quadrants that its column touches; in 3D a row of 16 lanes is a row of the
// region and the neighbours' sums come by DPP, so a node takes 4.5 (3D) or 6 (2D)
// LDS reads a step instead of 35 or 13.  Bound by the vector units (200 instructions a
// wave for 4 planes of 64 nodes, 4 waves a SIMD) and, below 256 blocks, by one block's chain
// of steps.  Four steps, against four launches of one step each: 17^3 nodes in
// double 11.5 us (18.5), 33^3 13.2 us (18.6), 65^3 27 us (50), in single 65^3 22 us (27);
// eight steps in 2D, 129^2 in double 7.2 us (26), 1025^2 52 us (105).  A 9^3 level's 16
// steps take 17.5 us (23 us in a workgroup with a thread per node), 25^2 8.1 us (27 us).
template <int DIM>
struct SweepShape;
template <>
struct SweepShape<3> {
  static constexpr int WX = 14, WY = 14, RUN = 4, SEG = 4, HALO = 4, THREADS = 896;
};
template <>
struct SweepShape<2> {
  static constexpr int WX = 30, WY = 1, RUN = 2, SEG = 15, HALO = 8, THREADS = 512;
};
// the region's largest extent in direction d
template <int DIM>
constexpr __host__ __device__ int sweep_width(int d) {
  using S = SweepShape<DIM>;
  return d == DIM - 1 ? S::RUN * S::SEG : (d == 0 ? S::WX : S::WY);
}
// cores of the blocks in each direction: the first is outer, the others inner
struct SweepTiles {
  int outer[3], inner[3], margin;
};
// neighbour lane within a row of 16 (0 past its ends)
template <int CTRL>
__device__ __forceinline__ float row_neighbour(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double row_neighbour(double v) {
  const long long i = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)i, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(i >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int DIM, typename T>
__global__ void __launch_bounds__(SweepShape<DIM>::THREADS)
    k_mass_sweeps(const LevelDesc L, const SweepTiles W, const T *xin, T *xout, const T *__restrict__ b,
                  const T *__restrict__ dinv, const T *__restrict__ ieta, const MassChebSeq seq, const int x_zero) {
  using S = SweepShape<DIM>;
  constexpr int RUN = S::RUN, X = S::WX + 2, Y = S::WY + 2;
  constexpr int ROW = X, SLICE = DIM == 3 ? X * Y : X;  // strides: y in a plane, along the runs
  constexpr int ENTRIES = SLICE * (RUN * S::SEG + 2);
  constexpr int Q = DIM == 3 ? 4 : 2;
  __shared__ T sm[2][ENTRIES];
  const int blk[3] = {(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z};
  int o[3], lo[3], hi[3], w_[3];  // LDS entry (0, 0, 0) is node o; nodes [lo, hi) are written
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    lo[d] = blk[d] == 0 ? 0 : W.outer[d] + (blk[d] - 1) * W.inner[d];
    hi[d] = min(blk[d] == 0 ? W.outer[d] : lo[d] + W.inner[d], L.np[d]);
    if (blk[d] + 1 == (int)(d == 0 ? gridDim.x : (d == 1 ? gridDim.y : gridDim.z))) hi[d] = L.np[d];
    const int from = max(lo[d] - W.margin, 0), to = min(hi[d] + W.margin, L.np[d]);
    o[d] = from - 1;
    w_[d] = to - from;
  }
  auto offset = [&](int x, int y, int z) { return x + L.np[0] * (y + L.np[1] * z); };
  auto inside = [&](int x, int y, int z) {
    return (unsigned)x < (unsigned)L.np[0] && (unsigned)y < (unsigned)L.np[1] && (DIM == 2 || (unsigned)z < (unsigned)L.np[2]);
  };
  // x into the first buffer, 1/eta (entry = the cell above its node) into the second
  for (int i = threadIdx.x; i < ENTRIES; i += S::THREADS) {
    const int x = o[0] + i % X, y = o[1] + (DIM == 3 ? i / X % Y : i / X), z = DIM == 3 ? o[2] + i / SLICE : 0;
    sm[0][i] = !x_zero && inside(x, y, z) ? xin[offset(x, y, z)] : (T)0;
    const bool cell = (unsigned)x < (unsigned)L.n[0] && (unsigned)y < (unsigned)L.n[1] &&
                      (DIM == 2 || (unsigned)z < (unsigned)L.n[2]);
    sm[1][i] = cell ? ieta[x + L.n[0] * (y + L.n[1] * z)] : (T)0;
  }
  // rows of 16 lanes in 3D (the ring's lanes idle), columns packed in 2D
  const int row = DIM == 3 ? threadIdx.x / X : threadIdx.x / w_[0];
  const int cx = DIM == 3 ? (int)threadIdx.x % X : (int)threadIdx.x - row * w_[0] + 1;
  const int seg = DIM == 3 ? row / w_[1] : row, cy = DIM == 3 ? row - seg * w_[1] + 1 : 0;
  const bool work = seg * RUN < w_[DIM - 1];
  const bool active = work && cx >= 1 && cx <= w_[0];
  // entry of the thread's column below its first node, and the one its cells are read around
  const int e0 = work ? cx + ROW * cy + SLICE * RUN * seg : X, ew = active ? e0 : X + 1;
  T bi[RUN], di[RUN], dd[RUN], w[RUN + 1][Q];
  int at[RUN];
#pragma unroll
  for (int r = 0; r < RUN; ++r) {
    const int x = o[0] + cx, y = DIM == 3 ? o[1] + cy : o[1] + 1 + RUN * seg + r;
    const int z = DIM == 3 ? o[2] + 1 + RUN * seg + r : 0;
    const bool ok = active && inside(x, y, z);
    const int k = ok ? offset(x, y, z) : 0;
    const T bk = b[k], dk = dinv[k];
    bi[r] = ok ? bk : (T)0;
    di[r] = ok ? dk : (T)0;
    dd[r] = 0;
    const bool write = ok && x >= lo[0] && x < hi[0] && y >= lo[1] && y < hi[1] && (DIM == 2 || (z >= lo[2] && z < hi[2]));
    at[r] = write ? k : -1;
  }
  __syncthreads();
  using LC = LevelConst<T>;
  // the smallest reference entry, 1/6 per direction, rounded as in mass_node; the others are
  // 2, 4 and 8 times it there too.  So the smoother and the V-cycle's residual, which mass_node
  // forms, share their entries: in single 1.1e-7 off, but by the same.  With vol s^2 / 216,
  // nearer by itself, single V-cycles on 16^3 cells ended 9.2e-8 from the 64-bit result, now 6.5e-8
  constexpr T half3 = T(1) / T(3) / T(2);
  const T scale = LC::vol(L) * LC::s(L) * LC::s(L) * (DIM == 3 ? half3 * half3 * half3 : half3 * half3);
#pragma unroll
  for (int p = 0; p <= RUN; ++p)
#pragma unroll
    for (int q = 0; q < Q; ++q) w[p][q] = scale * sm[1][ew + SLICE * p + (q & 1) - 1 + (DIM == 3 ? ROW * ((q >> 1) - 1) : 0)];
  __syncthreads();
  for (int i = threadIdx.x; i < ENTRIES; i += S::THREADS) sm[1][i] = sm[0][i];
  T xi[RUN];
#pragma unroll
  for (int r = 0; r < RUN; ++r) xi[r] = sm[0][e0 + SLICE * (r + 1)];
  __syncthreads();
  for (int s = 0; s < seq.n; ++s) {
    const T f1 = (T)seq.f1[s], f2 = (T)seq.f2[s];
    const int first = seq.first[s];
    T v[RUN];
#pragma unroll
    for (int r = 0; r < RUN; ++r) v[r] = 0;
    if (work && !(x_zero && s == 0)) {
      const T *const u = sm[s & 1] + e0;
      T below[Q];
#pragma unroll
      for (int p = 0; p < RUN + 2; ++p) {
        const T *const g = u + SLICE * p;
        T m[Q];
        if constexpr (DIM == 3) {
          const T two = g[0] + g[0], l = two + g[-ROW], h = two + g[ROW];
          m[0] = l + l + row_neighbour<0x111>(l);
          m[1] = l + l + row_neighbour<0x101>(l);
          m[2] = h + h + row_neighbour<0x111>(h);
          m[3] = h + h + row_neighbour<0x101>(h);
        } else {
          const T two = g[0] + g[0];
          m[0] = two + g[-1];
          m[1] = two + g[1];
        }
        if (p > 0) {  // the cells between plane p - 1 and plane p
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            if (p > 1) v[p - 2] += w[p - 1][q] * (below[q] + below[q] + m[q]);
            if (p <= RUN) v[p - 1] += w[p - 1][q] * (m[q] + m[q] + below[q]);
          }
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) below[q] = m[q];
      }
    }
    T *const out = sm[(s + 1) & 1] + e0;
#pragma unroll
    for (int r = 0; r < RUN; ++r) {
      const T res = bi[r] - v[r];
      dd[r] = first ? di[r] * res * f2 : f1 * dd[r] + f2 * di[r] * res;
      xi[r] += dd[r];
      if (active) out[SLICE * (r + 1)] = xi[r];
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < RUN; ++r)
    if (at[r] >= 0) xout[at[r]] = xi[r];
}

// The steps of one launch: as many whole sweeps (from a first step up to the next) as
// the margins allow, all of them where the region covers the level.  False where not even one
// sweep fits (a degree above the halo, or the steps above MassChebSeq::MAX), and
// on large 3D levels in single: the region's halo costs 4.6 times the arithmetic, and a step
// of its own halves its traffic there (97^3: 61 us for four steps here, 50 us in four
// launches; 129^3: 133 against 93; in double 80 against 105 and 176 against 208).
template <typename T>
bool launch_mass_sweeps(const LevelDesc &L, T *x, T *other, const T *b, const T *dinv, const T *ieta,
                        const MassChebSeq &seq, bool x_zero, hipStream_t st) {
  if (!ieta || seq.n < 1 || !mass_nodes_ok(L)) return false;
  if (L.dim == 3 && sizeof(T) == 4 && L.pnodes > 500000) return false;
  auto go = [&](auto dimc) {
    constexpr int DIM = decltype(dimc)::value;
    bool whole = true;
    for (int d = 0; d < DIM; ++d) whole = whole && L.np[d] <= sweep_width<DIM>(d);
    std::vector<int> ends;  // step after the last one of each launch
    for (int s = 0, from = 0; s < seq.n;) {
      int e = s + 1;
      while (e < seq.n && !seq.first[e]) ++e;
      if (whole || e - from <= SweepShape<DIM>::HALO) {
        if (s == from)
          ends.push_back(e);
        else
          ends.back() = e;
        s = e;
      } else {
        if (s == from) return false;
        from = s;
      }
    }
    T *cur = x, *alt = other;
    if (!whole && x_zero && (ends.size() & 1)) std::swap(cur, alt);
    for (size_t i = 0, from = 0; i < ends.size(); ++i) {
      MassChebSeq part{};
      for (int s = (int)from; s < ends[i]; ++s, ++part.n) {
        part.f1[part.n] = seq.f1[s];
        part.f2[part.n] = seq.f2[s];
        part.first[part.n] = seq.first[s];
      }
      const bool zero = x_zero && i == 0;
      SweepTiles W{{1, 1, 1}, {1, 1, 1}, whole ? 0 : part.n - 1};
      dim3 grid(1, 1, 1);
      for (int d = 0; d < DIM; ++d) {
        // as few blocks as hold the level, with cores as equal as the one-sided margins of the first and last allow
        const int np = L.np[d], full = sweep_width<DIM>(d), one = full - W.margin, both = one - W.margin;
        const int nt = np <= full ? 1 : 2 + std::max(0, (np - 2 * one + both - 1) / both);
        W.inner[d] = nt < 3 ? 1 : std::min(both, (np + nt - 1) / nt);
        W.outer[d] = nt == 1 ? np : (np - (nt - 2) * W.inner[d] + 1) / 2;
        (d == 0 ? grid.x : (d == 1 ? grid.y : grid.z)) = (unsigned)nt;
      }
      hipLaunchKernelGGL((k_mass_sweeps<DIM, T>), grid, dim3(SweepShape<DIM>::THREADS), 0, st, L, W, cur,
                         whole ? cur : alt, b, dinv, ieta, part, zero ? 1 : 0);
      MFS_HIP(hipGetLastError());
      if (!whole) std::swap(cur, alt);
      from = ends[i];
    }
    if (cur != x) MFS_HIP(hipMemcpyAsync(x, cur, L.pnodes * sizeof(T), hipMemcpyDeviceToDevice, st));
    return true;
  };
  return L.dim == 3 ? go(std::integral_constant<int, 3>()) : go(std::integral_constant<int, 2>());
}
template bool launch_mass_sweeps<double>(const LevelDesc &, double *, double *, const double *, const double *,
                                         const double *, const MassChebSeq &, bool, hipStream_t);
template bool launch_mass_sweeps<float>(const LevelDesc &, float *, float *, const float *, const float *,
                                        const float *, const MassChebSeq &, bool, hipStream_t);

}  // namespace mfs
