// gfx950 kernels for the Q2 x Q1 Stokes operator and A block on uniform box
// levels with one viscosity per cell (every multigrid level, and the active
// level under material averaging).
//
// Restates, per cell:
//   StokesOperator::local_apply   source/simulator/solver/matrix_free_operators.cc:376-547
//   ABlockOperator::inner_cell_operation / local_apply   :974-1052
//
// On a uniform level with one viscosity per cell the cell operator is the
// viscosity times one constant matrix (81 x 81 in 3D).  The cell is symmetric
// under reflection in each direction, so in the basis of differences of
// opposite nodes (per direction a - 2 b + c, b, a - c) that matrix
// splits into blocks of equal symmetry: 795 entries instead of 6561 in 3D (64
// instead of 324 in 2D), B^T and B into one entry per velocity mode.  That is
// 3.5 times less arithmetic than the sum factorization over quadrature points
// and needs no quadrature data.  The integrals are exact, as the Gauss rule's
// are (degree 4 in each direction).  A constant is the mode b in all
// directions, whose entries vanish: applied to a constant the operator gives
// zero to the last bit.  With a + c for a - 2 b + c it did so only up to the
// rounding of the entries, the same in every cell: 15 GMRES steps on 12 2D
// problems of 16^2 to 128^2 cells then ended 1.9e-13 to 2.9e-13 from the
// result of 64 bits, now 3.5e-14 to 4.2e-14 (from quadrature 5e-14 to 1e-13),
// at the same speed.
//
// A workgroup owns the nodes of a box of cells and computes every cell that
// touches them, so each node is finished by one thread: no work array, no
// second pass, no atomics, one launch, fixed summation order.  The price is
// one extra layer of cells at the low side of the box (of at most 64 columns 40 to 49
// are owned) and one below each march.
//
// Against the split quadrature kernels (kernels_planes.hip, kernels_gather.hip):
// FP64 Stokes apply 96^3 417 -> 173 us, 8^3 16.7 -> 4.6 us; FP32 A block 96^3
// 209 -> 92 us; 64^3 preconditioner 2.46 -> 2.15 ms; 2D ensemble 81 -> 49 ms.
// Bound (96^3, counters): in FP64 latency, 1.6 waves a SIMD wait 41 % of the time at
// the two barriers of a layer and for loads; the vector units are 40 % busy and memory
// moves 2.65 TB/s, 54 % of what a copy reaches.  In FP32 the vector units, 70 % busy.

#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>
#include <vector>

#include "mfs_internal.h"
#include "tile_common.h"

namespace mfs {

// ------------------------------------------------------------------ cell matrices
namespace {

constexpr int MARCH_CHEB = 3;  // besides MODE_SET / RESID / ADD

// 1D integrals over [0, 1] of the modes of the quadratic basis (nodes 0, 1/2, 1
// with values a, b, c): modes a - 2 b + c, b and a - c, whose functions are
// (1 - 2x)^2 / 2, 1 and (1 - 2x) / 2; and of the linear basis' modes a + c and
// a - c with functions 1 / 2 and (1 - 2x) / 2.  Mass, stiffness, derivative
// times value, and the two products with the linear basis.  The derivative of
// mode 1 is zero: a constant has exactly no strain, however the other entries
// are rounded.  (With modes a + c, b, a - c the entries cancel for a constant
// only up to their rounding, the same in every cell of a level, which acts like
// a small mass term and which a solve amplifies with the condition of the level.)
constexpr long double kM[3][3] = {{1.0L / 20, 1.0L / 6, 0}, {1.0L / 6, 1, 0}, {0, 0, 1.0L / 12}};
constexpr long double kK[3][3] = {{4.0L / 3, 0, 0}, {0, 0, 0}, {0, 0, 1}};
constexpr long double kD[3][3] = {{0, 0, -1.0L / 3}, {0, 0, 0}, {-1.0L / 6, -1, 0}};
constexpr long double kPM[3][2] = {{1.0L / 12, 0}, {1.0L / 2, 0}, {0, 1.0L / 12}};
constexpr long double kPD[3][2] = {{0, -1.0L / 3}, {0, 0}, {-1.0L / 2, 0}};

// modes 0, 1 are even, mode 2 is odd
constexpr __host__ __device__ int par(int m) { return m == 2; }

// 2D: does the block (output component c, input component d) couple output
// mode m with input mode q?  The parities agree in both directions, or differ
// in both for an off-diagonal block; the constant (mode 1 in both directions) couples with none
constexpr __host__ __device__ bool couples2(int c, int d, int m, int q) {
  if (m == 4 || q == 4) return false;
  const bool x = par(m % 3) == par(q % 3), y = par(m / 3) == par(q / 3);
  return c == d ? x && y : !x && !y;
}
// pressure mode that couples with velocity mode m of component c (bit e: odd in direction e)
constexpr __host__ __device__ int pressure_mode2(int c, int m) { return (par(m % 3) | par(m / 3) << 1) ^ (1 << c); }

// 2D coefficients per output component c: the blocks of the input components c
// and c + 1 (mod 2), input mode by input mode, then the B^T entry of every mode.
struct March2 {
  static constexpr int NM = 9, STRIDE = 18 + 14 + NM;
};

// 3D coefficients per output component c, in register rows of 16 (k_march3).
// Modes and components are numbered from direction c on (mode m_c + 3 m_{c+1} +
// 9 m_{c+2}, directions mod 3), so that one code serves every component.  The
// blocks of the input components c, c + 1, c + 2, each by symmetry class of its
// input modes, every input of a class with every output of the
// class it couples with.  The products of class sizes are powers of two.  Class 0
// of the diagonal block, even in all directions, leaves out what vanishes
// (class0_in): 2 rows and 12 places.  By size the diagonal block fills 2 rows,
// one of 12 + 4, 3 rows and one of 4 + 4 + 1, another block 4 rows and one of
// 4 x 4; then B^T by class: 8 + 4 + 4, 4 + 2 + 2 + 2 + 1.
struct March3 {
  static constexpr int ROWS = 17, STRIDE = (ROWS + 2) * 16;
};
// k-th symmetry class (bit e: odd in direction e) in table order; the diagonal
// block's order also is the B^T rows' order
constexpr __host__ __device__ int class_at(int c, int d, int k) {
  if (c == d) {
    constexpr int by_size[8] = {0, 1, 2, 4, 3, 5, 6, 7};
    return by_size[k];
  }
  // the classes even in the third direction first
  const int t = 3 - c - d, lo = t == 0 ? 2 : 1, hi = t == 2 ? 2 : 4;
  return ((k & 1) ? lo : 0) | ((k & 2) ? hi : 0) | (k >= 4 ? 1 << t : 0);
}
// the class of component c that class cls of component d couples with
constexpr __host__ __device__ int class_out(int c, int d, int cls) { return c == d ? cls : cls ^ (1 << c) ^ (1 << d); }
constexpr __host__ __device__ int class_size(int cls) { return 8 >> ((cls & 1) + (cls >> 1 & 1) + (cls >> 2 & 1)); }
// j-th mode (x + 3 y + 9 z) of a class
constexpr __host__ __device__ int class_mode(int cls, int j) {
  int m = 0;
  for (int e = 0, t = 1; e < 3; ++e, t *= 3) {
    if (cls >> e & 1) {
      m += 2 * t;
    } else {
      m += (j & 1) * t;
      j >>= 1;
    }
  }
  return m;
}
// Class 0 of the diagonal block: an entry needs a direction in which both modes
// have a derivative (index bit 0 of that direction).  The i-th input: four that
// couple with all outputs, then three with one such direction, each with the four
// outputs that have it too; the constant with none.  Its j-th output
constexpr __host__ __device__ int class0_in(int i) {
  constexpr int in[7] = {0, 1, 2, 4, 3, 5, 6};
  return in[i];
}
constexpr __host__ __device__ int class0_out(int i, int j) {
  return i < 4 ? j : (i == 4 ? j : (i == 5 ? (j & 1) | (j & 2) << 1 : j << 1));
}
// m: mode numbered from direction c on; the same mode numbered from direction 0 on
constexpr __host__ __device__ int mode_from0(int c, int m) {
  constexpr int t[3] = {1, 3, 9};
  return m % 3 * t[c] + m / 3 % 3 * t[(c + 1) % 3] + m / 9 * t[(c + 2) % 3];
}
// m: mode numbered from direction 0 on; the same mode numbered from direction c on
constexpr __host__ __device__ int mode_from(int c, int m) { return mode_from0((3 - c) % 3, m); }
// first lane, over the rows, of class k of block r (input component c + r)
constexpr __host__ __device__ int class_lane(int r, int k) {
  constexpr int diag[8] = {0, 48, 64, 80, 44, 96, 100, 104};
  return r == 0 ? diag[k] : 112 + 80 * (r - 1) + (k < 4 ? 16 * k : 64 + 4 * (k - 4));
}
// first lane of class k in the B^T rows
constexpr __host__ __device__ int bt_lane(int k) {
  constexpr int lane[8] = {0, 8, 12, 16, 20, 22, 24, 26};
  return lane[k];
}

// integrals of a cell's modes
struct CellIntegrals {
  const LevelDesc &L;
  // int d_a phi_m d_b phi_q over the cell
  long double grad(int a, int b, int m, int q) const {
    const int mi[3] = {m % 3, m / 3 % 3, m / 9}, qi[3] = {q % 3, q / 3 % 3, q / 9};
    if (mi[a] == 1 || qi[b] == 1) return 0;
    long double v = (long double)L.vol * L.ih[a] * L.ih[b];
    for (int e = 0; e < L.dim; ++e)
      v *= e == a ? (e == b ? kK[mi[e]][qi[e]] : kD[mi[e]][qi[e]]) : (e == b ? kD[qi[e]][mi[e]] : kM[mi[e]][qi[e]]);
    return v;
  }
  // entry (component c, mode m), (component d, mode q) of the A block at viscosity 1
  long double block(int c, int m, int d, int q) const {
    long double v = grad(d, c, m, q);
    if (c == d)
      for (int e = 0; e < L.dim; ++e) v += grad(e, e, m, q);
    if (L.compressible) v -= 2.0L / 3.0L * grad(c, d, m, q);
    return v;
  }
  // entry of B^T at pressure scaling 1: component c, mode m, pressure mode s
  long double bt(int c, int m, int s) const {
    long double v = -(long double)L.vol * L.ih[c];
    for (int e = 0, t = 1; e < L.dim; ++e, t *= 3) {
      const int i = m / t % 3, j = s >> e & 1;
      v *= e == c ? kPD[i][j] : kPM[i][j];
    }
    return v;
  }
};

void cell_tables2(const CellIntegrals &I, std::vector<long double> &out) {
  out.assign(2 * March2::STRIDE, 0);
  for (int c = 0; c < 2; ++c) {
    long double *at = out.data() + c * March2::STRIDE;
    for (int r = 0; r < 2; ++r)
      for (int q = 0; q < March2::NM; ++q)
        for (int m = 0; m < March2::NM; ++m)
          if (couples2(c, (c + r) % 2, m, q)) *at++ = I.block(c, m, (c + r) % 2, q);
    for (int m = 0; m < March2::NM; ++m) *at++ = I.bt(c, m, pressure_mode2(c, m));
  }
}
void cell_tables3(const CellIntegrals &I, std::vector<long double> &out) {
  out.assign(3 * March3::STRIDE, 0);
  for (int c = 0; c < 3; ++c) {
    long double *const row = out.data() + c * March3::STRIDE;
    for (int r = 0; r < 3; ++r)
      for (int k = 0; k < 8; ++k) {
        const int in = class_at(0, r, k), to = class_out(0, r, in);
        const bool c0 = r == 0 && k == 0;
        long double *at = row + class_lane(r, k);
        for (int i = 0; i < (c0 ? 7 : class_size(in)); ++i)
          for (int o = 0; o < (c0 && i > 3 ? 4 : class_size(to)); ++o)
            *at++ = I.block(c, mode_from0(c, class_mode(to, c0 ? class0_out(i, o) : o)), (c + r) % 3,
                            mode_from0(c, class_mode(in, c0 ? class0_in(i) : i)));
      }
    for (int k = 0; k < 8; ++k) {
      const int cls = class_at(0, 0, k), s = cls ^ 1;  // pressure mode, numbered from direction c on
      for (int j = 0; j < class_size(cls); ++j)
        row[16 * March3::ROWS + bt_lane(k) + j] = I.bt(c, mode_from0(c, class_mode(cls, j)), (s << c | s << c >> 3) & 7);
    }
  }
}

}  // namespace

bool march_level(const LevelDesc &L) { return L.k == 2; }
template <typename T>
std::vector<T> march_tables(const LevelDesc &L0, int n_levels) {
  const CellIntegrals I{L0};
  std::vector<long double> base;
  if (L0.dim == 3)
    cell_tables3(I, base);
  else
    cell_tables2(I, base);
  // cells of the next level have half the extents: powers of two, so that every
  // level's entries are those of its own integrals to the last bit
  const size_t stride = L0.dim == 3 ? March3::STRIDE : March2::STRIDE, bt = stride - (L0.dim == 3 ? 32 : March2::NM);
  std::vector<T> t(base.size() * n_levels);
  T *out = t.data();
  for (int l = 0; l < n_levels; ++l) {
    const long double fa = std::ldexp(1.0L, l * (2 - L0.dim)), fb = std::ldexp(1.0L, l * (1 - L0.dim));
    for (const long double *p = base.data(); p != base.data() + base.size(); p += stride) {
      for (size_t i = 0; i < bt; ++i) *out++ = (T)(p[i] * fa);
      for (size_t i = bt; i < stride; ++i) *out++ = (T)(p[i] * fb);
    }
  }
  return t;
}
template std::vector<double> march_tables<double>(const LevelDesc &, int);
template std::vector<float> march_tables<float>(const LevelDesc &, int);

namespace {

// Coefficients are read through the scalar cache (wave-uniform addresses)
template <typename T>
using CoefPtr = const T __attribute__((address_space(4))) *;

// value of lane (this - 1)
template <typename T>
__device__ __forceinline__ T lane_left(T v) {
  if constexpr (sizeof(T) == 4) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, false));
  } else {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x138, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x138, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
  }
}
// value of the lane whose byte index (4 * lane) is idx
template <typename T>
__device__ __forceinline__ T lane_at(int idx, T v) {
  if constexpr (sizeof(T) == 4) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(idx, __float_as_int(v)));
  } else {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_ds_bpermute(idx, (int)b);
    const int hi = __builtin_amdgcn_ds_bpermute(idx, (int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
  }
}
// Global pointer in scalar registers: addresses then are one scalar base and
// the lane's 32-bit byte offset (the compiler would rather keep a 64-bit sum per offset)
template <typename T>
using Global = T __attribute__((address_space(1))) *;
template <typename T>
__device__ __forceinline__ Global<T> scalar_base(T *p) {
  Global<T> g = (Global<T>)p;
  asm("" : "+s"(g));
  return g;
}
// an offset the compiler may not widen to 64 bits ahead of its use
__device__ __forceinline__ unsigned lane_offset(unsigned off) {
  asm volatile("" : "+v"(off));
  return off;
}
template <typename T>
__device__ __forceinline__ T at(Global<const T> base, unsigned byte_offset, int i = 0) {
  return ((Global<const T>)((Global<const char>)base + byte_offset))[i];
}
template <typename T>
__device__ __forceinline__ void put(Global<T> base, unsigned byte_offset, int i, T v) {
  ((Global<T>)((Global<char>)base + byte_offset))[i] = v;
}

// v where bit k of m is set, else zero (whatever v is)
template <typename T>
__device__ __forceinline__ T keep_if(unsigned m, int k, T v) {
  const int all = (int)(m << (31 - k)) >> 31;
  if constexpr (sizeof(T) == 4)
    return __int_as_float(__float_as_int(v) & all);
  else
    return __longlong_as_double(__double_as_longlong(v) & (long long)all);
}

// modes of three node values a, b, c: a - 2 b + c (zero to the last bit for a
// constant), b, a - c.  As (a - b) + (c - b), exact where the field is smooth, the
// first took one operation more: 3D applies 1 % slower, 2D solves not nearer to the
// 64-bit result than twice (1.5e-14 to 3.6e-14 against 3.5e-14 to 4.2e-14)
template <typename T>
__device__ __forceinline__ void line_modes(T &a, const T b, T &c) {
  const T e = a + c;
  c = a - c;
  a = e - 2 * b;
}
// modes along x and y of a 3 x 3 node plane [3 j + i]
template <typename T>
__device__ __forceinline__ void plane_modes(T (&p)[9]) {
#pragma unroll
  for (int j = 0; j < 3; ++j) line_modes<T>(p[3 * j], p[3 * j + 1], p[3 * j + 2]);
#pragma unroll
  for (int i = 0; i < 3; ++i) line_modes<T>(p[i], p[3 + i], p[6 + i]);
}
// tested modes of a cell's node plane to the sums at the cell's own four nodes
// (i, j in {0, 1}), with the left and lower neighbours' shares
template <typename T>
__device__ __forceinline__ void plane_nodes(const T (&y)[9], int below, T (&o)[2][2]) {
  T n[2][3];  // [i][y mode]
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    n[0][m] = y[3 * m] + y[3 * m + 2] + lane_left<T>(y[3 * m] - y[3 * m + 2]);
    n[1][m] = y[3 * m + 1] - 2 * y[3 * m];
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    o[0][i] = n[i][0] + n[i][2] + lane_at<T>(below, n[i][0] - n[i][2]);
    o[1][i] = n[i][1] - 2 * n[i][0];
  }
}

// acc += coefficient * x with the coefficient taken from lane n of every row of
// 16 lanes of k: a register holds 16 coefficients, which so need no operand of
// their own, no scalar loads (36 dependent ones a layer: 4.5 us instead of
// 1.2) and stay resident over all layers.  A group of them is one asm
// statement, begun by the two wait states that a DPP read of a register needs
// after a VALU write (the compiler may have moved k).
#define MARCH_FMAC(T, m, q, n) \
  "v_fmac_" T "_dpp %[a" #m "], %[k], %[x" #q "] row_newbcast:%c[n" #n "] row_mask:0xf bank_mask:0xf\n"
#define MARCH_ROW8(T, q, n0, n1, n2, n3, n4, n5, n6, n7)                                                          \
  MARCH_FMAC(T, 0, q, n0) MARCH_FMAC(T, 1, q, n1) MARCH_FMAC(T, 2, q, n2) MARCH_FMAC(T, 3, q, n3)                 \
  MARCH_FMAC(T, 4, q, n4) MARCH_FMAC(T, 5, q, n5) MARCH_FMAC(T, 6, q, n6) MARCH_FMAC(T, 7, q, n7)
#define MARCH_ROW4(T, q, n0, n1, n2, n3) \
  MARCH_FMAC(T, 0, q, n0) MARCH_FMAC(T, 1, q, n1) MARCH_FMAC(T, 2, q, n2) MARCH_FMAC(T, 3, q, n3)
#define MARCH_A1 [a0] "+v"(a[0])
#define MARCH_A2 MARCH_A1, [a1] "+v"(a[1])
#define MARCH_A4 MARCH_A2, [a2] "+v"(a[2]), [a3] "+v"(a[3])
#define MARCH_A8 MARCH_A4, [a4] "+v"(a[4]), [a5] "+v"(a[5]), [a6] "+v"(a[6]), [a7] "+v"(a[7])
#define MARCH_X1 [x0] "v"(x[0])
#define MARCH_X2 MARCH_X1, [x1] "v"(x[1])
#define MARCH_X4 MARCH_X2, [x2] "v"(x[2]), [x3] "v"(x[3])
#define MARCH_X8 MARCH_X4, [x4] "v"(x[4]), [x5] "v"(x[5]), [x6] "v"(x[6]), [x7] "v"(x[7])
#define MARCH_N4 [n0] "n"(N), [n1] "n"(N + 1), [n2] "n"(N + 2), [n3] "n"(N + 3)
#define MARCH_N8 MARCH_N4, [n4] "n"(N + 4), [n5] "n"(N + 5), [n6] "n"(N + 6), [n7] "n"(N + 7)
#define MARCH_N16                                                                                                 \
  [n0] "n"(0), [n1] "n"(1), [n2] "n"(2), [n3] "n"(3), [n4] "n"(4), [n5] "n"(5), [n6] "n"(6), [n7] "n"(7),         \
      [n8] "n"(8), [n9] "n"(9), [n10] "n"(10), [n11] "n"(11), [n12] "n"(12), [n13] "n"(13), [n14] "n"(14),        \
      [n15] "n"(15)
// I inputs, O outputs, coefficients from lane N of k on, input by input
template <int I, int O, int N, typename T>
__device__ __forceinline__ void fmac_group(const T k, const T *x, T *a) {
  static_assert((I * O & (I * O - 1)) == 0 && I * O <= 16 && N + I * O <= 16, "groups of a register row");
#define MARCH_GROUP(TY)                                                                                           \
  if constexpr (I == 2 && O == 8)                                                                                 \
    asm("s_nop 1\n" MARCH_ROW8(TY, 0, 0, 1, 2, 3, 4, 5, 6, 7) MARCH_ROW8(TY, 1, 8, 9, 10, 11, 12, 13, 14, 15)     \
        : MARCH_A8                                                                                                \
        : [k] "v"(k), MARCH_X2, MARCH_N16);                                                                       \
  else if constexpr (I == 1 && O == 8)                                                                            \
    asm("s_nop 1\n" MARCH_ROW8(TY, 0, 0, 1, 2, 3, 4, 5, 6, 7) : MARCH_A8 : [k] "v"(k), MARCH_X1, MARCH_N8);       \
  else if constexpr (I == 4 && O == 4)                                                                             \
    asm("s_nop 1\n" MARCH_ROW4(TY, 0, 0, 1, 2, 3) MARCH_ROW4(TY, 1, 4, 5, 6, 7) MARCH_ROW4(TY, 2, 8, 9, 10, 11)   \
            MARCH_ROW4(TY, 3, 12, 13, 14, 15)                                                                     \
        : MARCH_A4                                                                                                \
        : [k] "v"(k), MARCH_X4, MARCH_N16);                                                                       \
  else if constexpr (I == 8 && O == 2)                                                                            \
    asm("s_nop 1\n" MARCH_FMAC(TY, 0, 0, 0) MARCH_FMAC(TY, 1, 0, 1) MARCH_FMAC(TY, 0, 1, 2) MARCH_FMAC(TY, 1, 1, 3) \
            MARCH_FMAC(TY, 0, 2, 4) MARCH_FMAC(TY, 1, 2, 5) MARCH_FMAC(TY, 0, 3, 6) MARCH_FMAC(TY, 1, 3, 7)       \
                MARCH_FMAC(TY, 0, 4, 8) MARCH_FMAC(TY, 1, 4, 9) MARCH_FMAC(TY, 0, 5, 10)                          \
                    MARCH_FMAC(TY, 1, 5, 11) MARCH_FMAC(TY, 0, 6, 12) MARCH_FMAC(TY, 1, 6, 13)                    \
                        MARCH_FMAC(TY, 0, 7, 14) MARCH_FMAC(TY, 1, 7, 15)                                         \
        : MARCH_A2                                                                                                \
        : [k] "v"(k), MARCH_X8, MARCH_N16);                                                                       \
  else if constexpr (I == 1 && O == 4)                                                                            \
    asm("s_nop 1\n" MARCH_ROW4(TY, 0, 0, 1, 2, 3) : MARCH_A4 : [k] "v"(k), MARCH_X1, MARCH_N4);                   \
  else if constexpr (I == 4 && O == 1)                                                                            \
    asm("s_nop 1\n" MARCH_FMAC(TY, 0, 0, 0) MARCH_FMAC(TY, 0, 1, 1) MARCH_FMAC(TY, 0, 2, 2) MARCH_FMAC(TY, 0, 3, 3) \
        : MARCH_A1                                                                                                \
        : [k] "v"(k), MARCH_X4, MARCH_N4);                                                                        \
  else if constexpr (I == 2 && O == 2)                                                                            \
    asm("s_nop 1\n" MARCH_FMAC(TY, 0, 0, 0) MARCH_FMAC(TY, 1, 0, 1) MARCH_FMAC(TY, 0, 1, 2) MARCH_FMAC(TY, 1, 1, 3) \
        : MARCH_A2                                                                                                \
        : [k] "v"(k), MARCH_X2, MARCH_N4);                                                                        \
  else if constexpr (I == 8 && O == 1)                                                                            \
    asm("s_nop 1\n" MARCH_FMAC(TY, 0, 0, 0) MARCH_FMAC(TY, 0, 1, 1) MARCH_FMAC(TY, 0, 2, 2) MARCH_FMAC(TY, 0, 3, 3) \
            MARCH_FMAC(TY, 0, 4, 4) MARCH_FMAC(TY, 0, 5, 5) MARCH_FMAC(TY, 0, 6, 6) MARCH_FMAC(TY, 0, 7, 7)       \
        : MARCH_A1                                                                                                \
        : [k] "v"(k), MARCH_X8, MARCH_N8);                                                                        \
  else if constexpr (I == 1 && O == 2)                                                                            \
    asm("s_nop 1\n" MARCH_FMAC(TY, 0, 0, 0) MARCH_FMAC(TY, 1, 0, 1)                                              \
        : MARCH_A2                                                                                                \
        : [k] "v"(k), MARCH_X1, [n0] "n"(N), [n1] "n"(N + 1));                                                    \
  else if constexpr (I == 2 && O == 1)                                                                            \
    asm("s_nop 1\n" MARCH_FMAC(TY, 0, 0, 0) MARCH_FMAC(TY, 0, 1, 1)                                              \
        : MARCH_A1                                                                                                \
        : [k] "v"(k), MARCH_X2, [n0] "n"(N), [n1] "n"(N + 1));                                                    \
  else                                                                                                            \
    asm("s_nop 1\n" MARCH_FMAC(TY, 0, 0, 0) : MARCH_A1 : [k] "v"(k), MARCH_X1, [n0] "n"(N));
  if constexpr (sizeof(T) == 8) {
    MARCH_GROUP("f64")
  } else {
    MARCH_GROUP("f32")
  }
#undef MARCH_GROUP
}

// Everything below is numbered from the output component's direction on.
// acc += class 0 of the diagonal block
template <int I, typename T>
__device__ __forceinline__ void apply_class0_input(const T k, const T x, T (&acc)[27]) {
  T a[4];
#pragma unroll
  for (int o = 0; o < 4; ++o) a[o] = acc[class_mode(0, class0_out(I, o))];
  fmac_group<1, 4, 4 * (I - 4), T>(k, &x, a);
#pragma unroll
  for (int o = 0; o < 4; ++o) acc[class_mode(0, class0_out(I, o))] = a[o];
}
template <typename T>
__device__ __forceinline__ void apply_class0(const T *k, const T *comp, T (&acc)[27]) {
  T u[7], a[8];
#pragma unroll
  for (int i = 0; i < 7; ++i) u[i] = comp[class_mode(0, class0_in(i)) * 64];
#pragma unroll
  for (int o = 0; o < 8; ++o) a[o] = acc[class_mode(0, o)];
  fmac_group<2, 8, 0, T>(k[0], u, a);
  fmac_group<2, 8, 0, T>(k[1], u + 2, a);
#pragma unroll
  for (int o = 0; o < 8; ++o) acc[class_mode(0, o)] = a[o];
  apply_class0_input<4, T>(k[2], u[4], acc);
  apply_class0_input<5, T>(k[2], u[5], acc);
  apply_class0_input<6, T>(k[2], u[6], acc);
}
// acc += block R of the modes of component R, which are stored numbered from
// direction R on (comp: the column's entries), from class K on; k: coefficients
// by register row
template <int R, int K, typename T>
__device__ __forceinline__ void apply_block(const T *k, const T *comp, T (&acc)[27]) {
  if constexpr (R == 0 && K == 0) {
    apply_class0<T>(k, comp, acc);
  } else {
    constexpr int in = class_at(0, R, K), to = class_out(0, R, in);
    constexpr int I = class_size(in), O = class_size(to), lane = class_lane(R, K);
    T u[I], a[O];
#pragma unroll
    for (int i = 0; i < I; ++i) u[i] = comp[mode_from(R, class_mode(in, i)) * 64];
#pragma unroll
    for (int o = 0; o < O; ++o) a[o] = acc[class_mode(to, o)];
    fmac_group<I, O, lane % 16, T>(k[lane / 16], u, a);
#pragma unroll
    for (int o = 0; o < O; ++o) acc[class_mode(to, o)] = a[o];
  }
  if constexpr (K < 7) apply_block<R, K + 1, T>(k, comp, acc);
}
// acc[m] += b[m] * (pressure mode of its class), from class K on
template <int K, typename T>
__device__ __forceinline__ void add_bt(const T (&b)[2], const T (&ps)[8], T (&acc)[27]) {
  constexpr int cls = class_at(0, 0, K), O = class_size(cls);
  T a[O];
#pragma unroll
  for (int o = 0; o < O; ++o) a[o] = acc[class_mode(cls, o)];
  fmac_group<1, O, bt_lane(K) % 16, T>(b[bt_lane(K) / 16], &ps[cls ^ 1], a);
#pragma unroll
  for (int o = 0; o < O; ++o) acc[class_mode(cls, o)] = a[o];
  if constexpr (K < 7) add_bt<K + 1, T>(b, ps, acc);
}
// acc[pressure mode] += sum b[m] * u[m] over the modes of component C
template <int C, int K, typename T>
__device__ __forceinline__ void add_div(const T (&b)[2], const T (&u)[27], T (&acc)[8]) {
  constexpr int cls = class_at(0, 0, K), I = class_size(cls), s = cls ^ 1;
  T x[I];
#pragma unroll
  for (int i = 0; i < I; ++i) x[i] = u[class_mode(cls, i)];
  fmac_group<I, 1, bt_lane(K) % 16, T>(b[bt_lane(K) / 16], x, &acc[(s << C | s << C >> 3) & 7]);
  if constexpr (K < 7) add_div<C, K + 1, T>(b, u, acc);
}
// modes of a cell from its node planes, to component C's place
template <int C, typename T>
__device__ __forceinline__ void store_modes(const T (&lo)[9], const T (&mid)[9], const T (&hi)[9], T *to) {
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    T a = lo[k], c = hi[k];
    line_modes<T>(a, mid[k], c);
    to[mode_from(C, k) * 64] = a;
    to[mode_from(C, 9 + k) * 64] = mid[k];
    to[mode_from(C, 18 + k) * 64] = c;
  }
}
// tested modes of component C to its node planes: lower (with the share carried
// from the layer below), middle, and the upper one's share to carry on
template <int C, typename T>
__device__ __forceinline__ void split_planes(const T (&acc)[27], T (&y)[2][9], T (&carry)[9]) {
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const T e = acc[mode_from(C, q)], o = acc[mode_from(C, 18 + q)];
    y[0][q] = e + o + carry[q];
    y[1][q] = acc[mode_from(C, 9 + q)] - 2 * e;
    carry[q] = e - o;
  }
}

// LDS barrier that also fences the instruction scheduler: global loads hoisted
// above it would be live across the block products, which need the registers
__device__ __forceinline__ void march_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  lds_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

struct MarchShape {
  int tx, ty, lz;  // cells of a workgroup along x and y (one of each is the low-side halo), owned layers along z
  int ntx, nty;
};

// constrained by a face type on the faces (low, high) of one direction
__device__ __forceinline__ bool face_con(int g, int last, int lo, int hi, bool normal) {
  const int b = g == 0 ? lo : (g == last ? hi : 0);
  return b == 2 || (b == 1 && normal);
}

// the vectors of a finished node, at a plane's base
template <typename T>
struct NodeIO {
  Global<const T> src, rhs, dinv;
  Global<T> dst, d;
};
template <int MODE, typename T>
__device__ __forceinline__ NodeIO<T> node_io(const T *src, const T *rhs, T *dst, const ChebOut<T> &ch, long long base) {
  NodeIO<T> io{};
  io.src = scalar_base(src + base);
  io.dst = scalar_base(dst + base);
  if constexpr (MODE == MODE_RESID || MODE == MARCH_CHEB) io.rhs = scalar_base(rhs + base);
  if constexpr (MODE == MARCH_CHEB) {
    io.dinv = scalar_base(ch.dinv + base);
    io.d = scalar_base(ch.d + base);
  }
  return io;
}
// what a finished node needs besides the operator's value
template <int MODE, typename T>
struct NodeIn {
  T x = 0, rhs = 0, dinv = 0, d = 0;  // MODE_ADD: rhs is dst
  __device__ __forceinline__ void read(const NodeIO<T> &io, unsigned off, int i, const ChebOut<T> &ch) {
    if constexpr (MODE == MODE_RESID || MODE == MARCH_CHEB) rhs = at<T>(io.rhs, off, i);
    if constexpr (MODE == MODE_ADD) rhs = at<T>(io.dst, off, i);
    if constexpr (MODE == MARCH_CHEB) {
      x = at<T>(io.src, off, i);
      dinv = at<T>(io.dinv, off, i);
      if (!ch.first) d = at<T>(io.d, off, i);
    }
  }
};
// val: the operator's value at the node, for a constrained row the source's
template <int MODE, typename T>
__device__ __forceinline__ void finish_node(T val, const NodeIn<MODE, T> &in, const NodeIO<T> &io, unsigned off, int i,
                                            const ChebOut<T> &ch) {
  if constexpr (MODE == MARCH_CHEB) {
    const T r = in.rhs - val;
    const T dd = ch.first ? in.dinv * r * ch.f2 : ch.f1 * in.d + ch.f2 * in.dinv * r;
    put<T>(io.d, off, i, dd);
    put<T>(io.dst, off, i, in.x + dd);
  } else if constexpr (MODE == MODE_SET) {
    put<T>(io.dst, off, i, val);
  } else if constexpr (MODE == MODE_RESID) {
    put<T>(io.dst, off, i, in.rhs - val);
  } else {
    put<T>(io.dst, off, i, in.rhs + val);
  }
}
template <int MODE, typename T>
__device__ __forceinline__ void finish_node(T val, const NodeIO<T> &io, unsigned off, int i, const ChebOut<T> &ch) {
  NodeIn<MODE, T> in;
  in.read(io, off, i, ch);
  finish_node<MODE, T>(val, in, io, off, i, ch);
}

// 3D: a workgroup owns tx - 1 by ty - 1 columns of cells (lane = column, 64
// columns with the halo) and marches lz layers in z; one wave per velocity
// component, and for the Stokes operator a fourth wave for the pressure.  Per
// layer a velocity wave reads the two new node planes of its component and
// forms their modes (the lower plane's are kept from the layer below), writes
// them to LDS for the other waves, applies its own block while they arrive, then
// the other components' blocks; the tested modes of the upper plane are carried
// to the next layer.  The shares of the left and lower columns come by lane
// moves.  A column or layer with index n holds no cell, only the last nodes.
template <bool STOKES, int MODE, typename T>
__global__ void __launch_bounds__(STOKES ? 256 : 192, sizeof(T) == 8 ? 2 : (MODE == MARCH_CHEB ? 3 : 4))
    k_march3(const LevelDesc L, const MarchShape sh, const T *__restrict__ src_u, const T *__restrict__ src_p,
             const T *__restrict__ eta, const T *__restrict__ rhs_u, const T *__restrict__ rhs_p,
             T *__restrict__ dst_u, T *__restrict__ dst_p, const ChebOut<T> ch) {
  constexpr int CT = 64;
  __shared__ T modes[(81 + (STOKES ? 8 : 0)) * CT];
  const int bid = (int)xcd_order(blockIdx.x, gridDim.x);
  const int bx = bid % sh.ntx, by = (bid / sh.ntx) % sh.nty, bz = bid / (sh.ntx * sh.nty);
  const int c = threadIdx.x & (CT - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool act = c < sh.tx * sh.ty;
  const int ly = act ? c / sh.tx : 0, lx = act ? c - ly * sh.tx : 0;
  const int x0 = bx * (sh.tx - 1) - 1, y0 = by * (sh.ty - 1) - 1;
  const int cx = x0 + lx, cy = y0 + ly;
  const int n0 = L.n[0], n1 = L.n[1], n2 = L.n[2];
  const bool own_column = act && lx > 0 && ly > 0 && cx <= n0 && cy <= n1;
  const bool valid = cx >= 0 && cy >= 0 && cx < n0 && cy < n1;
  // a box of columns away from the x and y faces: every column valid, no constrained node in the planes
  const bool interior = x0 >= 1 && y0 >= 1 && x0 + sh.tx <= n0 - 1 && y0 + sh.ty <= n1 - 1;
  const int z0 = bz * sh.lz, z1 = min(z0 + sh.lz, n2 + 1), zs = max(z0 - 1, 0);
  const int below = 4 * ((c - sh.tx) & (CT - 1));
  const T *const kall = static_cast<const T *>(L.kmat) + (c & 15);

  if (STOKES && w == 3) {
    // ---- pressure wave
    const T s = LevelConst<T>::s(L);
    unsigned po[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        po[j][i] = (unsigned)(min(max(cx + i, 0), n0) + (n0 + 1) * min(max(cy + j, 0), n1)) * (unsigned)sizeof(T);
    const long long pplane = (long long)L.np[0] * L.np[1];
    auto load = [&](int gz, T (&p)[4]) {
      Global<const T> base = scalar_base(src_p + pplane * gz);
#pragma unroll
      for (int k = 0; k < 4; ++k) p[k] = at<T>(base, lane_offset(po[k >> 1][k & 1]));
      if (!interior)
#pragma unroll
        for (int k = 0; k < 4; ++k) p[k] = valid ? p[k] : (T)0;
    };
    auto xy = [&](T (&p)[4]) {  // sums and differences along x and y: bit 0 / bit 1 set = odd
      const T a = p[0] + p[1], b = p[0] - p[1], d = p[2] + p[3], e = p[2] - p[3];
      p[0] = a + d;
      p[1] = b + e;
      p[2] = a - d;
      p[3] = b - e;
    };
    T lo[4], hi[4], carry[4] = {0, 0, 0, 0};
    T kb[3][2];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int r = 0; r < 2; ++r) kb[d][r] = kall[d * March3::STRIDE + 16 * (March3::ROWS + r)];
    load(zs, lo);
    xy(lo);
    load(min(zs + 1, n2), hi);
    xy(hi);
    for (int z = zs; z < z1; ++z) {
      T y[4];
      if (z < n2) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          modes[(81 + k) * CT + c] = s * (lo[k] + hi[k]);
          modes[(85 + k) * CT + c] = s * (lo[k] - hi[k]);
          lo[k] = hi[k];
        }
        load(min(z + 2, n2), hi);
        march_barrier();
        T acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        {
          T u[3][27];
#pragma unroll
          for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int m = 0; m < 27; ++m) u[d][m] = modes[(27 * d + m) * CT + c];
          add_div<0, 0, T>(kb[0], u[0], acc);
          add_div<1, 0, T>(kb[1], u[1], acc);
          add_div<2, 0, T>(kb[2], u[2], acc);
        }
        march_barrier();
        xy(hi);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          y[j] = s * (acc[j] + acc[4 + j]) + carry[j];
          carry[j] = s * (acc[j] - acc[4 + j]);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = carry[j];
      }
      if (z >= z0) {
        T n[2];
#pragma unroll
        for (int m = 0; m < 2; ++m)
          n[m] = y[2 * m] + y[2 * m + 1] + lane_left<T>(y[2 * m] - y[2 * m + 1]);
        const T val = n[0] + n[1] + lane_at<T>(below, n[0] - n[1]);
        // (a Chebyshev step has no pressure)
        const NodeIO<T> io = node_io<MODE, T>(src_p, rhs_p, dst_p, ch, pplane * z);
        if (own_column) finish_node<MODE, T>(val, io, lane_offset(po[0][0]), 0, ch);
      }
    }
    return;
  }

  // ---- velocity waves
  const int comp = w;
  // a column without cells reads those of the nearest one (all masked)
  const int ex = min(max(cx, 0), n0 - 1), ey = min(max(cy, 0), n1 - 1);
  unsigned row[3], out[2];  // byte offsets in a plane: first node of the cell's rows, of the column's own rows
#pragma unroll
  for (int j = 0; j < 3; ++j) row[j] = (unsigned)(2 * ex + L.nv[0] * (2 * ey + j)) * (unsigned)sizeof(T);
#pragma unroll
  for (int j = 0; j < 2; ++j) out[j] = (unsigned)(2 * cx + L.nv[0] * (2 * cy + j)) * (unsigned)sizeof(T);
  // bit 3 j + i: node read as stored; bit 9 + 2 j + i: owned node, free in the plane; bit 13 + 2 j + i: owned, constrained
  unsigned bits = 0;
  {
    const int l0 = L.nv[0] - 1, l1 = L.nv[1] - 1;
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int gx = 2 * cx + i, gy = 2 * cy + j;
        const bool cn = face_con(gx, l0, L.bc[0], L.bc[1], comp == 0) ||
                        face_con(gy, l1, L.bc[2], L.bc[3], comp == 1);
        if (valid && !cn) bits |= 1u << (3 * j + i);
        if (i < 2 && j < 2) {
          if (own_column && gx <= l0 && gy <= l1) bits |= 1u << ((cn ? 13 : 9) + 2 * j + i);
        }
      }
  }
  const int lastz = L.nv[2] - 1;
  const bool zlo = L.bc[4] == 2 || (L.bc[4] == 1 && comp == 2), zhi = L.bc[5] == 2 || (L.bc[5] == 1 && comp == 2);
  auto zcon = [&](int gz) { return (gz == 0 && zlo) || (gz == lastz && zhi); };
  const long long plane = (long long)L.nv[0] * L.nv[1], cofs = comp * L.vnodes;
  auto load = [&](int gz, T (&p)[9]) {
    Global<const T> base = scalar_base(src_u + cofs + plane * gz);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const Global<const T> r = (Global<const T>)((Global<const char>)base + lane_offset(row[j]));
#pragma unroll
      for (int i = 0; i < 3; ++i) p[3 * j + i] = r[i];
    }
  };
  auto mask = [&](int gz, T (&p)[9]) {
    if (interior && !zcon(gz)) return;
    const unsigned m = zcon(gz) ? 0u : bits;
#pragma unroll
    for (int k = 0; k < 9; ++k) p[k] = keep_if(m, k, p[k]);
  };
  // tile-blocked viscosity of the column's cells
  const unsigned eofs =
      ((unsigned)((ex >> 2) + L.ntiles[0] * (ey >> 2)) * 64u + (unsigned)((ex & 3) + 4 * (ey & 3))) * (unsigned)sizeof(T);
  const long long etz = (long long)L.ntiles[0] * L.ntiles[1] * 64;
  auto load_eta = [&](int z) { return at<T>(scalar_base(eta + etz * (z >> 2) + 16 * (z & 3)), lane_offset(eofs)); };

  T kc[March3::ROWS], kb[2] = {0, 0};  // the component's coefficients, 16 to a register
#pragma unroll
  for (int r = 0; r < March3::ROWS; ++r) kc[r] = kall[comp * March3::STRIDE + 16 * r];
  if constexpr (STOKES) {
#pragma unroll
    for (int r = 0; r < 2; ++r) kb[r] = kall[comp * March3::STRIDE + 16 * (March3::ROWS + r)];
  }
  T lo[9], mid[9], hi[9], carry[9], et = 0;
#pragma unroll
  for (int k = 0; k < 9; ++k) carry[k] = 0;
  auto to_modes = [&](int z) {  // of the loaded planes 2 z + 1 and 2 z + 2
    mask(2 * z + 1, mid);
    plane_modes(mid);
    mask(2 * z + 2, hi);
    plane_modes(hi);
  };
  if (zs < n2) {
    load(2 * zs, lo);
    load(2 * zs + 1, mid);
    load(2 * zs + 2, hi);
    et = load_eta(zs);
    mask(2 * zs, lo);
    plane_modes(lo);
    to_modes(zs);
  }
  const T *const comp0 = modes + w * 27 * CT + c, *const comp1 = modes + (w == 2 ? 0 : w + 1) * 27 * CT + c,
                 *const comp2 = modes + (w == 0 ? 2 : w - 1) * 27 * CT + c;
  for (int z = zs; z < z1; ++z) {
    T y[2][9];
    if (z < n2) {
      const T e = valid ? et : (T)0;
      if (w == 0)
        store_modes<0, T>(lo, mid, hi, modes + c);
      else if (w == 1)
        store_modes<1, T>(lo, mid, hi, modes + 27 * CT + c);
      else
        store_modes<2, T>(lo, mid, hi, modes + 54 * CT + c);
#pragma unroll
      for (int k = 0; k < 9; ++k) lo[k] = hi[k];
      // the next layer's planes, in flight during the block products and
      // complete before this layer's stores are issued (a wait for a load
      // waits for the stores before it)
      const int zn = min(z + 1, n2 - 1);
      load(2 * zn + 1, mid);
      load(2 * zn + 2, hi);
      et = load_eta(zn);
      march_barrier();
      T acc[27];
#pragma unroll
      for (int m = 0; m < 27; ++m) acc[m] = 0;
      apply_block<0, 0, T>(kc, comp0, acc);
      apply_block<1, 0, T>(kc, comp1, acc);
      apply_block<2, 0, T>(kc, comp2, acc);
#pragma unroll
      for (int m = 0; m < 27; ++m) acc[m] *= e;
      if constexpr (STOKES) {
        T ps[8];  // pressure modes, numbered from direction w on
#pragma unroll
        for (int m = 0; m < 8; ++m) ps[m] = modes[(81 + ((m << w | m << w >> 3) & 7)) * CT + c];
        add_bt<0, T>(kb, ps, acc);
      }
      march_barrier();
      if (w == 0)
        split_planes<0, T>(acc, y, carry);
      else if (w == 1)
        split_planes<1, T>(acc, y, carry);
      else
        split_planes<2, T>(acc, y, carry);
    } else {
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        y[0][k] = carry[k];
        y[1][k] = 0;
      }
    }
    if (z < z0) {  // the halo layer's own planes belong to the workgroup below
      to_modes(z + 1);
      continue;
    }
    // the nodes' other operands, in flight while their sums are formed
    const unsigned ofs[2] = {lane_offset(out[0]), lane_offset(out[1])};
    NodeIO<T> io[2];
    NodeIn<MODE, T> in[2][4];
    bool writes[2];  // the plane exists and is free in this component
    auto read_plane = [&](int kk) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (bits >> (9 + q) & 1) in[kk][q].read(io[kk], ofs[q >> 1], q & 1, ch);
    };
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int gz = min(2 * z + kk, lastz);
      writes[kk] = 2 * z + kk <= lastz && !zcon(gz);
      io[kk] = node_io<MODE, T>(src_u, rhs_u, dst_u, ch, cofs + plane * gz);
    }
    constexpr bool BOTH = MODE != MARCH_CHEB || sizeof(T) == 4;  // registers for the operands of both planes
    if constexpr (BOTH) {
      read_plane(0);
      read_plane(1);
    }
    if (z + 1 < z1) to_modes(min(z + 1, n2 - 1));
    if constexpr (!BOTH) {
      __builtin_amdgcn_sched_barrier(0);
      read_plane(0);
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      T o[2][2];
      plane_nodes(y[kk], below, o);
      if (!writes[kk]) {
      } else if (interior) {
        if (own_column)
#pragma unroll
          for (int q = 0; q < 4; ++q) finish_node<MODE, T>(o[q >> 1][q & 1], in[kk][q], io[kk], ofs[q >> 1], q & 1, ch);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (bits >> (9 + q) & 1)
            finish_node<MODE, T>(o[q >> 1][q & 1], in[kk][q], io[kk], ofs[q >> 1], q & 1, ch);
      }
      if constexpr (!BOTH) {
        __builtin_amdgcn_sched_barrier(0);
        if (kk == 0) read_plane(1);
      }
    }
  }
  // constrained rows are identity rows (outside the march: their source values
  // are loads that nothing else waits for)
  for (int gz = 2 * z0; gz < min(2 * z1, lastz + 1); ++gz) {
    const bool zc = zcon(gz);
    if (interior && !zc) continue;
    const unsigned rows = bits >> 13 | (zc ? bits >> 9 : 0u);
    const NodeIO<T> io = node_io<MODE, T>(src_u, rhs_u, dst_u, ch, cofs + plane * gz);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (rows >> q & 1) finish_node<MODE, T>(at<T>(io.src, out[q >> 1], q & 1), io, out[q >> 1], q & 1, ch);
  }
}

// 2D: one wave per box of cells (lane = cell), both components and the
// pressure in the lane's registers.
template <bool STOKES, int MODE, typename T>
__global__ void __launch_bounds__(64)
    k_march2(const LevelDesc L, const MarchShape sh, const T *__restrict__ src_u, const T *__restrict__ src_p,
             const T *__restrict__ eta, const T *__restrict__ rhs_u, const T *__restrict__ rhs_p,
             T *__restrict__ dst_u, T *__restrict__ dst_p, const ChebOut<T> ch) {
  constexpr int NM = March2::NM, CT = 64;
  const int bid = (int)xcd_order(blockIdx.x, gridDim.x);
  const int bx = bid % sh.ntx, by = bid / sh.ntx;
  const int c = threadIdx.x;
  const bool act = c < sh.tx * sh.ty;
  const int ly = act ? c / sh.tx : 0, lx = act ? c - ly * sh.tx : 0;
  const int cx = bx * (sh.tx - 1) - 1 + lx, cy = by * (sh.ty - 1) - 1 + ly;
  const int n0 = L.n[0], n1 = L.n[1], l0 = L.nv[0] - 1, l1 = L.nv[1] - 1;
  const bool own = act && lx > 0 && ly > 0 && cx <= n0 && cy <= n1;
  const bool valid = cx >= 0 && cy >= 0 && cx < n0 && cy < n1;
  const int below = 4 * ((c - sh.tx) & (CT - 1));
  CoefPtr<T> k = (CoefPtr<T>)(uintptr_t)L.kmat;
  unsigned vo[3][3];
  unsigned con[2] = {0, 0};  // bit 3 j + i: constrained node
  T u[2][9];
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int gx = 2 * cx + i, gy = 2 * cy + j;
      vo[j][i] = (unsigned)(min(max(gx, 0), l0) + L.nv[0] * min(max(gy, 0), l1)) * (unsigned)sizeof(T);
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        u[d][3 * j + i] = at<T>((Global<const T>)(src_u + d * L.vnodes), vo[j][i]);
        if (face_con(gx, l0, L.bc[0], L.bc[1], d == 0) || face_con(gy, l1, L.bc[2], L.bc[3], d == 1))
          con[d] |= 1u << (3 * j + i);
      }
    }
  unsigned po[2][2];
  T p[4];
  if constexpr (STOKES) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      po[q >> 1][q & 1] = (unsigned)(min(max(cx + (q & 1), 0), n0) + (n0 + 1) * min(max(cy + (q >> 1), 0), n1)) *
                          (unsigned)sizeof(T);
      p[q] = at<T>((Global<const T>)src_p, po[q >> 1][q & 1]);
    }
  }
  const int ex = min(max(cx, 0), n0 - 1), ey = min(max(cy, 0), n1 - 1);
  const T er = eta[((unsigned)(ex >> 3) + (unsigned)L.ntiles[0] * (unsigned)(ey >> 3)) * 64u +
                   (unsigned)((ex & 7) + 8 * (ey & 7))];
  const T e = valid ? er : (T)0;
  T raw[2][4];  // the owned nodes as stored
#pragma unroll
  for (int d = 0; d < 2; ++d) {
#pragma unroll
    for (int q = 0; q < 4; ++q) raw[d][q] = u[d][3 * (q >> 1) + (q & 1)];
#pragma unroll
    for (int q = 0; q < 9; ++q) u[d][q] = valid && !(con[d] >> q & 1) ? u[d][q] : (T)0;
    plane_modes(u[d]);
  }
  const T s = LevelConst<T>::s(L);
  T ps[4] = {0, 0, 0, 0}, pt[4] = {0, 0, 0, 0};
  if constexpr (STOKES) {
#pragma unroll
    for (int q = 0; q < 4; ++q) p[q] = valid ? s * p[q] : (T)0;
    const T a = p[0] + p[1], b = p[0] - p[1], d = p[2] + p[3], f = p[2] - p[3];
    ps[0] = a + d;
    ps[1] = b + f;
    ps[2] = a - d;
    ps[3] = b - f;
  }
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    T acc[9];
#pragma unroll
    for (int m = 0; m < NM; ++m) acc[m] = 0;
    int n = d * March2::STRIDE;
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int q = 0; q < NM; ++q)
#pragma unroll
        for (int m = 0; m < NM; ++m)
          if (couples2(d, (d + r) % 2, m, q)) acc[m] += k[n++] * u[(d + r) % 2][q];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      if constexpr (STOKES) {
        const T b = k[n + m];
        acc[m] = e * acc[m] + b * ps[pressure_mode2(d, m)];
        pt[pressure_mode2(d, m)] += b * u[d][m];
      } else {
        acc[m] *= e;
      }
    }
    T o[2][2];
    plane_nodes(acc, below, o);
    const NodeIO<T> io = node_io<MODE, T>(src_u, rhs_u, dst_u, ch, d * L.vnodes);
    if (own) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (2 * cx + (q & 1) <= l0 && 2 * cy + (q >> 1) <= l1) {
          const T val = con[d] >> (3 * (q >> 1) + (q & 1)) & 1 ? raw[d][q] : o[q >> 1][q & 1];
          finish_node<MODE, T>(val, io, vo[q >> 1][q & 1], 0, ch);
        }
    }
  }
  if constexpr (STOKES) {
    T n[2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
      n[m] = pt[2 * m] + pt[2 * m + 1] + lane_left<T>(pt[2 * m] - pt[2 * m + 1]);
    const T val = s * (n[0] + n[1] + lane_at<T>(below, n[0] - n[1]));
    const NodeIO<T> io = node_io<MODE, T>(src_p, rhs_p, dst_p, ch, 0);
    if (own) finish_node<MODE, T>(val, io, lane_offset(po[0][0]), 0, ch);
  }
}

// Shape of a launch: the box of at most 64 columns that needs fewest boxes,
// and in 3D the layers of a march.  More layers mean fewer halo layers (one
// per march) but fewer workgroups: the rule takes the least
// (rounds of workgroups) x (layers + start), rounds rounded up while they are
// few, at 2 (FP64) or 4 (FP32) workgroups per CU and up to 11 or 6 layers.
// Measured A-block applies, layers taken against the best and one layer: 32^3
// FP64 16.1 (2 layers) and 20.3 us, 64^3 72 and 109, 128^3 404 and 716; FP32
// 12.2 (1), 41 (4) and 55, 211 (6) and 314 us.
MarchShape march_shape(const LevelDesc &L, size_t elem) {
  MarchShape s{};
  long long best = -1;
  for (int tx = 3; tx <= 21; ++tx) {
    const int ty = 64 / tx;
    const long long nt = (long long)((L.n[0] + tx - 1) / (tx - 1)) * ((L.n[1] + ty - 1) / (ty - 1));
    if (best < 0 || nt <= best) {
      best = nt;
      s.tx = tx;
      s.ty = ty;
    }
  }
  s.ntx = (L.n[0] + s.tx - 1) / (s.tx - 1);  // columns 0 .. n
  s.nty = (L.n[1] + s.ty - 1) / (s.ty - 1);
  s.lz = 1;
  if (L.dim == 2) return s;
  const double slots = elem == 8 ? 512.0 : 1024.0;
  double least = 0;
  for (const int lz : {1, 2, 3, 4, 6, 8, 11}) {
    if (lz > (elem == 8 ? 11 : 6)) break;
    const double wg = (double)best * ((L.n[2] + lz) / lz), r = wg / slots;
    const double cost = (r < 3 ? std::ceil(r) : r + 0.5) * (lz + 1.5);
    if (lz == 1 || cost < least) {
      least = cost;
      s.lz = lz;
    }
  }
  return s;
}

template <bool STOKES, int MODE, typename T>
void launch_march_m(const LevelDesc &L, const T *su, const T *sp, const T *eta, const T *ru, const T *rp, T *du, T *dp,
                    const ChebOut<T> &ch, hipStream_t st) {
  const MarchShape sh = march_shape(L, sizeof(T));
  if (L.dim == 3) {
    const long long nb = (long long)sh.ntx * sh.nty * ((L.n[2] + sh.lz) / sh.lz);  // layers 0 .. n
    hipLaunchKernelGGL((k_march3<STOKES, MODE, T>), dim3((unsigned)nb), dim3(STOKES ? 256 : 192), 0, st, L, sh, su, sp,
                       eta, ru, rp, du, dp, ch);
  } else {
    hipLaunchKernelGGL((k_march2<STOKES, MODE, T>), dim3((unsigned)(sh.ntx * sh.nty)), dim3(64), 0, st, L, sh, su, sp,
                       eta, ru, rp, du, dp, ch);
  }
  MFS_HIP(hipGetLastError());
}

// in [a, a + n) and [b, b + n): does a workgroup write what another one still reads?
template <typename T>
bool overlap(const T *a, const T *b, long long n) {
  return a < b + n && b < a + n;
}

}  // namespace

// what the kernels assume: degree 2 on a uniform box with its cell matrices in
// this precision, one viscosity per cell, constrained values read as zero,
// byte offsets in a plane and viscosity indices in 32 bits
template <typename T>
bool march_fits(const LevelDesc &L, int eta_per_qp) {
  return L.k == 2 && !L.geo && !L.plain_read && !eta_per_qp && L.kmat && L.kmat_size == (int)sizeof(T) &&
         (long long)L.nv[0] * L.nv[1] * (long long)sizeof(T) < (1LL << 31) && L.ntiles_total < (1LL << 24);
}
template bool march_fits<double>(const LevelDesc &, int);
template bool march_fits<float>(const LevelDesc &, int);

template <typename T>
bool launch_march(Op op, Mode mode, const LevelDesc &L, const T *su, const T *sp, const T *eta, int eta_per_qp,
                  const T *ru, const T *rp, T *du, T *dp, hipStream_t st) {
  if ((op != OP_STOKES && op != OP_ABLOCK) || !march_fits<T>(L, eta_per_qp)) return false;
  if (overlap<T>(su, du, L.dim * L.vnodes) || (op == OP_STOKES && overlap<T>(sp, dp, L.pnodes))) return false;
  const ChebOut<T> no{};
  auto go = [&](auto stokes) {
    constexpr bool S = decltype(stokes)::value;
    if (mode == MODE_SET)
      launch_march_m<S, MODE_SET, T>(L, su, sp, eta, ru, rp, du, dp, no, st);
    else if (mode == MODE_RESID)
      launch_march_m<S, MODE_RESID, T>(L, su, sp, eta, ru, rp, du, dp, no, st);
    else
      launch_march_m<S, MODE_ADD, T>(L, su, sp, eta, ru, rp, du, dp, no, st);
  };
  if constexpr (std::is_same<T, double>::value) {
    if (op == OP_STOKES) {
      go(std::true_type());
      return true;
    }
  }
  if (op == OP_STOKES) return false;
  go(std::false_type());
  return true;
}
template <typename T>
bool launch_march_cheb(const LevelDesc &L, const T *xin, const T *b, const T *eta, int eta_per_qp, const T *dinv, T *d,
                       T *xout, T f1, T f2, int first, hipStream_t st) {
  if (!march_fits<T>(L, eta_per_qp)) return false;
  if (xin == xout) throw std::runtime_error("launch_march_cheb: x_in and x_out must differ");
  const ChebOut<T> ch{dinv, d, f1, f2, first};
  launch_march_m<false, MARCH_CHEB, T>(L, xin, nullptr, eta, b, nullptr, xout, nullptr, ch, st);
  return true;
}
template bool launch_march<double>(Op, Mode, const LevelDesc &, const double *, const double *, const double *, int,
                                   const double *, const double *, double *, double *, hipStream_t);
template bool launch_march<float>(Op, Mode, const LevelDesc &, const float *, const float *, const float *, int,
                                  const float *, const float *, float *, float *, hipStream_t);
template bool launch_march_cheb<double>(const LevelDesc &, const double *, const double *, const double *, int,
                                        const double *, double *, double *, double, double, int, hipStream_t);
template bool launch_march_cheb<float>(const LevelDesc &, const float *, const float *, const float *, int,
                                       const float *, float *, float *, float, float, int, hipStream_t);

}  // namespace mfs
