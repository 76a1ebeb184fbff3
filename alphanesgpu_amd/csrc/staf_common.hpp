// Shared device/host helpers of the gfx950 STAF kernels.
//
// One templated source serves fp32 and fp64: every kernel is a template on
// `real` and the extern "C" entry points instantiate it twice (_f32/_f64).
// Wavefronts are 64 lanes wide; all cross-lane reductions below use a fixed
// butterfly tree, so a sum's rounding does not depend on scheduling.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <unordered_map>
#include <vector>

#include "../../include/staf_ops.h"

namespace staf {

constexpr int WAVE = 64;
constexpr int NT_MAX = 8;  // species supported by the per-type bookkeeping

template <typename real> struct Vec2;
template <> struct Vec2<float> { using type = float2; };
template <> struct Vec2<double> { using type = double2; };
// 16 bytes of reals: the widest LDS and global access
template <typename real> struct Vec16;
template <> struct Vec16<float> { using type = float4; };
template <> struct Vec16<double> { using type = double2; };
template <typename real> struct Vec4;
template <> struct Vec4<float> { using type = float4; };
template <> struct Vec4<double> { using type = double4; };

// The reference's value of pi (STAF/src/descriptor_builder/reforce.cu.cc:15).
template <typename real> __host__ __device__ inline real pi_ref() { return real(3.141592654); }

__device__ inline float r_exp(float x) { return expf(x); }
__device__ inline double r_exp(double x) { return exp(x); }
__device__ inline float r_cos(float x) { return cosf(x); }
__device__ inline double r_cos(double x) { return cos(x); }
__device__ inline float r_sin(float x) { return sinf(x); }
__device__ inline double r_sin(double x) { return sin(x); }
__device__ inline void r_sincos(float x, float* s, float* c) { sincosf(x, s, c); }
__device__ inline void r_sincos(double x, double* s, double* c) { sincos(x, s, c); }
// sin and cos of an argument in [0, pi] (the cutoff functions' pi r / Rc, r < Rc): reduction by a multiple of pi/2 in
// two parts, then the polynomials of fdlibm's kernel_sin / kernel_cos on [-pi/4, pi/4].  Maximum error 1.1e-16
// absolute over the range against the C library's sin and cos; an eighth of the instructions of the general routine,
// which has to cope with any argument.  Single precision keeps the library routine.
__device__ inline void r_sincos_0pi(float x, float* s, float* c) { sincosf(x, s, c); }
__device__ inline void r_sincos_0pi(double x, double* sn, double* cs) {
  const double k = rint(x * 0.63661977236758134308);
  double y = fma(-k, 1.57079632673412561417e+00, x);
  y = fma(-k, 6.07710050650619224932e-11, y);
  const double z = y * y;
  double ps = 1.58969099521155010221e-10;
  ps = fma(ps, z, -2.50507602534068634195e-08);
  ps = fma(ps, z, 2.75573137070700676789e-06);
  ps = fma(ps, z, -1.98412698298579493134e-04);
  ps = fma(ps, z, 8.33333333332248946124e-03);
  ps = fma(ps, z, -1.66666666666666324348e-01);
  const double s = fma(y * z, ps, y);
  double pc = -1.13596475577881948265e-11;
  pc = fma(pc, z, 2.08757232129817482790e-09);
  pc = fma(pc, z, -2.75573143513906633035e-07);
  pc = fma(pc, z, 2.48015872894767294178e-05);
  pc = fma(pc, z, -1.38888888888741095749e-03);
  pc = fma(pc, z, 4.16666666666666019037e-02);
  const double c = 1.0 - (0.5 * z - z * z * pc);
  const int q = (int)k;   // 0, 1 or 2
  *sn = q == 0 ? s : (q == 1 ? c : -s);
  *cs = q == 0 ? c : (q == 1 ? -s : -c);
}
__device__ inline float r_sqrt(float x) { return sqrtf(x); }
__device__ inline double r_sqrt(double x) { return sqrt(x); }
__device__ inline float r_pow(float x, float n) { return powf(x, n); }
__device__ inline double r_pow(double x, double n) { return pow(x, n); }
__device__ inline float r_rint(float x) { return rintf(x); }
__device__ inline double r_rint(double x) { return rint(x); }
__device__ inline float r_floor(float x) { return floorf(x); }
__device__ inline double r_floor(double x) { return floor(x); }
__device__ inline float r_fma(float a, float b, float c) { return fmaf(a, b, c); }
__device__ inline double r_fma(double a, double b, double c) { return fma(a, b, c); }

__device__ inline int lane_id() { return threadIdx.x & (WAVE - 1); }

// Butterfly all-reduce over the 64 lanes of a wave; every lane returns the sum.
template <typename T>
__device__ inline T wave_sum(T v) {
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
  return v;
}
// Data-parallel-primitive lane moves: lane l receives the value of another lane of its row of 16 (or of the
// previous rows for the broadcasts); lanes without a source receive 0.
template <int CTRL, int ROW_MASK>
__device__ inline float dpp_get(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xf, false));
}
template <int CTRL, int ROW_MASK>
__device__ inline unsigned dpp_get(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
}
// Doubles move in two halves.  The hardware writes the 0 itself for a lane without a source (bound_ctrl) as long as every
// row takes part; a result that starts as a register holding 0 costs two more moves per value.
template <int CTRL>
__device__ inline double dpp_row(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// The same with rows that take no part: they keep `keep`, which holds 0 there.  The result serves as `keep` of the next
// value, so that a sequence of moves needs one pair of zeroes.
template <int CTRL, int ROW_MASK>
__device__ inline double dpp_rows(double keep, double v) {
  const long long b = __double_as_longlong(v), k = __double_as_longlong(keep);
  const int lo = __builtin_amdgcn_update_dpp((int)(k & 0xffffffffll), (int)(b & 0xffffffffll), CTRL, ROW_MASK, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(k >> 32), (int)(b >> 32), CTRL, ROW_MASK, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// The two steps that carry a prefix across the rows of 16 lanes: s += (lane 15 of the row before) in rows 1 and 3,
// then s += (lane 31) in rows 2 and 3.  Written as `s += dpp_get<..>(s)` each costs a zero, a move and an add,
// because the rows that receive nothing need a 0 to add; as one add whose result is written in the selected rows
// only (the others keep s) it is a single instruction.  Single precision only: the lane moves are 32 bits wide.
// A lane move reads a register two cycles after the instruction that wrote it at the earliest: the idle cycles
// stand in front of the moves, and behind them for whatever lane operation follows.
__device__ inline void dpp_rows_carry(float& a) {
  asm("s_nop 1\n\t"
      "v_add_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa\n\t"
      "s_nop 1\n\t"
      "v_add_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc\n\t"
      "s_nop 1"
      : "+v"(a));
}
__device__ inline void dpp_rows_carry(float& a, float& b, float& c, float& d) {
  asm("s_nop 1\n\t"
      "v_add_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa\n\t"
      "v_add_f32_dpp %1, %1, %1 row_bcast:15 row_mask:0xa\n\t"
      "v_add_f32_dpp %2, %2, %2 row_bcast:15 row_mask:0xa\n\t"
      "v_add_f32_dpp %3, %3, %3 row_bcast:15 row_mask:0xa\n\t"
      "v_add_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc\n\t"
      "v_add_f32_dpp %1, %1, %1 row_bcast:31 row_mask:0xc\n\t"
      "v_add_f32_dpp %2, %2, %2 row_bcast:31 row_mask:0xc\n\t"
      "v_add_f32_dpp %3, %3, %3 row_bcast:31 row_mask:0xc\n\t"
      "s_nop 1"
      : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}
__device__ inline void dpp_rows_carry(unsigned& a) {
  asm("s_nop 1\n\t"
      "v_add_u32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa\n\t"
      "s_nop 1\n\t"
      "v_add_u32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc\n\t"
      "s_nop 1"
      : "+v"(a));
}
__device__ inline void dpp_rows_carry(double& s) {
  s += dpp_rows<0x142, 0xa>(0.0, s);   // lane 15 of a row -> every lane of the next row (rows 1 and 3 take it)
  s += dpp_rows<0x143, 0xc>(0.0, s);   // lane 31 -> rows 2 and 3
}
// several values, step by step: the moves of one fill the wait states of the others
template <int N>
__device__ inline void dpp_rows_carry(double (&s)[N]) {
  double t = 0;
#pragma unroll
  for (int c = 0; c < N; c++) { t = dpp_rows<0x142, 0xa>(t, s[c]); s[c] += t; }
  t = 0;
#pragma unroll
  for (int c = 0; c < N; c++) { t = dpp_rows<0x143, 0xc>(t, s[c]); s[c] += t; }
}

// Inclusive prefix sums over the 64 lanes with register-to-register lane moves only, of N values at once: inside each
// row of 16, then row 0->1, 2->3, and rows 0-1 -> 2-3.  Single precision: prefix steps 1, 2, 3 of the value itself, then 4
// and 8 of the sum (an add takes its move along, and this is the shorter chain); double precision: 1, 2, 4 and 8 of the sum
// (a step is two moves and an add).
template <int N>
__device__ inline void wave_scan(float (&v)[N]) {
  float s[N];
#pragma unroll
  for (int c = 0; c < N; c++) s[c] = v[c] + dpp_get<0x111, 0xf>(v[c]);
#pragma unroll
  for (int c = 0; c < N; c++) s[c] += dpp_get<0x112, 0xf>(v[c]);
#pragma unroll
  for (int c = 0; c < N; c++) s[c] += dpp_get<0x113, 0xf>(v[c]);
#pragma unroll
  for (int c = 0; c < N; c++) s[c] += dpp_get<0x114, 0xf>(s[c]);
#pragma unroll
  for (int c = 0; c < N; c++) s[c] += dpp_get<0x118, 0xf>(s[c]);
  if constexpr (N == 4) {
    dpp_rows_carry(s[0], s[1], s[2], s[3]);
  } else {
#pragma unroll
    for (int c = 0; c < N; c++) dpp_rows_carry(s[c]);
  }
#pragma unroll
  for (int c = 0; c < N; c++) v[c] = s[c];
}
template <int N>
__device__ inline void wave_scan(double (&s)[N]) {
#pragma unroll
  for (int c = 0; c < N; c++) s[c] += dpp_row<0x111>(s[c]);
#pragma unroll
  for (int c = 0; c < N; c++) s[c] += dpp_row<0x112>(s[c]);
#pragma unroll
  for (int c = 0; c < N; c++) s[c] += dpp_row<0x114>(s[c]);
#pragma unroll
  for (int c = 0; c < N; c++) s[c] += dpp_row<0x118>(s[c]);
  dpp_rows_carry(s);
}
// Sum over the 64 lanes by the same steps; the total is valid in lane 63 alone.
template <typename T>
__device__ inline T wave_sum_to_last(T v) {
  if constexpr (sizeof(T) == 8) {
    double s[1] = {v};
    wave_scan(s);
    return s[0];
  } else {
    T s = v + dpp_get<0x111, 0xf>(v);
    s += dpp_get<0x112, 0xf>(v);
    s += dpp_get<0x113, 0xf>(v);
    s += dpp_get<0x114, 0xf>(s);
    s += dpp_get<0x118, 0xf>(s);
    dpp_rows_carry(s);
    return s;
  }
}
// Sums over the 64 lanes of twelve values: halves of the lanes trade values until a row of sixteen lanes holds one value of
// four, then three prefix sums in the rows (63 instructions for doubles where twelve of wave_scan are 216).  The sum of
// v[4 q + place] is v[q] of the last lane of row 0, 2, 1, 3 for place 0, 1, 2, 3.
__device__ inline void lanes_trade32(double& a, double& b) {
  const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  a = __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0]));
  b = __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}
__device__ inline void lanes_trade16(double& a, double& b) {
  const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  a = __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0]));
  b = __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}
__device__ inline void lanes_trade32(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]); b = __uint_as_float(r[1]);
}
__device__ inline void lanes_trade16(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]); b = __uint_as_float(r[1]);
}
template <typename T>
__device__ inline void wave_sums12(T (&v)[12]) {
#pragma unroll
  for (int p = 0; p < 6; p++) { lanes_trade32(v[2 * p], v[2 * p + 1]); v[p] = v[2 * p] + v[2 * p + 1]; }
#pragma unroll
  for (int q = 0; q < 3; q++) { lanes_trade16(v[2 * q], v[2 * q + 1]); v[q] = v[2 * q] + v[2 * q + 1]; }
#pragma unroll
  for (int q = 0; q < 3; q++) {
    if constexpr (sizeof(T) == 8) {
      v[q] += dpp_row<0x111>(v[q]);
      v[q] += dpp_row<0x112>(v[q]);
      v[q] += dpp_row<0x114>(v[q]);
      v[q] += dpp_row<0x118>(v[q]);
    } else {
      T s = v[q] + dpp_get<0x111, 0xf>(v[q]);
      s += dpp_get<0x112, 0xf>(v[q]);
      s += dpp_get<0x113, 0xf>(v[q]);
      s += dpp_get<0x114, 0xf>(s);
      s += dpp_get<0x118, 0xf>(s);
      v[q] = s;
    }
  }
}
// Wave-uniform value loaded through a vector path (e.g. from LDS) moved to a scalar register, so that loop
// bounds and addresses derived from it stay scalar.
__device__ inline int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ inline int wave_max(int v) {
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, WAVE));
  return v;
}

// Index arithmetic of the hot kernels uses the 24-bit multiplier (full rate; the 32-bit integer multiply takes
// four times as long): operands here are slot, species and channel counts far below 2^23.
__device__ inline int mul24(int a, int b) { return __mul24(a, b); }

// First flat index of row j in the row-major upper triangle over m items
// (pairs j<k): the reference's triplet numbering,
// STAF/src/descriptor_builder/reforce.cu.cc:137-146.  j m - j (j + 1) / 2 = j (2 m - 1 - j) / 2, m <= 2048.
__device__ inline int tri_rowstart(int j, int m) { return mul24(j, 2 * m - 1 - j) >> 1; }

// Inverse of the numbering: nn -> (j,k), 0 <= nn < m(m-1)/2, m <= 2048.
// With t = 2m - 1 the row is j = floor((t - sqrt(t^2 - 8 nn)) / 2); the root is an integer exactly at a row's first
// pair, where a rounding error would decide the row.
// m <= 255: the root is taken of t^2 - 8 nn - 4 instead, which moves the quotient 1/(t - 2j) >= 0.002 away from the
// integers on either side (up at a row's first pair, down at the last pair of the row before) -- sixty times the
// error of the single-precision root and subtraction, so the truncation is the row and no correction step follows
// (checked for every m <= 255 and every nn, with the root off by up to two units in the last place).
// m > 255: the hardware square root (1 ulp) puts the row estimate within one of the exact row (two steps each way
// are taken); the row start follows the row in steps of the row length m - 1 - j, so that the comparisons with the
// exact integer row starts cost no multiply.
__device__ inline void tri_decode(int nn, int m, int& j, int& k) {
  const int t = 2 * m - 1;
  if (m <= 255) {
    const int jj = (int)(((float)t - __builtin_amdgcn_sqrtf((float)(mul24(t, t) - 4 - 8 * nn))) * 0.5f);
    j = jj;
    k = nn - (mul24(jj, t - jj) >> 1) + jj + 1;
    return;
  }
  int jj = (int)(((float)t - __builtin_amdgcn_sqrtf((float)(mul24(t, t) - 8 * nn))) * 0.5f);
  jj = jj < 0 ? 0 : (jj > m - 2 ? m - 2 : jj);
  int rs = mul24(jj, t - jj) >> 1;
#pragma unroll
  for (int it = 0; it < 2; it++) {   // row 0 starts at 0 <= nn: never stepped below
    const bool down = rs > nn;
    rs = down ? rs - (m - jj) : rs;
    jj = down ? jj - 1 : jj;
  }
#pragma unroll
  for (int it = 0; it < 2; it++) {   // the row after row m - 2 would start at m (m - 1) / 2 > nn: never stepped to
    const int next = rs + (m - 1 - jj);
    const bool up = next <= nn;
    rs = up ? next : rs;
    jj = up ? jj + 1 : jj;
  }
  j = jj;
  k = nn - rs + jj + 1;
}

// Minimum-image Cartesian separation r_i - r_j from Cartesian positions and
// box6 = [Lx, xy, xz, Ly, yz, Lz]: cart -> frac, rint, back to cart
// (STAF/include/staf_force_pbc.cuh:16-49; used by the virial forms only).  skip_pbc: no wrap, the neighbour
// already carries its periodic image (staf_force_skip_pbc there).
template <typename real>
__device__ inline void mic_cart_from_cart(const real* pi, const real* pj, const real* bx, int skip_pbc, real* d) {
  const real i0 = real(1) / bx[0];
  const real i1 = -bx[1] / (bx[0] * bx[3]);
  const real i2 = (bx[1] * bx[4]) / (bx[0] * bx[3] * bx[5]) - bx[2] / (bx[0] * bx[5]);
  const real i3 = real(1) / bx[3];
  const real i4 = -bx[4] / (bx[3] * bx[5]);
  const real i5 = real(1) / bx[5];
  real rx = (i0 * pi[0] + i1 * pi[1] + i2 * pi[2]) - (i0 * pj[0] + i1 * pj[1] + i2 * pj[2]);
  real ry = (i3 * pi[1] + i4 * pi[2]) - (i3 * pj[1] + i4 * pj[2]);
  real rz = i5 * pi[2] - i5 * pj[2];
  if (!skip_pbc) {
    rx -= r_rint(rx);
    ry -= r_rint(ry);
    rz -= r_rint(rz);
  }
  d[0] = bx[0] * rx + bx[1] * ry + bx[2] * rz;
  d[1] = bx[3] * ry + bx[4] * rz;
  d[2] = bx[5] * rz;
}

// Pair index q inside an n-item triangle (x<y) -> (x,y); same numbering.
__device__ inline void tri_decode_xy(int q, int n, int& x, int& y) { tri_decode(q, n, x, y); }

// ---- library-owned device state (per device) -------------------------------
struct Workspace {
  void* buf = nullptr;
  size_t bytes = 0;
};

// Work areas are kept per stream: ops issued on different streams of one device (e.g. the per-species op chains,
// which do not depend on each other) never share scratch, so they may run concurrently.
struct StreamWork {
  Workspace scratch;         // per-slot partial forces / partial sums
  Workspace buckets;         // transpose a force op builds for itself: build counters, counts, keys
  size_t bucket_counters = 0;    // capacity, in ints, of each of the two counter parts
  size_t bucket_entries = 0;     // capacity, in ints, of the key part
  Workspace cells;           // cell list of the descriptor op: set toggle, two sets of cell counters, tables, records
  size_t cell_counters = 0;      // capacity, in ints, of each of the two counter sets
};

// The cell-list block of a stream (see cell_build_kernel).  The toggle and the counters live as long as the block:
// the counter set the toggle names reads zero whenever a descriptor call starts, whatever the shapes of the calls
// before it (a fresh block is cleared on the caller's stream).
struct CellBlock {
  int* toggle = nullptr;     // [1]
  int* counts = nullptr;     // [2][set_ints]
  size_t set_ints = 0;
  char* rest = nullptr;      // rest_bytes, 256-byte aligned: tables and records of this call
};

// What a force kernel needs to find the slots that list an atom (see staf_transpose.hpp).  Two forms:
//   symmetric = 1  the map is one the library's own neighbour search wrote for all N atoms of the frames: i lists
//                  j exactly when j lists i, so an atom's own row names the centres that list it, and the slot is
//                  found by looking the atom up in that centre's row.  `full` is the whole tensor [nf, N, nr+1].
//   symmetric = 0  a transposed map, receiver -> sorted (centre, slot) keys (caller-supplied lists, where ghost
//                  atoms are listed without listing anybody; maps of unknown origin).
struct TransposeRef {
  int symmetric = 0;
  const int* full = nullptr; // symmetric: the intmap2b tensor the view points into
  const unsigned* rowsum = nullptr;   // symmetric: [nf * N] checksum of every row as the descriptor op wrote it (row_hash
                                      // in staf_transpose.hpp), or null where no block could be had: an atom that
                                      // collects through its own row compares, and reports a stale map on a difference
  int* build_cnt = nullptr;  // [nf * Nrecv] fill cursors of a build, all zero between builds
  int* cnt = nullptr;        // [nf * Nrecv] keys per receiving atom
  int* keys = nullptr;       // [nf * Nrecv, cap]
  int cap = 0;
  int key_shift = 0;         // centre number (row in `full`) of row 0 of the map the force op was handed
};

// An intmap2b tensor the descriptor op has written: symmetric, with the checksums of its rows beside it.
struct KnownMap {
  const int* im2 = nullptr;      // the tensor [nf, N, nr+1]
  int nf = 0, N = 0, nr = 0;
  TransposeRef ref;
  Workspace sums;                // [nf * N] words
  unsigned long long stamp = 0;  // last use, for replacement
};
constexpr int KNOWN_MAPS = 8;    // descriptor output tensors remembered at a time
constexpr int STATUS_WORDS = 64;       // error words of a device, one per stream

struct DeviceState {
  int device = -1;
  // Error words kernels OR their bits into: one per stream that has used the device (STATUS_WORDS of them, allocated
  // with the state; later streams share the last one).  The synchronising return of an op reports and clears the word
  // of the op's own stream, so a condition goes to the caller that raised it; a poll reports and clears all of them.
  int* status_d = nullptr;   // [STATUS_WORDS]
  int* status_h = nullptr;   // pinned host mirror, [STATUS_WORDS]
  std::unordered_map<hipStream_t, int> status_slot;
  std::unordered_map<hipStream_t, StreamWork> work;
  KnownMap maps[KNOWN_MAPS];
  std::vector<void*> retired;   // outgrown blocks, freed by staf_ops_release
  unsigned long long map_clock = 0;
};

// For the current device, created on the first call (which allocates and synchronises: refused with null while
// `stream` is being captured).
DeviceState* device_state(hipStream_t stream);
// True while `stream` is being captured into a graph: memory may then neither be freed nor allocated, and a fill
// launched to initialise a fresh block would become part of the graph.
bool stream_is_capturing(hipStream_t stream);
// Dynamic LDS of a launch of `kernel`: up to 64 KB needs nothing, up to the 160 KB of a CU is requested for the
// kernel (host-side attribute, no stream work).  False: the launch cannot be made (STAF_E_LIMIT).
template <typename K>
inline bool lds_request(K kernel, size_t lds) {
  if (lds <= 64 * 1024) return true;
  return lds <= 160 * 1024 &&
         hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
}
// The error word of `stream` on this device (see DeviceState::status_d).
int* status_word(DeviceState* st, hipStream_t stream);
// What the stream's error word says, together with the bits `seen` that the caller has read from it; the word is cleared.
int take_status(DeviceState* st, hipStream_t stream, int seen);
// Both grow on demand and never shrink; under capture a request that does not fit what the stream already holds
// returns null (the caller reports STAF_E_CAPTURE) instead of freeing and allocating.
void* scratch_reserve(DeviceState* st, hipStream_t stream, size_t bytes);
bool cells_reserve(DeviceState* st, hipStream_t stream, size_t counters, size_t rest_bytes, CellBlock* out);
// Transpose a force op builds for itself (n_recv receiving atoms, cap keys each), in the stream's own work area.
bool bucket_reserve(DeviceState* st, size_t n_recv, int cap, hipStream_t stream, TransposeRef* out);
// Remembers the intmap2b tensor `im2` [nf, N, nr+1] that the descriptor op is about to write with its own neighbour search.
// No block for the checksums to be had -> false.
bool remember_map(DeviceState* st, const int* im2, int nf, int N, int nr, hipStream_t stream, TransposeRef* out);
// What is known of the map view a force op was handed (pointer into a descriptor output of N atoms, frame stride ld), if
// it is remembered.
bool find_map(DeviceState* st, const int* im2_view, int nf, int N, int Nl, int ld, int nr, TransposeRef* out);
int finish_op(DeviceState* st, hipStream_t stream);            // launch check (+ optional sync & status fetch)
// STAF_E_CAPTURE when the stream is being captured, else STAF_E_HIP: the code for a work area that could not be had
int reserve_failure(hipStream_t stream);
bool sync_errors_enabled();
struct DeferStatus {   // while one is alive, the calling thread's ops do not synchronise to report device conditions
  DeferStatus();
  ~DeferStatus();
};

// Optional timing of single kernels with HIP events on the stream they are launched on (off by default; switched on
// with staf_ops_kernel_timing).  A KernelTimer brackets one launch; the pairs are summed by staf_ops_kernel_time.
bool kernel_timing_enabled();
void kernel_timing_record(const char* kernel, hipEvent_t a, hipEvent_t b);
struct KernelTimer {
  hipEvent_t a = nullptr, b = nullptr;
  hipStream_t stream;
  const char* name;
  KernelTimer(const char* kernel, hipStream_t s) : stream(s), name(kernel) {
    if (!kernel_timing_enabled()) return;
    if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) { a = b = nullptr; return; }
    (void)hipEventRecord(a, stream);
  }
  ~KernelTimer() {
    if (!a) return;
    (void)hipEventRecord(b, stream);
    kernel_timing_record(name, a, b);
  }
};

// Descriptor geometry shared by all devices (set by construct_descriptors_light).
template <typename real>
struct DescConfig {
  bool ready = false;
  int nr = 0, na = 0, n_max = 0, max_batch = 0;
  real Rc = 0, Rs = 0, Ra = 0;
  real cA = 0, cB = 0, cC = 0, pa = 0, pb = 0;
  int dist2_fma = 0;
  int zero_padding = 0;
};

// Internal launchers shared with the MD entry (staf_api): descriptor op with an explicit configuration, an
// optional caller-supplied neighbour list (owned centres only, Npos >= N positions) and optional no-wrap mode.
// unit != null: radial-only call -- no triplet tensor is written (angdescr, intmap3b, der3b may be null) and unit
// [nf, N, 4, nr] receives the unit vectors centre - neighbour and 1/r of the sorted neighbours.
template <typename real>
int desc_configure(DescConfig<real>& c, real Rc, int nr, int na, real Rs, real Ra);
// the geometry construct_descriptors_light has set
template <typename real>
DescConfig<real> desc_current();
// A caller's neighbour list of one frame in the caller's order: centre i (a slot, 0 <= i < N) has howmany[row_of[i]]
// neighbours, the atoms slot_of[with[row_of[i] * pitch + k]].  The entries have been checked on the host.
// Where the forces on an atom are found is the caller's too (`tr` of desc_launch): for the own search the tensor the map
// goes to, for a list the build
// counters [Npos] (all zero), counts [Npos] and keys [Npos * cap] that the launch fills.  A
// call of several stages holds these itself: what the library remembers by a tensor's address is little, and other
// threads' calls take its place.
struct NeighList {
  const int* howmany;   // null: the library's own search
  const int* with;
  const int* row_of;    // [N]
  const int* slot_of;   // [Npos]
  int pitch;
};
template <typename real>
int desc_launch(const DescConfig<real>& c, const real* pos, const real* box, int nf, int N, int Npos,
                const NeighList* inj, const TransposeRef* tr, int skip_pbc, real* raddescr, real* angdescr,
                real* des3bsupp, int* intmap2b, int* intmap3b, real* der2b, real* der3b, real* der3bsupp,
                int* numtriplet, real* unit, hipStream_t stream);


// Force ops with the wrap switch of the virial forms given per call (skip_pbc = 1: neighbour positions already are
// periodic images; the extern "C" entry points pass the process-wide setting of staf_op_force_set_skip_pbc, the MD
// entry its own per call).  Argument lists as in include/staf_ops.h.  known != null: what the caller holds of the map
// (key_shift: the first row of the view); null: looked up, or the view is transposed first.
template <typename real>
int force_doublets(const real* G, const real* D, const real* dD, const int* im2, int nr, int N, int nf, int Ar,
                   const real* alpha2b, const real* emb2b, int nt, const int* tipos, const int* actual_type,
                   real* force, const int* type_map, int Nl, real* virial, const real* pos, const real* box, int ld,
                   int skip_pbc, void* stream, const TransposeRef* known = nullptr);
// unit != null: the fused forms of the MD entry (T and its Jacobian rebuilt from the radial-only descriptor call's
// unit vectors; Tang, d3b, im3 are not read and may be null).
template <typename real>
int angular_afs(const real* Dsup, const real* Tang, const real* unit, int nr, int na, real* out, int nf, int Nl,
                const int* im3, const int* im2, const real* alpha3b, int Aa, const real* emb3b, const int* type_map,
                const int* numtriplet, int nt, int ld, void* stream, int raw_emb = 0, int out_ld = 0);
// The 2-body inputs of the force launch that adds the pair forces to the 3-body slot forces (staf_force3.hpp).
template <typename real>
struct Force2In {
  const real* G2;       // [nf, Nl, Ar] dE/dAF2
  const real* D;        // raddescr [nf, ld, nr]
  const real* dD;       // der2b [nf, ld, 3, nr]
  const real* alpha2b;  // [nt, Ar]
  const real* emb2b;    // [nt, Ar]
  int Ar;
};

template <typename real>
int force_tripl(const real* G, const real* Dsup, const real* Tang, const real* dDsup, const real* d3b,
                const real* unit, const int* im2, const int* im3, int nr, int na, int N, int nf, int Aa,
                const real* emb3b, int nt,
                const int* tipos, const int* actual_type, real* force, const int* numtriplet, const real* alpha3b,
                const int* type_map, int Nl, real* virial, const real* pos, const real* box, int ld, int skip_pbc,
                void* stream, real* slots_out = nullptr, real* self_out = nullptr,
                const Force2In<real>* two_body = nullptr, const TransposeRef* known = nullptr, int raw_emb = 0);
template <typename real>
int force_total(const int* im2_full, int nr, int N, int nf, int nt, const int* n_local, const real* const* slot_forces,
                const real* const* self_forces, const real* const* force_2b, real* total, void* stream);

// The stages of a whole evaluation (the MD entry, one frame; the batch inference, several), every one a single launch
// over the centres of all species of all frames (species-sorted owned atoms, the species of sp[] in any order).
template <typename real>
struct StepSpecies {
  int first, Nl, Ar, Aa;      // first owned atom and owned atoms in a frame, fingerprints
  const real *alpha2b, *alpha3b, *emb2b, *emb3b;
  real *af2, *af3, *g2, *g3;  // [nf, Nl, Ar], [nf, Nl, Aa]: fingerprints and dE/d fingerprint
  const real* table;          // its parameters laid out (StepTablePart), or null
};
template <typename real>
struct StepRows {             // what the radial-only descriptor launch leaves, nr-wide rows of all owned atoms
  const real *raddescr, *des3bsupp, *der2b, *der3bsupp, *unit;
  const int *intmap2b, *numtriplet;
  int nr, na, nf, nlocal;     // nlocal rows per frame
  TransposeRef tr;            // what desc_launch was given
};
// The parameters of a species laid out for the kernels below (staf_step.hpp; step_table_reals has the size), written by the
// launch that lays out the networks (dev_mlp_pack).
constexpr int STEP_CHANNELS = 1024;
template <typename real>
struct StepTablePart {
  const real *alpha3b, *emb3b;
  real* table;
  size_t reals;      // what it may take up
  int Aa, raw_emb;   // emb3b is to be squared
};
// 2-body and 3-body fingerprints
template <typename real>
int step_fingerprints(const StepSpecies<real>* sp, int n, const StepRows<real>& R, const int* type_map, int nt,
                      hipStream_t stream);
// True: step_forces takes a species of these sizes.  Its workgroups hold the parameter rows of both bodies; sizes close to
// a CU's LDS that it does not take may still fit force_doublets and force_tripl, an op per body.
template <typename real>
bool step_forces_fits(int nr, int nt, int Ar, int Aa);
// forces on the centres' slots [nf, nlocal, nr, 3] and on the centres [nf, nlocal, 3]; vpart [nf, nlocal, 9]: their
// virials, or null
template <typename real>
int step_forces(const StepSpecies<real>* sp, int n, const StepRows<real>& R, const int* type_map, int nt, real* slots,
                real* self, real* vpart, hipStream_t stream);
// Forces of all nall atoms of every frame (force null: none), and the sums over the centres of a frame: nparts rows of
// (virial (9), energy) per frame, each of a share of the centres, in `parts` [nf, nparts, 10]; or, parts null, energy
// [nf] = half the sum of e_atom and virial [nf, 9] (zero without vpart).  e_atom of species k: nf rows of its atoms from
// nf times its first atom on.
template <typename real>
struct StepCollect {
  const real *slots, *self, *vpart, *e_atom;
  real *force, *parts, *energy, *virial;
  int nparts;
};
template <typename real>
int step_collect(const StepSpecies<real>* sp, int n, const StepRows<real>& R, int nall, const StepCollect<real>& out,
                 hipStream_t stream);

}  // namespace staf
