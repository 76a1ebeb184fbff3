// 3-body fingerprints of the paths that hold no tensor of the angular buffer's width (the MD entry, the batch inference), from
// the nr-wide rows of the radial-only descriptor launch, for up to 64 neighbours and angular buffers that hold all their
// pairs (step_slots), in launches that it leaves enough waves (RowsLaunch); the others go through tri_reduce_body.
//
// tri_reduce_body, which also rebuilds T where no angular tensor exists, stages the triplets of a class in LDS and reads a
// record and two table rows per (triplet, channel): its inner loop is as long as its LDS reads take, whatever it computes (the
// exponential from the table below took 8 of its 21 instructions away and no time), and without the loop the launch still
// takes 240 of 370 us: staging, seven to twelve barriers per centre, tables.  rows_body walks over the rows of the triplet
// triangle instead, four rows x of a class at a time against sixteen columns y:
//   * lane (r, l) forms T(x_r, y_l) once, and the sixteen lanes of row r, now a channel each, take it from its lane by a
//     broadcast within the row (DPP): triplets never go through LDS;
//   * e^(a1 D_x), e^(a2 D_x) of the lane's row are in registers, sum_y T e^(bT) e^(a2 D_y) and sum_y T e^(bT) e^(a1 D_y) are what
//     is summed (two multiply-adds per item instead of four operations), and the row's factors are applied once per row;
//   * one table entry per item is read from LDS, the same address for the four rows;
//   * all classes' tables are built at once, the rows of all classes are dealt to the waves: three barriers per centre.
// Launches of 24576, 4 x 768 (inference), 768 and 96 centres: 366 -> 335, 56.6 -> 52, 24.9 -> 19 and 12.5 -> 11.0 us in double
// precision (157 -> 137 M vector instructions, 28 -> 13 M LDS instructions for 24576), 4 x 768 in single 31.8 -> 25.3; the vector
// instructions of 24576 centres fill 0.66 of the issue slots, the rest is latency at four waves per SIMD (127 registers; five would
// need 96, and less than the 38 KB of LDS that 60 slots of two species take).
#pragma once
#include <vector>

#include "staf_tri.hpp"

namespace staf {

// What the kernel needs of a species' parameters, laid out once for a loaded model, once a call where the
// parameters are a caller's tensors: the channels of every sigma whose embedding is not 0, in ascending order, then
// zeros up to the pitch, which is the largest number of such channels in whole sixteens.
//   [STEP_HEAD]  N, the largest number of such channels, N', pitch; [8 + sigma] the number of such channels
//   [nsig][pitch][4]  alpha1, alpha2, embedding, channel
//   [nsig][pitch]     beta
//   double: [nsig][N + 1][pitch]  e^(beta i/N), and [nsig][N' + 1][pitch] of (e^(alpha1 i/N'), e^(alpha2 i/N'))
// The last part: e^(beta T) = g + g p(beta (T - i/N)) with g from the row nearest to T.  What the reduction of HotExp does per
// triplet and channel -- the integer part, the remainder, the power of two -- is done once per triplet, with exact results: i
// and T - i/N.  N is the smallest power of two with |beta| / (2 N) <= 2^-7 for every channel (trained values are between -10 and
// 4; beyond EXP_ROWS / 64 = 64, and where a beta is not a number, N is 0 and HotExp::product is used); there p, of degree 5 through 0 with
// slope 1 and the values of e^x at four Chebyshev points, is off by at most 4e-17.  N' likewise, up to PAIR_ROWS / 64 = 16: a slot's
// entries are few beside the triplets.  Launch of 5832 centres of two species with a beta of -20 and -60: 82.7 us in the staged form, 90.1
// without rows, 78.0 and 78.4 with them.  A loaded model whose N is 0 takes the staged form; the batch inference, whose host does not
// know, does not: 46.5 -> 59.4 us for 4 x 729 centres.
constexpr int EXP_ROWS = 4096, PAIR_ROWS = 1024, STEP_HEAD = 32;
__host__ __device__ inline int step_pitch(int channels) { return channels > 16 ? (channels + 15) & ~15 : 16; }
// where the parts lie, in reals
struct StepTable {
  int N, Np, pitch;   // as in the head
  size_t par, beta, rows, pairs, end;
  __host__ __device__ StepTable(int nsig, int pitch_, int N_, int Np_) : N(N_), Np(Np_), pitch(pitch_) {
    const size_t lines = (size_t)nsig * pitch;
    par = STEP_HEAD;
    beta = par + 4 * lines;
    rows = beta + lines;
    pairs = rows + (N ? lines * (N + 1) : 0);
    end = pairs + (Np ? lines * (Np + 1) * 2 : 0);
  }
};
// What is kept for a table whose parameters are a caller's tensors, which the host does not read: the most rows of beta and 128 of the
// alphas with every channel in use, or what takes no more.  A table that does not fit is laid out without the rows of the alphas.
template <typename real>
inline size_t step_table_reals(int nt, int Aa) {
  constexpr bool rows = sizeof(real) == 8;
  return StepTable(2 * nt - 1, step_pitch(Aa), rows ? EXP_ROWS : 0, rows ? 128 : 0).end;
}
// rows of a table for exponents up to `largest` (which is rounded: 2^-24 of it do not count), 0 where they would be more than `rows`
__host__ __device__ inline int exp_rows(float largest, int rows) {
  int N = largest <= (float)(rows / 64) ? 1 : 0;
  while (N && (float)N < 64 * largest) N *= 2;
  return N;
}
// e^(a t): the product's rounding is made good
__host__ __device__ inline double exp_of(double a, double t) {
  const double hi = a * t, e = exp(hi);
  return fma(e, fma(a, t, -hi), e);
}
// the larger of `a` and |v|; 1e30 where a v is beyond that or not a number
__host__ __device__ inline float exp_larger(float a, float v) {
  return !(fabsf(v) <= 1e30f) ? 1e30f : fmaxf(a, fabsf(v));
}
// The table of a loaded model, on the host; emb3b squared.  step_table_body is the same on the device.
inline std::vector<double> step_table_host(const double* alpha3b, const double* emb3b, int nt, int Aa) {
  const int nsig = 2 * nt - 1;
  float most = 0, most_a = 0;
  std::vector<int> ch[2 * NT_MAX];
  size_t active = 0;
  for (int s = 0; s < nsig; s++) {
    for (int a = 0; a < Aa; a++) {
      if (emb3b[s * Aa + a] == 0) continue;
      const double* al = alpha3b + 3 * ((size_t)s * Aa + a);
      most_a = exp_larger(exp_larger(most_a, (float)al[0]), (float)al[1]);
      most = exp_larger(most, (float)al[2]);
      ch[s].push_back(a);
    }
    active = ch[s].size() > active ? ch[s].size() : active;
  }
  const StepTable L(nsig, step_pitch((int)active), exp_rows(most, EXP_ROWS), exp_rows(most_a, PAIR_ROWS));
  std::vector<double> t(L.end, 0.0);
  t[0] = L.N; t[1] = (double)active; t[2] = L.Np; t[3] = L.pitch;
  for (int s = 0; s < nsig; s++) {
    t[8 + s] = (double)ch[s].size();
    for (size_t c = 0; c < ch[s].size(); c++) {
      const double* al = alpha3b + 3 * ((size_t)s * Aa + ch[s][c]);
      const size_t at = (size_t)s * L.pitch + c;
      double* const par = &t[L.par + 4 * at];
      par[0] = al[0]; par[1] = al[1]; par[2] = emb3b[s * Aa + ch[s][c]]; par[3] = ch[s][c];
      t[L.beta + at] = al[2];
      for (int i = 0; L.N && i <= L.N; i++) t[L.rows + ((size_t)s * (L.N + 1) + i) * L.pitch + c] = exp_of(al[2], (double)i / L.N);
      for (int i = 0; L.Np && i <= L.Np; i++)
        for (int k = 0; k < 2; k++)
          t[L.pairs + (((size_t)s * (L.Np + 1) + i) * L.pitch + c) * 2 + k] = exp_of(al[k], (double)i / L.Np);
    }
  }
  return t;
}
// where T lies: its row, and its distance from it
__device__ inline int exp_place(double T, double n, double inv_n, int N, double& rest) {
  const double r = rint(T * n);
  rest = fma(-r, inv_n, T);
  const int i = (int)r;
  return i < 0 ? 0 : (i > N ? N : i);
}
// g e^x for |x| <= 2^-7
__device__ inline double exp_near(double x, double g) {
  double q = fma(x, 0.008333345443492365, 0.041666751437797855);
  q = fma(q, x, 0.1666666666665743);
  q = fma(q, x, 0.49999999999935324);
  q = fma(q, x, 1.0);
  return fma(g, q * x, g);
}

// A slot's entry of the pair tables, (e^(alpha1 D), e^(alpha2 D)) of one channel, by the table's rows (n > 0) or HotExp::product.  D is a
// cutoff function's value, between 0 and 1.
template <typename real>
struct PairTable {
  const real* rows;
  int n, pitch;
  __device__ PairTable(const real* table, const StepTable& L) : rows(table + L.pairs), n(L.Np), pitch(L.pitch) {}
  // what a slot's entries have in common: its row and its distance from it
  __device__ int place(real D, real& rest) const {
    if constexpr (sizeof(real) == 8) {
      return exp_place(D, (real)n, real(1) / (real)n, n, rest);
    } else {
      rest = 0;
      return 0;
    }
  }
  __device__ typename Vec2<real>::type operator()(real a1, real a2, int sg, int channel, real D, int row, real rest) const {
    using HE = HotExp<real>;
    typename Vec2<real>::type v;
    if constexpr (sizeof(real) == 8) {
      if (n) {
        const auto g = ((const typename Vec2<real>::type*)rows)[(unsigned)(sg * (n + 1) + row) * (unsigned)pitch + channel];
        v.x = exp_near(a1 * rest, g.x);
        v.y = exp_near(a2 * rest, g.y);
        return v;
      }
    }
    v.x = HE::product(a1, D);
    v.y = HE::product(a2, D);
    return v;
  }
};

// broadcast of lane L of every row of sixteen lanes
template <int L>
__device__ inline double row_lane(double v) {
  return __longlong_as_double(__builtin_amdgcn_update_dpp(0ll, __double_as_longlong(v), 0x150 + L, 0xf, 0xf, true));
}
template <int L>
__device__ inline float row_lane(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + L, 0xf, 0xf, true));
}
template <int L>
__device__ inline unsigned row_lane(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + L, 0xf, 0xf, true);
}
// read-only memory through the scalar cache: addresses are uniform
template <typename T>
__device__ inline const __attribute__((address_space(4))) T* scalar_ptr(const T* p) {
  return (const __attribute__((address_space(4))) T*)p;
}

__host__ __device__ inline bool step_slots(int nr, int na, int nt) {
  return nr > 0 && nr <= WAVE && na >= nr * (nr - 1) / 2 && nt <= NT_MAX;
}

// Slots grouped by species, by one full wave: lane s holds slot s (its species t_s, anything for lanes that take no part: on
// false).  Behind every group lie `pad` places that hold no slot.  off [nt + 1]; returns the place of the lane's slot.
__device__ inline int group_lane(int nt, int t_s, bool on, int pad, int* off) {
  const int lane = lane_id();
  int pos = 0, base = 0;
  for (int t = 0; t < nt; t++) {
    const unsigned long long mask = __ballot(on && t_s == t);
    if (lane == 0) off[t] = base;
    if (on && t_s == t) pos = base + __popcll(mask & ((1ull << lane) - 1ull));
    base += __popcll(mask) + pad;
  }
  if (lane == 0) off[nt] = base;
  return pos;
}

// ---------------------------------------------------------------------------
// The table, by workgroup `part` of `parts` of sigma sg.  Every workgroup finds the largest exponents and the numbers of active channels of
// all sigmas for itself -- their parameters are read at once, whether their channels are active or not: a read that waits for
// another one is what the launch would last for --, the first one of a sigma writes the parameters, all of them the rows.
// ---------------------------------------------------------------------------
constexpr int STEP_TABLE_BLOCK = 256;
template <typename real>
inline size_t step_table_lds(int Aa) { return (size_t)Aa * 5 * sizeof(real); }
template <typename real>
constexpr int STEP_TABLE_PARTS = sizeof(real) == 8 ? 32 : 1;   // (single precision has no rows)
template <typename real>
__device__ inline void step_table_body(const StepTablePart<real>& P, int nt, int sg, int part, int parts) {
  using real4 = typename Vec4<real>::type;
  constexpr bool DBL = sizeof(real) == 8;
  constexpr int WAVES = STEP_TABLE_BLOCK / WAVE;
  extern __shared__ __align__(16) unsigned char smem[];
  real4* const own = (real4*)smem;                 // [Aa] alpha1, alpha2, embedding, channel of the active channels of sigma sg
  real* const own_beta = (real*)(own + P.Aa);      // [Aa]
  __shared__ float top[WAVES][2];
  __shared__ int act[WAVES], active;
  const int nsig = 2 * nt - 1, Aa = P.Aa;
  const int tid = threadIdx.x, lane = lane_id(), wave = tid / WAVE;
  float most = 0, most_a = 0;
  int channels = 0;
  for (int s = wave; s < nsig; s += WAVES) {
    int base = 0;
    for (int a0 = 0; a0 < Aa; a0 += WAVE) {
      const int a = a0 + lane;
      real4 x;
      x.x = x.y = x.z = x.w = 0;
      real be = 0;
      if (a < Aa) {
        const real* al = P.alpha3b + 3 * ((size_t)s * Aa + a);
        x.z = P.emb3b[s * Aa + a];
        x.x = al[0]; x.y = al[1]; be = al[2];
        x.w = real(a);
        if (P.raw_emb) x.z *= x.z;
      }
      const bool on = x.z != real(0);
      const unsigned long long mask = __ballot(on);
      if (on) {
        most_a = exp_larger(exp_larger(most_a, (float)x.x), (float)x.y);
        most = exp_larger(most, (float)be);
        if (s == sg) {
          const int at = base + __popcll(mask & ((1ull << lane) - 1ull));
          own[at] = x;
          own_beta[at] = be;
        }
      }
      base += __popcll(mask);
    }
    channels = base > channels ? base : channels;
    if (s == sg && lane == 0) active = base;
  }
#pragma unroll
  for (int d = WAVE / 2; d > 0; d >>= 1) {
    most = fmaxf(most, __shfl_xor(most, d, WAVE));
    most_a = fmaxf(most_a, __shfl_xor(most_a, d, WAVE));
  }
  if (lane == 0) { top[wave][0] = most; top[wave][1] = most_a; act[wave] = channels; }
  __syncthreads();
  for (int w = 0; w < WAVES; w++) {
    most = fmaxf(most, top[w][0]);
    most_a = fmaxf(most_a, top[w][1]);
    channels = act[w] > channels ? act[w] : channels;
  }
  const int N = DBL ? exp_rows(most, EXP_ROWS) : 0, Np = DBL ? exp_rows(most_a, PAIR_ROWS) : 0;
  StepTable L(nsig, step_pitch(channels), N, Np);
  if (L.end > P.reals) L = StepTable(nsig, L.pitch, N, 0);
  if (part == 0) {
    if (tid == 0) {
      P.table[8 + sg] = real(active);
      if (sg == 0) { P.table[0] = real(L.N); P.table[1] = real(channels); P.table[2] = real(L.Np); P.table[3] = real(L.pitch); }
    }
    real4* const par = (real4*)(P.table + L.par) + (size_t)sg * L.pitch;
    real* const beta = P.table + L.beta + (size_t)sg * L.pitch;
    for (int c = tid; c < L.pitch; c += STEP_TABLE_BLOCK) {
      real4 x;
      x.x = x.y = x.z = x.w = 0;
      real be = 0;
      if (c < active) { x = own[c]; be = own_beta[c]; }
      par[c] = x;
      beta[c] = be;
    }
  }
  if constexpr (DBL) {
    // sixteen values at a time: rows 0 .. N of beta, then those of alpha1 and alpha2 in turn (1/N and 1/N' are exact)
    const int n = L.N ? L.N + 1 : 0, np = L.Np ? L.Np + 1 : 0;
    const real inv = real(1) / L.N, inv_p = real(1) / L.Np;
    real* const rows = P.table + L.rows + (size_t)sg * n * L.pitch;
    real* const pairs = P.table + L.pairs + (size_t)sg * np * L.pitch * 2;
    for (int q = part * (STEP_TABLE_BLOCK / 16) + tid / 16; q < n + 2 * np; q += parts * (STEP_TABLE_BLOCK / 16))
      for (int c = tid & 15; c < L.pitch; c += 16) {
        const int k = (q - n) & 1, i = q < n ? q : (q - n) >> 1;
        real v = 0;
        if (c < active) v = exp_of(q < n ? own_beta[c] : k ? own[c].y : own[c].x, real(i) * (q < n ? inv : inv_p));
        (q < n ? rows + (size_t)i * L.pitch + c : pairs + ((size_t)i * L.pitch + c) * 2 + k)[0] = v;
      }
  }
}

// ---------------------------------------------------------------------------
// Fingerprints
// ---------------------------------------------------------------------------
template <typename real, int WAVES>
struct RowsCfg {
  static constexpr int THREADS = WAVES * WAVE;
  static constexpr int PAD = 3;            // rows of zeros behind every species', which a step of four may read
  static constexpr int MIN_WAVES = sizeof(real) == 8 ? 4 : 8;
  __host__ __device__ static int rows(int nr, int nt) { return nr + nt * PAD; }
  __host__ __device__ static size_t bytes(int nr, int Aa, int nt) {
    const size_t r = rows(nr, nt);
    size_t b = (nt * r * TRI_CAP * 2 + 5 * r + (size_t)WAVES * Aa) * sizeof(real);
    b += (r + NT_MAX + 1) * sizeof(int);
    return (b + 15) & ~(size_t)15;
  }
};
// LDS of a workgroup of a launch that takes rows_body with WAVES waves per centre for a species of these sizes: that of rows_body, or
// that of the workgroups of the 2-body fingerprints.
template <typename real, int WAVES>
inline size_t rows_lds(int nr, int nt, int Ar, int Aa) {
  const size_t two_body = (size_t)2 * nt * Ar * sizeof(real) + (size_t)WAVES * nr * (sizeof(real) + sizeof(int));
  const size_t b = RowsCfg<real, WAVES>::bytes(nr, Aa, nt);
  return b > two_body ? b : two_body;
}
// workgroups whose LDS a CU's 160 KB hold at once: they are handed out in pieces of 1280 bytes
inline int lds_workgroups(size_t lds) { return (int)(128 / ((lds + 1279) / 1280)); }
// True: there are launches in which rows_body takes a species of these sizes.  Its table is held to 32 MB.
template <typename real>
inline bool rows_fits(int nr, int na, int nt, int Ar, int Aa) {
  return step_slots(nr, na, nt) && Ar > 0 && Aa > 0 && Aa <= STEP_CHANNELS && lds_workgroups(rows_lds<real, 8>(nr, nt, Ar, Aa)) > 0 &&
         step_table_reals<real>(nt, Aa) * sizeof(real) <= (size_t)32 << 20;
}
// Which form a launch takes.  The tables of rows_body hold nt rows per slot where tri_reduce_body has one: with three species, 60 slots
// and 40 channels a CU holds two workgroups of four waves in double precision, not four.  Where waves are few the launch is slower than the
// staged form, unless all its centres are there at once: then it lasts as long as a centre takes.  Launches of the staged form, of
// rows_body with four and (up to 729) with eight waves per centre, us; the channels dealt to the classes in blocks:
//                                      centres  512                 729                 2197         5832
//   double, two species, 60 slots, 4 per CU:    18.3 / 15.3         20.4 / 16.5         38.8 / 36.6  82.7 / 77.3
//   double, three, 32 slots, 4 per CU:                              20.2 / 16.3         39.7 / 39.2  80.5 / 77.2
//   double, three, 48 slots, 3 per CU:          21.7 / 16.5 / 17.7  22.1 / 20.4 / 21.7  43.3 / 44.0  90.7 / 100.9
//   double, three, 60 slots, 2 per CU:          22.6 / 20.2 / 19.0  24.9 / 28.3 / 23.7  51.1 / 85.0  112.7 / 147.7
//   double, four, 40 slots, 2 per CU:                               26.7 / 30.2         57.8 / 70.5  123.4 / 156.5
//                                      centres  729                 1458                2916         11664
//   single, three, 40 slots, 7 per CU:          17.7 / 14.0                             36.4 / 29.7  104.0 / 88.5
//   single, three, 60 slots, 5 per CU:          18.7 / 15.2         22.6 / 23.3         39.9 / 37.9  114.8 / 110.9
//   single, four, 60 slots, 4 per CU:           24.1 / 18.2         28.8 / 29.1         52.9 / 46.5  156.4 / 152.9
//   single, five, 60 slots, 3 per CU:           31.2 / 23.9                                          274.5 / 235.3
// So rows_body takes launches whose centres are all resident, and others where a CU holds FULL workgroups: four in double precision, what
// its registers admit, three in single.  (With a weight of every channel in every class, which training does not make of blocks -- a
// weight of 0 has no gradient --, the last three rows are 36.5 / 31.4 and 49.3 / 39.5 for 729, but 83.3 / 89.7, 111.6 / 112.4 and
// 146.0 / 168.7 for 2916 and 257.9 / 278.2, 349.1 / 390.9 and 648.9 / 626.5 for 11664.)
// Eight waves per centre up to 448 centres: two species, 60 slots, four and eight waves 13.5 and 10.7 us for 96 centres, 13.9 and 10.8
// for 225, 15.6 and 13.4 for 378, 16.1 and 16.8 for 504, 17.1 and 19.0 for 576, 18.5 and 21.6 for 768.
constexpr int ROWS_CUS = 256, WIDE_ROWS_CENTRES = 448;
template <typename real>
struct RowsLaunch {
  bool fits = true;
  size_t lds4 = 0, lds8 = 0;
  long long centres = 0;
  void add(int nr, int na, int nt, int Ar, int Aa, long long n) {   // a species with n centres
    if (n <= 0) return;
    fits = fits && rows_fits<real>(nr, na, nt, Ar, Aa);
    if (!fits) return;
    const size_t four = rows_lds<real, 4>(nr, nt, Ar, Aa), eight = rows_lds<real, 8>(nr, nt, Ar, Aa);
    lds4 = four > lds4 ? four : lds4;
    lds8 = eight > lds8 ? eight : lds8;
    centres += n;
  }
  // waves per centre of rows_body; 0: tri_reduce_body
  int waves() const {
    constexpr int FULL = sizeof(real) == 8 ? 4 : 3;
    if (!fits || centres == 0) return 0;
    if (centres <= WIDE_ROWS_CENTRES && centres <= ROWS_CUS * lds_workgroups(lds8)) return 8;
    const int held = lds_workgroups(lds4);
    return held >= FULL || centres <= ROWS_CUS * held ? 4 : 0;
  }
};

template <typename real, int WAVES>
__device__ __forceinline__ void rows_body(const TriArgs<real>& A, const real* __restrict__ table, const int first_centre,
                                          const int stride) {
  using real2 = typename Vec2<real>::type;
  using real4 = typename Vec4<real>::type;
  using HE = HotExp<real>;
  using L = RowsCfg<real, WAVES>;
  constexpr bool DBL = sizeof(real) == 8;
  constexpr int THREADS = L::THREADS;
  extern __shared__ __align__(16) unsigned char smem[];
  const int nr = A.nr, Aa = A.Aa, nt = A.nt;
  const int EP = L::rows(nr, nt);                  // rows of a partner species' block of the table
  real2* E = (real2*)smem;                         // [partner species][grouped slot][channel]
  real2* slots = E + (size_t)nt * EP * TRI_CAP;    // [grouped slot] unit vector, cutoff value
  real* rst = (real*)(slots + 2 * EP);             // [grouped slot] distance from its row of the pair tables
  real* outw = rst + EP;
  int* stp = (int*)(outw + (size_t)WAVES * Aa);    // [grouped slot] species | row of the pair tables << 8, -1: none
  int* off = stp + EP;                             // [nt + 1] first grouped slot of a species
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = uniform(tid / WAVE);
  const int ia = lane & (TRI_CAP - 1), r = lane / TRI_CAP;
  real* const my_out = outw + wave * Aa;
  const auto head = scalar_ptr(table);
  auto size = [&](int i) { return uniform((int)head[i]); };   // (converted by a vector instruction)
  const int maxact = size(1);
  const StepTable TL(2 * nt - 1, size(3), DBL ? size(0) : 0, DBL ? size(2) : 0);
  const int exp_n = TL.N, pitch = TL.pitch;
  const real4* const parA = (const real4*)(table + TL.par);
  const real* const beta = table + TL.beta;
  const PairTable<real> pairs(table, TL);
  const real exp_nr = real(exp_n), exp_inv = real(1) / exp_nr;
  const int exp_row = pitch * (int)sizeof(real);

  const int total = A.nf * A.Nl;
  // what a centre's set-up reads from its own rows: issued while the centre before it is summed
  int m_n = 0, nj_n = 0;
  real d_n = 0, u_n[3] = {0, 0, 0};
  auto request = [&](int atom) {   // (by the first wave)
    if (wave > 0) return;
    const int b = atom / A.Nl, p = atom - b * A.Nl;
    const size_t row = (size_t)b * A.ld + p;
    m_n = A.numtriplet[row];
    if (lane < nr) {
      nj_n = A.im2[row * (nr + 1) + 1 + lane];
      d_n = A.Dsup[row * nr + lane];
#pragma unroll
      for (int c = 0; c < 3; c++) u_n[c] = A.unit[(row * 4 + c) * nr + lane];
    }
  };
  request(first_centre);

  for (int atom = first_centre;;) {
    // ---- slots grouped by species
    if (wave == 0) {
      const int m = m_n > nr ? nr : m_n;
      int t_s = 0;
      if (lane < m) t_s = A.type_map[nj_n];
      const int pos = group_lane(nt, t_s, lane < m, L::PAD, off);
      if (lane < m) {
        real2 v, w;
        v.x = u_n[0]; v.y = u_n[1]; w.x = u_n[2]; w.y = d_n;
        slots[2 * pos] = v;
        slots[2 * pos + 1] = w;
        stp[pos] = t_s | (pairs.place(d_n, rst[pos]) << 8);
      }
      __builtin_amdgcn_wave_barrier();
      __threadfence_block();
      if (lane < nt * L::PAD) stp[off[lane / L::PAD + 1] - 1 - lane % L::PAD] = -1;
    }
    __syncthreads();
    const int rows = uniform(off[nt]);
    const int next = stride > total - 1 - atom ? -1 : atom + stride;

    for (int c0 = 0; c0 < maxact; c0 += TRI_CAP) {
      if (c0 > 0) __syncthreads();   // the table of the channels before is consumed
      // ---- table: E[tb][g][ia] = (exp(a1 D), exp(a2 D)) with the parameters of sigma = species + tb
      {
        int g = wave * 4 + r, tb = 0;
        for (;; g += 4 * WAVES) {
          while (g >= rows && tb < nt) { g -= rows; tb++; }
          if (tb >= nt) break;
          real2 v;
          v.x = v.y = 0;
          if (const int at = stp[g]; at >= 0) {
            const int sg = (at & 255) + tb;
            const real2 par = *(const real2*)(parA + sg * pitch + c0 + ia);
            v = pairs(par.x, par.y, sg, c0 + ia, slots[2 * g + 1].y, at >> 8, rst[g]);
          }
          E[(tb * EP + g) * TRI_CAP + ia] = v;
        }
      }
      __syncthreads();
      if (c0 == 0)
        for (int a = lane; a < Aa; a += WAVE) my_out[a] = 0;
      if (c0 + TRI_CAP >= maxact && next >= 0) request(next);
      // ---- rows, four at a time, of every class, dealt to the waves
      int turn = 0;
      for (int ta = 0; ta < nt; ta++) {
        const int oa = uniform(off[ta]), na_ = uniform(off[ta + 1]) - oa - L::PAD;
        for (int tb = ta; tb < nt; tb++) {
          const int ob = uniform(off[tb]), nb_ = uniform(off[tb + 1]) - ob - L::PAD;
          const bool same = ta == tb;
          if (same ? na_ < 2 : na_ * nb_ == 0) continue;
          const int sg = ta + tb;
          if (c0 >= (int)head[8 + sg]) continue;
          // rows x of one species, columns y of the other one (the same: y < x)
          const bool flip = !same && ((na_ + 3) >> 2) * nb_ > ((nb_ + 3) >> 2) * na_;
          const int nx = flip ? nb_ : na_, ny = flip ? na_ : nb_;
          const int ox = flip ? ob : oa, oy = flip ? oa : ob;
          const int tx = flip ? tb : ta, ty = flip ? ta : tb;
          const int blocks = ((same ? nx - 1 : nx) + 3) >> 2;
          int blk = (wave - turn) & (WAVES - 1);
          turn = (turn + blocks) & (WAVES - 1);
          if (blk >= blocks) continue;
          const int at = sg * pitch + c0 + ia;
          const real be = beta[at];
          const real4 par = parA[at];
          const unsigned char* const exp_base =
              (const unsigned char*)(table + TL.rows + c0) + (size_t)sg * (exp_n + 1) * exp_row;
          const unsigned exp_lane = (unsigned)ia * sizeof(real);
          real acc = 0;
          for (; blk < blocks; blk += WAVES) {
            const int x = same ? nx - 1 - 4 * blk - r : 4 * blk + r;
            const int len = same ? nx - 1 - 4 * blk : ny;          // of the block's longest row
            const bool row_ok = x >= 0 && x < nx;
            const int mine = row_ok ? (same ? x : ny) : 0;
            const int gx = ox + (row_ok ? x : 0);
            const real2 x01 = slots[2 * gx], x23 = slots[2 * gx + 1];
            const real2 e1 = E[(ty * EP + gx) * TRI_CAP + ia];
            const real2* Ey = E + (tx * EP + oy) * TRI_CAP + ia;
            real F1 = 0, F2 = 0;
            for (int y0 = 0; y0 < len; y0 += 16, Ey += 16 * TRI_CAP) {
              // T of row r and column y0 + (lane & 15)
              const int y = y0 + ia, gy = oy + (y < ny ? y : ny - 1);
              const real2 y01 = slots[2 * gy], y23 = slots[2 * gy + 1];
              const real cs = x01.x * y01.x + x01.y * y01.y + x23.x * y23.x;
              real T = (real(0.5) * (cs + real(1))) * (x23.y * y23.y);
              T = y < mine ? T : real(0);
              real rest = 0;
              unsigned row = 0;
              if constexpr (DBL) row = (unsigned)mul24(exp_place(T, exp_nr, exp_inv, exp_n, rest), exp_row);
              const int left = len - y0;
              auto four = [&](auto q_c, auto near_c) {
                constexpr int Q = decltype(q_c)::value;
                constexpr bool NEAR = decltype(near_c)::value;
                real2 e2[4];
                real g[4], Tb[4], rb[4];
                auto load = [&](auto u_c) {
                  constexpr int u = decltype(u_c)::value;
                  Tb[u] = row_lane<Q + u>(T);
                  if constexpr (NEAR) {
                    g[u] = *(const real*)(exp_base + (row_lane<Q + u>(row) + exp_lane));
                    rb[u] = row_lane<Q + u>(rest);
                  }
                  e2[u] = Ey[(Q + u) * TRI_CAP];
                };
                load(std::integral_constant<int, 0>{});
                load(std::integral_constant<int, 1>{});
                load(std::integral_constant<int, 2>{});
                load(std::integral_constant<int, 3>{});
#pragma unroll
                for (int u = 0; u < 4; u++) {
                  real e;
                  if constexpr (NEAR) e = exp_near(be * rb[u], g[u]);
                  else e = HE::product(be, Tb[u]);
                  const real w = Tb[u] * e;
                  F2 = r_fma(w, e2[u].y, F2);
                  F1 = r_fma(w, e2[u].x, F1);
                }
              };
              auto sixteen = [&](auto near_c) {
                four(std::integral_constant<int, 0>{}, near_c);
                if (left > 4) four(std::integral_constant<int, 4>{}, near_c);
                if (left > 8) four(std::integral_constant<int, 8>{}, near_c);
                if (left > 12) four(std::integral_constant<int, 12>{}, near_c);
              };
              if constexpr (DBL) {
                if (exp_n) sixteen(std::true_type{});
                else sixteen(std::false_type{});
              } else {
                sixteen(std::false_type{});
              }
            }
            acc = r_fma(e1.x, F2, acc);
            acc = r_fma(e1.y, F1, acc);
          }
          acc += __shfl_xor(acc, 16, WAVE);
          acc += __shfl_xor(acc, 32, WAVE);
          if (lane < TRI_CAP && par.z != real(0)) my_out[(int)par.w] += acc * (par.z * real(0.5));
        }
      }
    }
    if (maxact == 0) {   // (no channel has a weight)
      for (int a = lane; a < Aa; a += WAVE) my_out[a] = 0;
      if (next >= 0) request(next);
    }
    __syncthreads();
    for (int a = (tid + THREADS - WAVE) % THREADS; a < Aa; a += THREADS) {   // (not by the first wave)
      real s = 0;
#pragma unroll
      for (int w = 0; w < WAVES; w++) s += outw[w * Aa + a];
      A.out[(size_t)atom * Aa + a] = s;
    }
    if (next < 0) break;
    atom = next;
  }
}

}  // namespace staf
