// Device-resident evaluation of the per-species MLP of the MD entry and the batch inference: x = log(af + 1e-3) - mu, Dense stack
// (tanh / relu / linear), atomic energy, and dE/d af by back-propagation -- the step between the fingerprint and
// the force kernels that the reference does on the host or through ONNX Runtime
// (Compute_NNEnergyandGradient_all, libstaf/vendor/jmd/nn_nn_mlp.cu:657-768; native evaluation
// libstaf/src/mlp/staf_mlp_ort.cc:186-233).
//
// The Dense layers are small matrix products ([out, in] x [in, atoms]) and run on the matrix cores: a workgroup takes
// 16 atoms, which are the columns of its 16x16x4 tiles (8 or 4 in launches of few atoms: columns of 4x4 tiles), and a wave takes tiles of 16 output features over the whole
// inner dimension, so that no partial sums meet in LDS and a layer costs one barrier per direction.  Activations lie in
// LDS as [feature][16 atoms] (8 atoms also for stacks with more features than fit that way): a tile step's read and the
// result's write are runs of consecutive words.  A layer's delta takes the place of its activations (the derivative needs
// nothing else), and the input the place of the second hidden layer: 39 KB for the reference's stack in double
// precision, four workgroups per CU.  The weights are kept in
// the order in which a wave reads them -- 16 bytes per lane, zero-padded to whole tiles -- forwards and transposed; a
// wave requests the first pieces of its next product ahead of the barrier it waits at and stays six pieces ahead.
// Bound: matrix cores and vector units in turn (16384 atoms in double precision: 25 us of matrix instructions, 16 us of
// activations and the rest, 60 us measured; 150 us before, when the inner dimension was sliced over sixteen waves and
// weights were read row by row), and for a single workgroup the chain of four products (22 us, with four atoms 14; 25 before
// either).  Asking for
// the weights' lines ahead of everything, and more than six pieces in flight, are slower.
#include "staf_mlp_dev.hpp"
#include "staf_step.hpp"

#include <algorithm>
#include <vector>

namespace staf {

constexpr int MLP_AHEAD = 6;     // 16-byte weight pieces a lane has in flight
constexpr int MLP_WAVES_MAX = 16;

template <typename T> struct MlpTile;
// operand layout of the 16x16x4 tiles: A[row = lane % 16][k = lane / 16], B[k = lane / 16][col = lane % 16];
// accumulator element v of a lane: (row(lane, v), col(lane, v)) (the two precisions differ); NV elements
template <> struct MlpTile<double> {
  typedef double acc_t __attribute__((ext_vector_type(4)));
  typedef double piece_t __attribute__((ext_vector_type(2)));
  static constexpr int NV = 4;
  __device__ static acc_t run(double a, const double* X, acc_t c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, *X, c, 0, 0, 0); }
  __device__ static int row(int lane, int v) { return lane / 16 + 4 * v; }
  __device__ static void values(const acc_t& c, int, double (&y)[NV]) {
#pragma unroll
    for (int v = 0; v < NV; v++) y[v] = c[v];
  }
  __device__ static int col(int lane, int) { return lane & 15; }
};
template <> struct MlpTile<float> {
  typedef float acc_t __attribute__((ext_vector_type(4)));
  typedef float piece_t __attribute__((ext_vector_type(4)));
  static constexpr int NV = 4;
  __device__ static acc_t run(float a, const float* X, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, *X, c, 0, 0, 0); }
  __device__ static void values(const acc_t& c, int, float (&y)[NV]) {
#pragma unroll
    for (int v = 0; v < NV; v++) y[v] = c[v];
  }
  __device__ static int row(int lane, int v) { return 4 * (lane / 16) + v; }
  __device__ static int col(int lane, int) { return lane & 15; }
};

// Workgroups of few atoms: four atoms to a tile, TA / 4 tiles beside each other, with the large tiles' operands: A[feature
// 4 b + i][k] and B[k][atom j] in lane 16 k + 4 b + (i or j).  Double precision: 4x4x4 tiles in four blocks b, element
// (feature 4 b + i, atom j) in lane 16 i + 4 b + j.  Single precision: 4x4x1 tiles in sixteen blocks, a block for every (k,
// b): the four k of an element are added at the end, and the lane of k keeps element i = k, as in double precision.  The
// matrix cores do four atoms at the rate of sixteen (measured 17 cycles an instruction, 66 for the large tile's four times
// the work; single precision 10 to 12 and 32).
template <typename T, int TILES> struct MlpTiles4;
template <int TILES>
struct MlpTiles4<double, TILES> {
  struct acc_t { double v[TILES]; };
  typedef double piece_t __attribute__((ext_vector_type(2)));
  static constexpr int NV = TILES;
  __device__ static acc_t run(double a, const double* X, acc_t c) {
#pragma unroll
    for (int t = 0; t < TILES; t++) c.v[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, X[4 * t], c.v[t], 0, 0, 0);
    return c;
  }
  __device__ static void values(const acc_t& c, int, double (&y)[NV]) {
#pragma unroll
    for (int t = 0; t < TILES; t++) y[t] = c.v[t];
  }
  __device__ static int row(int lane, int) { return (lane & 12) + lane / 16; }
  __device__ static int col(int lane, int v) { return 4 * v + (lane & 3); }
};
template <int TILES>
struct MlpTiles4<float, TILES> {
  typedef float four __attribute__((ext_vector_type(4)));
  struct acc_t { four v[TILES]; };
  typedef four piece_t;
  static constexpr int NV = TILES;
  __device__ static acc_t run(float a, const float* X, acc_t c) {
#pragma unroll
    for (int t = 0; t < TILES; t++) c.v[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, X[4 * t], c.v[t], 0, 0, 0);
    return c;
  }
  __device__ static void values(const acc_t& c, int lane, float (&y)[NV]) {
    const bool hi2 = lane & 32, hi1 = lane & 16;
#pragma unroll
    for (int t = 0; t < TILES; t++) {
      // each half of the lanes keeps two elements and hands the other two on, then each quarter one
      const four& e = c.v[t];
      const float p = (hi2 ? e[2] : e[0]) + __shfl_xor(hi2 ? e[0] : e[2], 32, WAVE);
      const float q = (hi2 ? e[3] : e[1]) + __shfl_xor(hi2 ? e[1] : e[3], 32, WAVE);
      y[t] = (hi1 ? q : p) + __shfl_xor(hi1 ? p : q, 16, WAVE);
    }
  }
  __device__ static int row(int lane, int) { return (lane & 12) + lane / 16; }
  __device__ static int col(int lane, int v) { return 4 * v + (lane & 3); }
};

template <typename T> __host__ __device__ constexpr int mlp_steps() { return 16 / (int)sizeof(T); }   // tile steps per piece
// features of a layer as they lie in LDS: whole tiles
__host__ __device__ inline int mlp_rows(int n) { return (n + 15) & ~15; }
__host__ __device__ inline int mlp_tiles(int n) { return (n + 15) / 16; }
template <typename T> __host__ __device__ inline int mlp_pieces(int n) { return mlp_rows(n) / (4 * mlp_steps<T>()); }

template <typename T>
struct MlpNet {
  int nl, n_af, act[DEV_MLP_MAX_LAYERS], in_f[DEV_MLP_MAX_LAYERS], out_f[DEV_MLP_MAX_LAYERS];
  const T* fw[DEV_MLP_MAX_LAYERS];
  const T* bw[DEV_MLP_MAX_LAYERS];
  const T* b[DEV_MLP_MAX_LAYERS];
  const T* mu;
};
template <typename real>
struct MlpSpecies {
  const real *af2, *af3;
  real *e_atom, *g2, *g3;
  int Ar, Aa, Nl, first;   // first workgroup of the species
};
template <typename T, typename real>
struct MlpArgs {
  int ns;
  MlpSpecies<real> sp[NT_MAX];
  MlpNet<T> net[NT_MAX];
};

__device__ inline float m_log(float x) { return logf(x); }
__device__ inline double m_log(double x) { return log(x); }
// tanh(x) = m / (m + 2), m = e^{2|x|} - 1, with the sign of x.  2|x| = n ln2 + r, |r| <= ln2/2, with ln2 in two parts
// (Cody and Waite), and m = 2^n (e^r - 1) + (2^n - 1), e^r - 1 by its Taylor polynomial (degree 13 / 7, truncation below a
// tenth of a unit in the last place of r): accurate relative to the result down to the smallest x.  Beyond 2|x| = 44 (20)
// the result is 1 to the last place.  Largest relative error of the formulas, evaluated with a reciprocal off both ways,
// 1.45 x 2^-52 (1.26 x 2^-23; tests/test_tanh.py).  28 (22) vector instructions instead of the C library's 150: with the latter a double-precision
// workgroup spent more time on the 4480 values of its two hidden layers than on its matrix products.
__device__ inline double m_tanh(double x) {
  const double y0 = 2.0 * fabs(x), y = y0 > 44.0 ? 44.0 : y0;   // (NaN stays)
  const double n = rint(y * 1.4426950408889634);
  double r = fma(n, -6.93147180369123816490e-01, y);
  r = fma(n, -1.90821492927058770002e-10, r);
  double p = 1.0 / 6227020800.0;                // 1/13!
  p = fma(p, r, 1.0 / 479001600.0);
  p = fma(p, r, 1.0 / 39916800.0);
  p = fma(p, r, 1.0 / 3628800.0);
  p = fma(p, r, 1.0 / 362880.0);
  p = fma(p, r, 1.0 / 40320.0);
  p = fma(p, r, 1.0 / 5040.0);
  p = fma(p, r, 1.0 / 720.0);
  p = fma(p, r, 1.0 / 120.0);
  p = fma(p, r, 1.0 / 24.0);
  p = fma(p, r, 1.0 / 6.0);
  p = fma(p, r, 0.5);
  p = fma(p, r * r, r);                         // e^r - 1
  const double s = ldexp(1.0, (int)n);
  const double m = fma(s, p, s - 1.0);
  // m / (m + 2): two Newton-Raphson steps on the hardware reciprocal, the quotient corrected once with its residual
  const double d = m + 2.0;
  double q = __builtin_amdgcn_rcp(d);
  q = fma(fma(-d, q, 1.0), q, q);
  q = fma(fma(-d, q, 1.0), q, q);
  double t = m * q;
  t = fma(fma(-d, t, m), q, t);
  return copysign(t, x);
}
__device__ inline float m_tanh(float x) {
  const float y0 = 2.0f * fabsf(x), y = y0 > 20.0f ? 20.0f : y0;
  const float n = rintf(y * 1.44269504f);
  float r = fmaf(n, -0.693145752f, y);
  r = fmaf(n, -1.42860677e-06f, r);
  float p = 1.0f / 5040.0f;
  p = fmaf(p, r, 1.0f / 720.0f);
  p = fmaf(p, r, 1.0f / 120.0f);
  p = fmaf(p, r, 1.0f / 24.0f);
  p = fmaf(p, r, 1.0f / 6.0f);
  p = fmaf(p, r, 0.5f);
  p = fmaf(p, r * r, r);
  const float s = ldexpf(1.0f, (int)n);
  const float m = fmaf(s, p, s - 1.0f);
  const float d = m + 2.0f;
  float q = __builtin_amdgcn_rcpf(d);
  q = fmaf(fmaf(-d, q, 1.0f), q, q);
  float t = m * q;
  t = fmaf(fmaf(-d, t, m), q, t);
  return copysignf(t, x);
}

// activation of the four values of a lane, and its derivative where the value is y
template <typename T, int NV>
__device__ inline void mlp_act(int act, T (&y)[NV]) {
  if (act == 1) {
#pragma unroll
    for (int v = 0; v < NV; v++) y[v] = m_tanh(y[v]);
  } else if (act == 2) {
#pragma unroll
    for (int v = 0; v < NV; v++) y[v] = y[v] < T(0) ? T(0) : y[v];   // (NaN stays)
  }
}
template <typename T>
__device__ inline T mlp_slope(int act, T y) {
  const T relu = act == 2 && y <= T(0) ? T(0) : T(1);
  return act == 1 ? T(1) - y * y : relu;
}

// (Single precision with 16 atoms is held to the eight waves per SIMD that 64 registers admit: with 70 and seven waves a launch
// of 24576 atoms takes 54.8 instead of 49.7 us.  With 8 atoms it would spill there.)
// TA: atoms per workgroup, 16, 8 or 4 (mlp_atoms).
template <typename T, typename real, int TA>
__global__ __launch_bounds__(MLP_WAVES_MAX * WAVE, sizeof(T) == 4 ? (TA == 16 ? 8 : 5) : 4) void mlp_kernel(const MlpArgs<T, real> A) {
  static_assert(TA == 4 || TA == 8 || TA == 16, "columns of the tiles");
  using M = std::conditional_t<(TA < 16), MlpTiles4<T, TA / 4>, MlpTile<T>>;
  using piece_t = typename M::piece_t;
  using acc_t = typename M::acc_t;
  constexpr int STEPS = mlp_steps<T>(), NV = M::NV;
  extern __shared__ __align__(16) unsigned char smem[];
  // [rows of the hidden layers][TA atoms], then the parts of the energy sums; the input lies where the second hidden
  // layer will
  T* const H = (T*)smem;
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = uniform(tid / WAVE), nw = blockDim.x / WAVE;
  int s = 0;
  while (s + 1 < A.ns && (int)blockIdx.x >= A.sp[s + 1].first) s++;
  const MlpSpecies<real>& S = A.sp[s];
  const MlpNet<T>& net = A.net[s];
  const int a0 = ((int)blockIdx.x - S.first) * TA;
  const int nl = net.nl, n_af = net.n_af;
  const int my = lane & (TA - 1);                              // the lane's atom outside the products
  const bool live = a0 + my < S.Nl;
  const size_t atom = (size_t)(live ? a0 + my : S.Nl - 1);     // (lanes without an atom follow the last one, storing nothing)
  auto col = [&](int v) -> int { return M::col(lane, v); };   // atom of a product's value v

  // The pieces requested ahead may lie beyond the tile's last one: in the next tile or, behind the last matrix, in the
  // spare pieces at the end of the block; they are not used.
  piece_t ring[MLP_AHEAD];
  // the first pieces of the wave's first tile of a product
  auto request = [&](const T* frag, int tile, int np) {
    const piece_t* f = (const piece_t*)frag + (size_t)tile * np * WAVE + lane;
#pragma unroll
    for (int u = 0; u < MLP_AHEAD; u++) ring[u] = f[u * WAVE];
  };
  auto product = [&](const T* frag, int tile, int np, const T* X, T (&out)[NV]) {
    const piece_t* f = (const piece_t*)frag + (size_t)tile * np * WAVE + lane;
    acc_t acc = {};
    const int whole = np / MLP_AHEAD, rest = np - whole * MLP_AHEAD;
    X += (lane / 16) * TA + col(0);
    for (int g = 0; g < whole; g++) {
      f += MLP_AHEAD * WAVE;
#pragma unroll
      for (int u = 0; u < MLP_AHEAD; u++) {
        const piece_t w = ring[u];
        ring[u] = f[u * WAVE];
#pragma unroll
        for (int j = 0; j < STEPS; j++) acc = M::run(w[j], X + (u * STEPS + j) * 4 * TA, acc);
      }
      X += MLP_AHEAD * STEPS * 4 * TA;
    }
#pragma unroll
    for (int u = 0; u + 1 < MLP_AHEAD; u++) {
      if (u >= rest) break;
#pragma unroll
      for (int j = 0; j < STEPS; j++) acc = M::run(ring[u][j], X + (u * STEPS + j) * 4 * TA, acc);
    }
    M::values(acc, lane, out);
  };

  const int np0 = mlp_pieces<T>(n_af);
  if (nl > 1 && wave < mlp_tiles(net.out_f[0])) request(net.fw[0], wave, np0);
  const int rows0 = mlp_rows(n_af);
  T* const input = H + (nl > 1 ? mlp_rows(net.out_f[0]) * TA : 0);
  for (int i = tid / TA; i < rows0; i += (int)blockDim.x / TA) {
    T v = 0;
    if (i < n_af && live) {
      const T afv = (T)(i < S.Ar ? S.af2[atom * S.Ar + i] : S.af3[atom * S.Aa + (i - S.Ar)]);
      v = m_log(afv + T(1e-3)) - net.mu[i];
    }
    input[i * TA + my] = v;
  }
  __syncthreads();
  // ---- forward through the hidden layers
  T* X = input;
  for (int l = 0; l + 1 < nl; l++) {
    const int in_f = net.in_f[l], out_f = net.out_f[l], act = net.act[l];
    const int np = mlp_pieces<T>(in_f), tiles = mlp_tiles(out_f);
    T* Y = l == 0 ? H : X + mlp_rows(in_f) * TA;
    for (int tile = wave; tile < tiles; tile += nw) {
      if (tile != wave) request(net.fw[l], tile, np);
      T y[NV];
#pragma unroll
      for (int v = 0; v < NV; v++) y[v] = net.b[l][tile * 16 + M::row(lane, v)];
      T acc[NV];
      product(net.fw[l], tile, np, X, acc);
#pragma unroll
      for (int v = 0; v < NV; v++) y[v] += acc[v];
      mlp_act<T, NV>(act, y);
      // (features beyond the last are 0 whatever their zero weights were multiplied with: an infinite value gives no number.
      // Only a layer's last tile has such, and writes them again behind the others' values: as a select of every value
      // this takes 2 % of the launch in double precision)
#pragma unroll
      for (int v = 0; v < NV; v++) Y[(tile * 16 + M::row(lane, v)) * TA + col(v)] = y[v];
      if (tile * 16 + 16 > out_f)
#pragma unroll
        for (int v = 0; v < NV; v++)
          if (tile * 16 + M::row(lane, v) >= out_f) Y[(tile * 16 + M::row(lane, v)) * TA + col(v)] = 0;
    }
    if (l + 2 < nl) {
      if (wave < mlp_tiles(net.out_f[l + 1])) request(net.fw[l + 1], wave, mlp_pieces<T>(out_f));
    } else if (wave < mlp_tiles(in_f)) {
      request(net.bw[l], wave, mlp_pieces<T>(out_f));
    }
    __syncthreads();
    X = Y;
  }
  // ---- the output neuron: every thread takes one atom's share of the features, the shares are added in a fixed order; the
  // delta of the last hidden layer takes the place of its values
  {
    const int in_f = net.in_f[nl - 1], act = net.act[nl - 1], hact = nl > 1 ? net.act[nl - 2] : 0;
    const int rows = mlp_rows(in_f);
    const T* w = net.fw[nl - 1];
    T* parts = X + (nl == 2 ? rows + rows0 : rows) * TA;
    const int np = (int)blockDim.x / TA, t = tid % TA, part = tid / TA;
    T sum = 0;
    for (int k = part; k < in_f; k += np) {
      const T h = X[k * TA + t];
      sum += h * w[k];
      if (act == 0 && nl > 1) X[k * TA + t] = w[k] * mlp_slope<T>(hact, h);
    }
    // the wave's shares of an atom (lanes TA apart) first, then the waves in ascending order
#pragma unroll
    for (int o = TA; o < WAVE; o *= 2) sum += __shfl_xor(sum, o, WAVE);
    if (lane < TA) parts[wave * TA + t] = sum;
    __syncthreads();
    if (tid < TA || act != 0) {
      T y = net.b[nl - 1][0];
      for (int p = 0; p < nw; p++) y += parts[p * TA + t];
      T ys[1] = {y};
      mlp_act<T, 1>(act, ys);
      y = ys[0];
      if (tid < TA && a0 + t < S.Nl) S.e_atom[a0 + t] = (real)y;
      if (act != 0 && nl > 1) {
        const T d = mlp_slope<T>(act, y);
        for (int k = part; k < in_f; k += np) {
          const T h = X[k * TA + t];
          X[k * TA + t] = w[k] * d * mlp_slope<T>(hact, h);
        }
      }
      // (every thread of an atom holds the same value; it goes where the input was, which nobody reads any more -- the
      // shares are still being added by other waves)
      if (nl == 1) X[t] = mlp_slope<T>(act, y);
    }
    if (act != 0 || nl == 1) __syncthreads();
  }
  // ---- backward: d sum(e) / d af = delta / (af + 1e-3)
  auto af_at = [&](int c, int i) -> T {   // (beyond the last atom or fingerprint: the last one)
    const size_t at = (size_t)(a0 + c < S.Nl ? a0 + c : S.Nl - 1);
    i = i < n_af ? i : n_af - 1;
    return (T)(i < S.Ar ? S.af2[at * S.Ar + i] : S.af3[at * S.Aa + (i - S.Ar)]);
  };
  auto put = [&](int c, int i, T delta, T afv) {
    const real g = (real)(delta / (afv + T(1e-3)));
    const size_t at = (size_t)(a0 + c);
    if (i < n_af && a0 + c < S.Nl) (i < S.Ar ? S.g2 + (at * S.Ar + i) : S.g3 + (at * S.Aa + (i - S.Ar)))[0] = g;
  };
  if (nl == 1) {
    const T d = X[my];
    for (int i = tid / TA; i < n_af; i += (int)blockDim.x / TA)
      put(my, i, net.fw[0][i] * d, af_at(my, i));
    return;
  }
  for (int l = nl - 2; l >= 0; l--) {
    const int in_f = net.in_f[l], out_f = net.out_f[l];
    const int np = mlp_pieces<T>(out_f), rows = mlp_rows(in_f), tiles = mlp_tiles(in_f);
    T* const D = X;                           // the layer's deltas
    if (l > 0) X = X - rows * TA;         // the layer's inputs
    const int act = l > 0 ? net.act[l - 1] : 0;
    for (int tile = wave; tile < tiles; tile += nw) {
      if (tile != wave) request(net.bw[l], tile, np);
      T other[NV];   // what the product is multiplied with: the inputs' values, or the fingerprints behind them
      T* const at = X + (tile * 16) * TA;
#pragma unroll
      for (int v = 0; v < NV; v++) other[v] = l > 0 ? at[M::row(lane, v) * TA + col(v)] : af_at(col(v), tile * 16 + M::row(lane, v));
      T acc[NV];
      product(net.bw[l], tile, np, D, acc);
#pragma unroll
      for (int v = 0; v < NV; v++) {
        if (l > 0) at[M::row(lane, v) * TA + col(v)] = acc[v] * mlp_slope<T>(act, other[v]);
        else put(col(v), tile * 16 + M::row(lane, v), acc[v], other[v]);
      }
      if (l > 0 && tile * 16 + 16 > in_f)
#pragma unroll
        for (int v = 0; v < NV; v++)
          if (tile * 16 + M::row(lane, v) >= in_f) at[M::row(lane, v) * TA + col(v)] = 0;
    }
    if (l > 0) {
      if (wave < mlp_tiles(net.in_f[l - 1])) request(net.bw[l - 1], wave, mlp_pieces<T>(in_f));
      __syncthreads();
    }
  }
}

// LDS of a workgroup: the rows of all layers' activations, and a part of the energy sums per thread
template <typename T>
static size_t mlp_lds(int rows, int waves, int ta) {
  return ((size_t)rows * ta + (size_t)waves * WAVE) * sizeof(T);
}
// Most atoms per workgroup for stacks of `rows`: 16 up to about 1200 features in all layers in double precision and 2480 in
// single, 8 up to twice as many (six layers of 430 in single precision, 768 atoms: 160 us, where the host takes 258 ms);
// 0: too many.
template <typename T>
static int mlp_atoms(int rows) {
  for (int ta : {16, 8})
    if (mlp_lds<T>(rows, MLP_WAVES_MAX, ta) <= 160 * 1024) return ta;
  return 0;
}

template <typename T>
static bool upload_net(const StafMlp* mlp, int type, DevMlpNet* net, hipStream_t stream) {
  const int nl = staf_mlp_internal_nlayers(mlp, type);
  if (nl <= 0 || nl > DEV_MLP_MAX_LAYERS) return false;
  net->nl = nl;
  net->n_af = staf_mlp_n_af(mlp, type);
  // every parameter of the stack in one block (one upload, neighbouring pages), each part on a 256-byte boundary
  std::vector<T> host;
  auto place = [&](size_t n) {
    const size_t at = (host.size() + 63) & ~(size_t)63;
    host.resize(at + n, T(0));
    return at;
  };
  // matrix [K, J] in the order in which the waves read it: tile of 16 columns, piece of STEPS steps of four rows,
  // lane (row of the step, column of the tile), step of the piece
  auto tiled = [&](int K, int J, auto&& value) {
    constexpr int STEPS = mlp_steps<T>();
    const int np = mlp_pieces<T>(K);
    const size_t at = place((size_t)mlp_tiles(J) * np * WAVE * STEPS);
    T* out = host.data() + at;
    for (int tile = 0; tile < mlp_tiles(J); tile++)
      for (int p = 0; p < np; p++)
        for (int lane = 0; lane < WAVE; lane++)
          for (int j = 0; j < STEPS; j++, out++) {
            const int k = (p * STEPS + j) * 4 + lane / 16, c = tile * 16 + lane % 16;
            *out = k < K && c < J ? value(k, c) : T(0);
          }
    return at;
  };
  const size_t at_mu = place(net->n_af);
  std::copy_n((const T*)staf_mlp_internal_mu(mlp, type), net->n_af, host.begin() + at_mu);
  size_t at_f[DEV_MLP_MAX_LAYERS], at_b[DEV_MLP_MAX_LAYERS], at_bias[DEV_MLP_MAX_LAYERS];
  int tiles = 1, rows = 0;
  for (int l = 0; l < nl; l++) {
    const void *Wv, *bv;
    if (staf_mlp_internal_layer(mlp, type, l, &net->act[l], &net->in_f[l], &net->out_f[l], &Wv, &bv) != 0) return false;
    const int in_f = net->in_f[l], out_f = net->out_f[l];
    if (in_f != (l ? net->out_f[l - 1] : net->n_af)) return false;
    const T* W = (const T*)Wv;
    if (l + 1 < nl) {
      at_f[l] = tiled(in_f, out_f, [&](int k, int j) { return W[(size_t)k * out_f + j]; });
      at_b[l] = tiled(out_f, in_f, [&](int j, int k) { return W[(size_t)k * out_f + j]; });
      tiles = std::max(tiles, std::max(mlp_tiles(in_f), mlp_tiles(out_f)));
      rows += l == 1 ? std::max(mlp_rows(out_f), mlp_rows(net->n_af)) : mlp_rows(out_f);
    } else {
      at_f[l] = at_b[l] = place(mlp_rows(in_f));
      std::copy_n(W, (size_t)in_f * out_f, host.begin() + at_f[l]);
    }
    at_bias[l] = place(mlp_tiles(out_f) * 16);
    std::copy_n((const T*)bv, out_f, host.begin() + at_bias[l]);
  }
  if (net->out_f[nl - 1] != 1) return false;
  if (nl <= 2) rows += mlp_rows(net->n_af);
  net->tiles = tiles;
  net->rows = rows;
  if (mlp_atoms<T>(rows) == 0) return false;   // a stack too wide for the kernel's LDS is left to the host evaluation
  (void)place((size_t)MLP_AHEAD * WAVE * mlp_steps<T>());   // the pieces a wave requests beyond the last matrix
  T* block = nullptr;
  if (hipMalloc((void**)&block, host.size() * sizeof(T)) != hipSuccess) return false;
  net->mu = block;   // mu leads the block
  // on the model's stream, not the legacy default stream (another host thread may be recording a graph)
  if (hipMemcpyAsync(block, host.data(), host.size() * sizeof(T), hipMemcpyHostToDevice, stream) != hipSuccess ||
      hipStreamSynchronize(stream) != hipSuccess)
    return false;
  for (int l = 0; l < nl; l++) {
    net->fw[l] = block + at_f[l];
    net->bw[l] = block + at_b[l];
    net->b[l] = block + at_bias[l];
  }
  return true;
}

bool dev_mlp_upload(const StafMlp* mlp, int type, DevMlpNet* net, hipStream_t stream) {
  *net = DevMlpNet();
  net->precision = staf_mlp_precision(mlp);
  return net->precision ? upload_net<double>(mlp, type, net, stream) : upload_net<float>(mlp, type, net, stream);
}

void dev_mlp_free(DevMlpNet* net) {
  if (net->mu) (void)hipFree(net->mu);   // one block holds mu and every layer
  *net = DevMlpNet();
}

// ---- networks held by the caller -------------------------------------------------------------------------------

// Sizes of a stack as the kernel wants them; false: a stack it does not take.
template <typename T>
static bool mlp_shape(const DevMlpSource& src, DevMlpNet* net) {
  if (src.nl <= 0 || src.nl > DEV_MLP_MAX_LAYERS || src.n_af <= 0 || src.out_f[src.nl - 1] != 1) return false;
  net->precision = sizeof(T) == 8;
  net->nl = src.nl;
  net->n_af = src.n_af;
  net->tiles = 1;
  net->rows = src.nl <= 2 ? mlp_rows(src.n_af) : 0;
  for (int l = 0; l < src.nl; l++) {
    const int in_f = l ? src.out_f[l - 1] : src.n_af, out_f = src.out_f[l];
    if (out_f <= 0 || (size_t)mlp_rows(in_f) * mlp_rows(out_f) > (1u << 28)) return false;
    net->act[l] = src.act[l]; net->in_f[l] = in_f; net->out_f[l] = out_f;
    if (l + 1 == src.nl) break;
    net->tiles = std::max(net->tiles, std::max(mlp_tiles(in_f), mlp_tiles(out_f)));
    net->rows += l == 1 ? std::max(mlp_rows(out_f), mlp_rows(src.n_af)) : mlp_rows(out_f);
  }
  return mlp_atoms<T>(net->rows) != 0;
}

// elements of matrix [K, J] in tile order
template <typename T>
__host__ __device__ inline size_t mlp_tiled(int K, int J) {
  return (size_t)mlp_tiles(J) * mlp_pieces<T>(K) * WAVE * mlp_steps<T>();
}
static size_t mlp_place(size_t at) { return (at + 63) & ~(size_t)63; }

template <typename T>
static size_t mlp_layout(const DevMlpSource& src, T* block, DevMlpNet* net, PackPart* parts, int* n_parts) {
  size_t at = 0;
  int n = 0;
  auto part = [&](const void* from, int K, int J, int kind, size_t elements) -> T* {
    at = mlp_place(at);
    T* to = block ? block + at : nullptr;
    if (parts) parts[n] = {from, to, K, J, kind};
    n++;
    at += elements;
    return to;
  };
  net->mu = part(src.mu, src.n_af, src.n_af, PACK_COPY, src.n_af);
  for (int l = 0; l < src.nl; l++) {
    const int in_f = net->in_f[l], out_f = net->out_f[l];
    if (l + 1 < src.nl) {
      net->fw[l] = part(src.W[l], in_f, out_f, PACK_TILES, mlp_tiled<T>(in_f, out_f));
      net->bw[l] = part(src.W[l], in_f, out_f, PACK_TILES_T, mlp_tiled<T>(out_f, in_f));
    } else {
      net->fw[l] = net->bw[l] = part(src.W[l], in_f, mlp_rows(in_f), PACK_COPY, mlp_rows(in_f));
    }
    net->b[l] = part(src.b[l], out_f, mlp_tiles(out_f) * 16, PACK_COPY, mlp_tiles(out_f) * 16);
  }
  if (n_parts) *n_parts = n;
  // the pieces a wave requests beyond the last matrix are read and not used
  return mlp_place(mlp_place(at) + (size_t)MLP_AHEAD * WAVE * mlp_steps<T>());
}

template <typename T>
size_t dev_mlp_block(const DevMlpSource& src) {
  DevMlpNet net;
  return mlp_shape<T>(src, &net) ? mlp_layout<T>(src, nullptr, &net, nullptr, nullptr) : 0;
}
template size_t dev_mlp_block<float>(const DevMlpSource&);
template size_t dev_mlp_block<double>(const DevMlpSource&);

template <typename T>
int dev_mlp_plan(const DevMlpSource& src, T* block, DevMlpNet* net, PackPart* parts) {
  int n = 0;
  *net = DevMlpNet();
  if (!mlp_shape<T>(src, net)) return 0;
  (void)mlp_layout<T>(src, block, net, parts, &n);
  return n;
}
template int dev_mlp_plan<float>(const DevMlpSource&, float*, DevMlpNet*, PackPart*);
template int dev_mlp_plan<double>(const DevMlpSource&, double*, DevMlpNet*, PackPart*);

constexpr int PACK_BLOCK = 256;
static_assert(PACK_BLOCK == STEP_TABLE_BLOCK, "one launch");
template <typename T>
struct PackArgs {
  int n, first[PACK_PARTS + 1];   // workgroups of a part; before the first one's those of the tables, which take longest
  PackPart part[PACK_PARTS];
  int nt;
  StepTablePart<T> table[NT_MAX];
};
template <typename T>
__host__ __device__ inline size_t pack_elements(const PackPart& p) {
  return p.kind == PACK_TILES ? mlp_tiled<T>(p.K, p.J) : p.kind == PACK_TILES_T ? mlp_tiled<T>(p.J, p.K) : (size_t)p.J;
}
// A thread per element of the destination: the order of upload_net's tiles.  Bound by its launch and the first read of the
// parameters: the two networks of a 60-140-140-1 stack in double precision are 0.9 MB, and the two tables of exponentials beside
// them 0.3 MB for exponents up to 2 and 14 channels in use of 40, 1.2 MB for trained ones (up to 10: 1025 and 513 rows).  Between
// events, four frames of 729 atoms: the networks alone 6.9 us, with the tables 7.6 and 8.5 (as wide as all 40 channels, with maxima in
// double precision and divisions per entry, 8.8 and 11.7).
template <typename T>
__global__ __launch_bounds__(PACK_BLOCK) void mlp_pack_kernel(const PackArgs<T> A) {
  if ((int)blockIdx.x < A.first[0]) {
    const int q = (int)blockIdx.x / STEP_TABLE_PARTS<T>, nsig = 2 * A.nt - 1;
    step_table_body<T>(A.table[q / nsig], A.nt, q % nsig, (int)blockIdx.x % STEP_TABLE_PARTS<T>, STEP_TABLE_PARTS<T>);
    return;
  }
  int e = 0;
  while (e + 1 < A.n && (int)blockIdx.x >= A.first[e + 1]) e++;
  const PackPart& p = A.part[e];
  const size_t i = (size_t)((int)blockIdx.x - A.first[e]) * PACK_BLOCK + threadIdx.x;
  if (i >= pack_elements<T>(p)) return;
  const T* src = (const T*)p.src;
  T v = 0;
  if (p.kind == PACK_COPY || p.kind == PACK_SQUARE) {
    if ((int)i < p.K) v = src[i];
    if (p.kind == PACK_SQUARE) v *= v;
  } else {
    constexpr int STEPS = mlp_steps<T>();
    const bool flip = p.kind == PACK_TILES_T;
    const int K = flip ? p.J : p.K, J = flip ? p.K : p.J, np = mlp_pieces<T>(K);   // of the matrix as it is read
    const int j = (int)(i % STEPS), lane = (int)(i / STEPS % WAVE);
    const size_t tp = i / (STEPS * WAVE);
    const int k = ((int)(tp % np) * STEPS + j) * 4 + lane / 16, c = (int)(tp / np) * 16 + lane % 16;
    if (k < K && c < J) v = flip ? src[(size_t)c * p.J + k] : src[(size_t)k * p.J + c];
  }
  ((T*)p.dst)[i] = v;
}

template <typename T>
int dev_mlp_pack(const PackPart* parts, int n, const StepTablePart<T>* tables, int n_tables, int nt, hipStream_t stream) {
  for (int at = 0; at < n; at += PACK_PARTS) {
    PackArgs<T> A = {};
    size_t blocks = 0, lds = 0;
    A.nt = nt;
    if (at == 0) {
      for (int k = 0; k < n_tables; k++) {
        A.table[k] = tables[k];
        lds = std::max(lds, step_table_lds<T>(tables[k].Aa));
      }
      blocks = (size_t)n_tables * (2 * nt - 1) * STEP_TABLE_PARTS<T>;
    }
    for (A.n = 0; A.n < PACK_PARTS && at + A.n < n; A.n++) {
      A.part[A.n] = parts[at + A.n];
      A.first[A.n] = (int)blocks;
      blocks += (pack_elements<T>(A.part[A.n]) + PACK_BLOCK - 1) / PACK_BLOCK;
    }
    A.first[A.n] = (int)blocks;
    if (blocks > 0x7fffffff) return STAF_E_LIMIT;
    KernelTimer kt_("mlp_pack_kernel", stream);
    if (blocks) hipLaunchKernelGGL(mlp_pack_kernel<T>, dim3((unsigned)blocks), dim3(PACK_BLOCK), lds, stream, A);
  }
  return hipGetLastError() == hipSuccess ? STAF_OK : STAF_E_HIP;
}
template int dev_mlp_pack<float>(const PackPart*, int, const StepTablePart<float>*, int, int, hipStream_t);
template int dev_mlp_pack<double>(const PackPart*, int, const StepTablePart<double>*, int, int, hipStream_t);

template <typename T, typename real, int TA>
static int eval_nets_by(const DevMlpCall<real>* calls, int n, int rows, int tiles, hipStream_t stream) {
  MlpArgs<T, real> A = {};
  int blocks = 0;
  for (int c = 0; c < n; c++) {
    const DevMlpCall<real>& C = calls[c];
    if (C.Nl <= 0) continue;
    const DevMlpNet& net = *C.net;
    MlpSpecies<real>& S = A.sp[A.ns];
    S.af2 = C.af2; S.af3 = C.af3; S.e_atom = C.e_atom; S.g2 = C.g2; S.g3 = C.g3;
    S.Ar = C.Ar; S.Aa = C.Aa; S.Nl = C.Nl; S.first = blocks;
    blocks += (C.Nl + TA - 1) / TA;
    MlpNet<T>& N = A.net[A.ns++];
    N.nl = net.nl; N.n_af = net.n_af; N.mu = (const T*)net.mu;
    for (int l = 0; l < net.nl; l++) {
      N.act[l] = net.act[l]; N.in_f[l] = net.in_f[l]; N.out_f[l] = net.out_f[l];
      N.fw[l] = (const T*)net.fw[l]; N.bw[l] = (const T*)net.bw[l]; N.b[l] = (const T*)net.b[l];
    }
  }
  if (blocks == 0) return STAF_OK;
  // A wave per tile of the widest product while a CU has one workgroup at most, or two small ones (double precision,
  // 60-140-140-1: 22.0 us with nine waves, 24.2 with five); two tiles per wave where it has several, whose products and
  // activations then overlap (1024 workgroups: 76.7 us with nine waves, 60.3 with five, 72 with three).
  const int waves = std::min(MLP_WAVES_MAX, std::max(2, blocks <= (TA == 16 ? 256 : 512) ? tiles : (tiles + 1) / 2));
  const size_t lds = mlp_lds<T>(rows, waves, TA);
  if (!lds_request(mlp_kernel<T, real, TA>, lds)) return STAF_E_LIMIT;
  KernelTimer kt_("mlp_kernel", stream);
  hipLaunchKernelGGL((mlp_kernel<T, real, TA>), dim3(blocks), dim3(waves * WAVE), lds, stream, A);
  return hipGetLastError() == hipSuccess ? STAF_OK : STAF_E_HIP;
}

template <typename T, typename real>
static int eval_nets(const DevMlpCall<real>* calls, int n, hipStream_t stream) {
  int rows = 0, tiles = 1, by4 = 0, by8 = 0;   // workgroups of four and of eight atoms
  for (int c = 0; c < n; c++) {
    if (calls[c].Nl <= 0) continue;
    rows = std::max(rows, calls[c].net->rows);
    tiles = std::max(tiles, calls[c].net->tiles);
    by4 += (calls[c].Nl + 3) / 4;
    by8 += (calls[c].Nl + 7) / 8;
  }
  // A launch of few atoms lasts as long as a workgroup's chain of products, which is shorter for fewer atoms as long as the
  // workgroups find a CU each: double precision by fours up to 256 workgroups (96 to 768 atoms 22.5 -> 14.1 us) and by
  // eights up to as many (1500 atoms by 16 / 8 / 4: 23.3 / 17.8 / 23.6; 3072: 24 / 29 / 34).  In single precision, whose
  // weights are half the bytes, two small workgroups share a CU (96 to 768 atoms 17.3 -> 12.3, 1500 atoms 17.8 / 15.7 / 15.2,
  // 3072 18.4 / 19.8 / 18.8).  (Times between the library's events.)  The lines are those of 60-140-140-1 stacks.  Others, by 16 /
  // 8 / 4, double: 60-300-300-1, 768 atoms 44.4 / 30.2 / 27.9, 1500 44.2 / 31.2 / 48.2, 2046 44.6 / 53.4 / 50.7; 60-32-32-1,
  // 768 14.1 / 11.4 / 10.1, 1500 13.7 / 11.4 / 10.6, 2046 13.8 / 11.7 / 10.8, 4096 18.6 / 15.5 / 13.6; single: 60-300-300-1, 768
  // 30.1 / 24.9 / 19.9, 1500 30.3 / 26.4 / 29.7, 2046 30.5 / 42.9 / 30.9; 60-32-32-1, 2046 12.9 / 11.6 / 10.3, 4096 16.4 / 14.8 / 12.4.
  // Narrow stacks' weights cost less than their chains, and few atoms pay for more workgroups than this; so do eight for 4096
  // atoms of 60-140-140-1 in double (34.0 / 30.6 / 42.8).
  const int most = mlp_atoms<T>(rows);
  if (most == 0) return STAF_E_LIMIT;
  if (by4 <= (sizeof(T) == 8 ? 256 : 512)) return eval_nets_by<T, real, 4>(calls, n, rows, tiles, stream);
  if (most == 8 || (sizeof(T) == 8 && by8 <= 256)) return eval_nets_by<T, real, 8>(calls, n, rows, tiles, stream);
  return eval_nets_by<T, real, 16>(calls, n, rows, tiles, stream);
}

template <typename real>
int dev_mlp_eval(const DevMlpCall<real>* calls, int n, hipStream_t stream) {
  if (n <= 0 || n > NT_MAX) return STAF_E_BAD_ARG;
  for (int c = 0; c < n; c++)
    if (calls[c].Ar + calls[c].Aa != calls[c].net->n_af || calls[c].net->precision != calls[0].net->precision)
      return STAF_E_BAD_ARG;
  if constexpr (sizeof(real) == 4) {
    return calls[0].net->precision ? STAF_E_BAD_ARG : eval_nets<float>(calls, n, stream);
  } else {
    return calls[0].net->precision ? eval_nets<double>(calls, n, stream) : eval_nets<float>(calls, n, stream);
  }
}
template int dev_mlp_eval<float>(const DevMlpCall<float>*, int, hipStream_t);
template int dev_mlp_eval<double>(const DevMlpCall<double>*, int, hipStream_t);

}  // namespace staf
