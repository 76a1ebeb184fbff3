// Device-resident per-species MLP of the MD entry (staf_mlp_dev.hip).
#pragma once
#include "staf_common.hpp"
#include "staf_mlp_internal.h"

namespace staf {

constexpr int DEV_MLP_MAX_LAYERS = 8;

struct DevMlpNet {
  int precision = 0;   // 0: float weights and arithmetic, 1: double
  int nl = 0, n_af = 0;
  int act[DEV_MLP_MAX_LAYERS] = {0}, in_f[DEV_MLP_MAX_LAYERS] = {0}, out_f[DEV_MLP_MAX_LAYERS] = {0};
  void* fw[DEV_MLP_MAX_LAYERS] = {nullptr};   // weights in matrix-tile order (the last layer's: a plain column)
  void* bw[DEV_MLP_MAX_LAYERS] = {nullptr};   // transposed weights in matrix-tile order (none for the last layer)
  void* b[DEV_MLP_MAX_LAYERS] = {nullptr};
  void* mu = nullptr;                         // the block that holds all of them starts here
  int rows = 0;                               // features of all layers as they lie in LDS
  int tiles = 0;                              // tiles of 16 features of the widest product
};

// One species of a network launch: fingerprints af2 [Nl, Ar], af3 [Nl, Aa] -> atomic energies e_atom [Nl] and
// d sum(e) / d af as g2 [Nl, Ar], g3 [Nl, Aa].
template <typename real>
struct DevMlpCall {
  const DevMlpNet* net;
  const real *af2, *af3;
  real *e_atom, *g2, *g3;
  int Ar, Aa, Nl;
};

bool dev_mlp_upload(const StafMlp* mlp, int type, DevMlpNet* net, hipStream_t stream);   // false: not representable (fall back to host)
void dev_mlp_free(DevMlpNet* net);
// The networks of n species (at most NT_MAX, of one precision; species without atoms are skipped) in one launch; the
// arithmetic is in the networks' precision (float64 fingerprints with a float32 network: like the host evaluation).
template <typename real>
int dev_mlp_eval(const DevMlpCall<real>* calls, int n, hipStream_t stream);

// Networks whose parameters are device tensors of a caller's program, laid out for the launch on every call.
struct DevMlpSource {
  int nl, n_af, act[DEV_MLP_MAX_LAYERS], out_f[DEV_MLP_MAX_LAYERS];
  const void *mu, *W[DEV_MLP_MAX_LAYERS], *b[DEV_MLP_MAX_LAYERS];   // mu [n_af], W [in, out], b [out]
};
// Elements of the block that holds a laid-out network; 0: a stack the kernel does not take.
template <typename T>
size_t dev_mlp_block(const DevMlpSource& src);
// A part of a device block that is written from a device tensor.
struct PackPart {
  const void* src;
  void* dst;
  int K, J, kind;   // PACK_*
};
// COPY / SQUARE: K elements, zeros up to J; TILES: matrix [K, J] in tile order; TILES_T: the transpose [J, K] of src [K, J]
// in tile order
enum { PACK_COPY, PACK_SQUARE, PACK_TILES, PACK_TILES_T };
constexpr int PACK_PARTS = 64;
// Describes the network laid out in `block` and appends the parts that fill it (at most 3 per layer and one).
template <typename T>
int dev_mlp_plan(const DevMlpSource& src, T* block, DevMlpNet* net, PackPart* parts);
// The same launch writes the tables of n_tables species (staf_step.hpp).
template <typename T>
int dev_mlp_pack(const PackPart* parts, int n, const StepTablePart<T>* tables, int n_tables, int nt, hipStream_t stream);

}  // namespace staf
