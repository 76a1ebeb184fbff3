// Energies, forces and virials of a batch of frames from one call: staf_op_frames of include/staf_ops.h, the native form
// of staf_full_inference.full_test (STAF/staf_models/staf_model_inference_full.py:84-143).
//
// Six launches (seven with a cell list), each over the centres of all species of all frames: the caller's parameters laid
// out for the kernels, descriptors (radial-only: no tensor of the angular buffer's width exists), fingerprints, networks,
// slot forces, collection.  Built from single ops by a Python program the same call was 103 launches, most of them
// shorter than the time the host needs to issue one: four frames of 768 atoms took 1590 us a call.
// Everything lies in a block of the caller's (staf_op_frames_work), so that nothing is allocated here and the block is
// the caller's allocator's to reuse in the order of the stream.
#include "staf_common.hpp"
#include "staf_mlp_dev.hpp"
#include "staf_step.hpp"

#include <vector>

namespace staf {

template <typename real>
struct FramesPlan {
  size_t bytes = 0;
  size_t raddescr, des3bsupp, der2b, der3bsupp, unit, slots, self, vpart, e_atom, intmap2b, numtriplet;
  size_t af2[NT_MAX], af3[NT_MAX], g2[NT_MAX], g3[NT_MAX], net[NT_MAX], emb2b[NT_MAX], emb3b[NT_MAX], table[NT_MAX];
  bool rows = false;   // the fingerprints' launch reads the species' tables
};

static DevMlpSource net_source(const StafFramesSpecies& s) {
  DevMlpSource n = {};
  n.nl = s.n_layers;
  n.n_af = s.nalpha_r + s.nsmooth_a;
  n.mu = s.mu;
  for (int l = 0; l < s.n_layers; l++) {
    n.act[l] = s.activation[l];
    n.out_f[l] = s.out_f[l];
    n.W[l] = s.W[l];
    n.b[l] = s.b[l];
  }
  return n;
}

// the map that the library's own search writes to `im2`
static TransposeRef own_map(const void* im2) {
  TransposeRef t;
  t.symmetric = 1;
  t.full = (const int*)im2;
  return t;
}

// Where everything lies in the caller's block; STAF_E_LIMIT: a model or a geometry the launches do not take.
template <typename real>
static int frames_plan(const DescConfig<real>& c, int nf, int N, int nt, const StafFramesSpecies* sp, FramesPlan<real>* P) {
  if (!c.ready) return STAF_E_NOT_CONSTRUCTED;
  if (nf <= 0 || N <= 0 || nt <= 0 || !sp) return STAF_E_BAD_ARG;
  if (nt > NT_MAX) return STAF_E_LIMIT;
  auto place = [&](size_t bytes) {
    const size_t at = P->bytes;
    P->bytes = (at + bytes + 255) & ~(size_t)255;
    return at;
  };
  const size_t rows = (size_t)nf * N, nr = c.nr;
  if (rows * nr > (1u << 30)) return STAF_E_LIMIT;   // (row numbers are 32-bit in the launches' grids)
  P->raddescr = place(rows * nr * sizeof(real));
  P->des3bsupp = place(rows * nr * sizeof(real));
  P->der2b = place(rows * 3 * nr * sizeof(real));
  P->der3bsupp = place(rows * 3 * nr * sizeof(real));
  P->unit = place(rows * 4 * nr * sizeof(real));
  P->slots = place(rows * 3 * nr * sizeof(real));
  P->self = place(rows * 3 * sizeof(real));
  P->vpart = place(rows * 9 * sizeof(real));
  P->e_atom = place(rows * sizeof(real));
  P->intmap2b = place(rows * (nr + 1) * sizeof(int));
  P->numtriplet = place(rows * sizeof(int));
  RowsLaunch<real> form;
  for (int k = 0; k < nt; k++) form.add(c.nr, c.na, nt, sp[k].nalpha_r, sp[k].nsmooth_a, (long long)nf * sp[k].n_local);
  // Up to 512 centres of one or two species in double precision the tables cost the parameters' launch what the fingerprints gain by
  // them, or more: both launches, in the staged form and by rows, exponents up to 2 and trained ones (up to 10), us:
  //                            centres  125                  343                  512
  //   one species                       24.3 / 26.4          29.2 / 28.6          32.4 / 33.4
  //   two, channels in blocks           19.8 / 20.0, 21.8    22.2 / 21.4, 23.0    25.3 / 23.9
  //   two, all channels in all classes  31.0 / 31.6, 36.7    36.3 / 35.3, 39.3    39.6 / 42.0
  //   three, in blocks                  25.2 / 23.7, 25.6    28.1 / 25.0, 27.4
  P->rows = form.waves() > 0 && (sizeof(real) == 4 || nt > 2 || form.centres > 512);
  long long sum = 0;
  for (int k = 0; k < nt; k++) {
    const StafFramesSpecies& s = sp[k];
    if (s.n_local < 0 || s.nalpha_r <= 0 || s.nsmooth_a <= 0) return STAF_E_BAD_ARG;
    if (s.n_layers <= 0 || s.n_layers > DEV_MLP_MAX_LAYERS) return STAF_E_LIMIT;
    sum += s.n_local;
    const size_t n = (size_t)nf * s.n_local, block = dev_mlp_block<real>(net_source(s));
    if (block == 0) return STAF_E_LIMIT;
    P->af2[k] = place(n * s.nalpha_r * sizeof(real));
    P->af3[k] = place(n * s.nsmooth_a * sizeof(real));
    P->g2[k] = place(n * s.nalpha_r * sizeof(real));
    P->g3[k] = place(n * s.nsmooth_a * sizeof(real));
    P->emb2b[k] = place((size_t)nt * s.nalpha_r * sizeof(real));
    P->emb3b[k] = place((size_t)nt * (nt + 1) / 2 * s.nsmooth_a * sizeof(real));
    P->net[k] = place(block * sizeof(real));
    P->table[k] = place(P->rows && s.n_local > 0 ? step_table_reals<real>(nt, s.nsmooth_a) * sizeof(real) : 0);
  }
  return sum == N ? STAF_OK : STAF_E_BAD_ARG;
}

template <typename real>
static int frames_work(int nf, int N, int nt, const StafFramesSpecies* sp, size_t* bytes) {
  if (!bytes) return STAF_E_BAD_ARG;
  FramesPlan<real> P;
  const int rc = frames_plan<real>(desc_current<real>(), nf, N, nt, sp, &P);
  *bytes = rc == STAF_OK ? P.bytes : 0;
  return rc;
}

template <typename real>
static int frames(const real* pos, const real* box, int nf, int N, int nt, const StafFramesSpecies* sp, const int* type_map,
                  void* work, size_t work_bytes, real* energy, real* force, real* virial, hipStream_t stream) {
  const DescConfig<real> c = desc_current<real>();
  FramesPlan<real> P;
  int rc = frames_plan<real>(c, nf, N, nt, sp, &P);
  if (rc != STAF_OK) return rc;
  if (!pos || !box || !type_map || !work || work_bytes < P.bytes || !energy || !virial) return STAF_E_BAD_ARG;
  for (int k = 0; k < nt; k++)   // (known before anything is launched: the caller has another way)
    if (force && sp[k].n_local > 0 && !step_forces_fits<real>(c.nr, nt, sp[k].nalpha_r, sp[k].nsmooth_a)) return STAF_E_LIMIT;
  char* const w = (char*)work;
  auto at = [&](size_t offset) { return (real*)(w + offset); };
  StepSpecies<real> S[NT_MAX];
  DevMlpNet nets[NT_MAX];
  DevMlpCall<real> calls[NT_MAX];
  std::vector<PackPart> parts;
  StepTablePart<real> tables[NT_MAX];
  int n = 0, first = 0, n_tables = 0;
  for (int k = 0; k < nt; first += sp[k].n_local, k++) {
    const StafFramesSpecies& s = sp[k];
    if (s.n_local == 0) continue;
    bool whole = s.alpha2b && s.alpha3b && s.type_emb2b && s.type_emb3b && s.mu;
    for (int l = 0; l < s.n_layers; l++) whole = whole && s.W[l] && s.b[l];
    if (!whole) return STAF_E_BAD_ARG;
    const int e2 = nt * s.nalpha_r, e3 = nt * (nt + 1) / 2 * s.nsmooth_a;
    PackPart mine[2 + 3 * DEV_MLP_MAX_LAYERS + 1];
    mine[0] = {s.type_emb2b, at(P.emb2b[k]), e2, e2, PACK_SQUARE};
    mine[1] = {s.type_emb3b, at(P.emb3b[k]), e3, e3, PACK_SQUARE};
    const int m = dev_mlp_plan<real>(net_source(s), at(P.net[k]), &nets[n], mine + 2);
    parts.insert(parts.end(), mine, mine + 2 + m);
    S[n] = {first, s.n_local, s.nalpha_r, s.nsmooth_a, (const real*)s.alpha2b, (const real*)s.alpha3b, at(P.emb2b[k]),
            at(P.emb3b[k]), at(P.af2[k]), at(P.af3[k]), at(P.g2[k]), at(P.g3[k]), nullptr};
    if (P.rows) {
      S[n].table = at(P.table[k]);
      tables[n_tables++] = {S[n].alpha3b, (const real*)s.type_emb3b, at(P.table[k]),
                            step_table_reals<real>(nt, s.nsmooth_a), s.nsmooth_a, 1};
    }
    calls[n] = {&nets[n], S[n].af2, S[n].af3, at(P.e_atom) + (size_t)nf * first, S[n].g2, S[n].g3, S[n].Ar, S[n].Aa,
                nf * s.n_local};
    n++;
  }
  DeviceState* st = device_state(stream);
  if (!st) return reserve_failure(stream);
  const StepRows<real> R = {at(P.raddescr), at(P.des3bsupp), at(P.der2b), at(P.der3bsupp), at(P.unit),
                            (int*)(w + P.intmap2b), (int*)(w + P.numtriplet), c.nr, c.na, nf, N, own_map(w + P.intmap2b)};
  {
    DeferStatus defer;   // conditions the kernels detect are read once, behind the last launch
    if ((rc = dev_mlp_pack<real>(parts.data(), (int)parts.size(), tables, n_tables, nt, stream)) != STAF_OK) return rc;
    rc = desc_launch<real>(c, pos, box, nf, N, N, nullptr, &R.tr, 0, at(P.raddescr), nullptr, at(P.des3bsupp),
                           (int*)(w + P.intmap2b), nullptr, at(P.der2b), nullptr, at(P.der3bsupp),
                           (int*)(w + P.numtriplet), at(P.unit), stream);
    if (rc != STAF_OK) return rc;
    if ((rc = step_fingerprints<real>(S, n, R, type_map, nt, stream)) != STAF_OK) return rc;
    if ((rc = dev_mlp_eval<real>(calls, n, stream)) != STAF_OK) return rc;
    real* const vpart = force ? at(P.vpart) : nullptr;
    if (force && (rc = step_forces<real>(S, n, R, type_map, nt, at(P.slots), at(P.self), vpart, stream)) != STAF_OK) return rc;
    const StepCollect<real> out = {at(P.slots), at(P.self), vpart, at(P.e_atom), force, nullptr, energy, virial, 1};
    if ((rc = step_collect<real>(S, n, R, N, out, stream)) != STAF_OK) return rc;
  }
  return finish_op(st, stream);
}

}  // namespace staf

extern "C" {

int staf_op_frames_work_f32(int nf, int N, int nt, const StafFramesSpecies* species, size_t* bytes) {
  return staf::frames_work<float>(nf, N, nt, species, bytes);
}
int staf_op_frames_work_f64(int nf, int N, int nt, const StafFramesSpecies* species, size_t* bytes) {
  return staf::frames_work<double>(nf, N, nt, species, bytes);
}
int staf_op_frames_f32(const float* positions, const float* boxer, int nf, int N, int nt, const StafFramesSpecies* species,
                       const int* type_map, void* work, size_t work_bytes, float* energy, float* force, float* virial,
                       void* stream) {
  return staf::frames<float>(positions, boxer, nf, N, nt, species, type_map, work, work_bytes, energy, force, virial,
                             (hipStream_t)stream);
}
int staf_op_frames_f64(const double* positions, const double* boxer, int nf, int N, int nt,
                       const StafFramesSpecies* species, const int* type_map, void* work, size_t work_bytes, double* energy,
                       double* force, double* virial, void* stream) {
  return staf::frames<double>(positions, boxer, nf, N, nt, species, type_map, work, work_bytes, energy, force, virial,
                              (hipStream_t)stream);
}

}  // extern "C"
