// MD-facing entry (LAMMPS `pair_style staf`): staf_load / staf_compute / staf_free of include/staf.h.
//
// Host logic follows libstaf/src/staf_api.cpp:192-412 (validation and return codes, species-sorted packing of
// the owned atoms, ghosts appended, neighbour-index remapping, un-packing of forces) and the step order of
// calculateforces (libstaf/vendor/jmd/nn_nn_mlp.cu:838-889): neighbour list (own, or the caller's with no
// periodic wrap) -> descriptors -> fingerprints of every species -> MLP -> 2-body + 3-body forces with virial.
// Everything on the GPU runs in float64.  The path is fused in the sense that matters for memory: no tensor of the
// angular buffer's width exists.  The descriptor kernel runs radial-only and leaves, per centre, its sorted
// neighbour list with unit vectors, 1/r, cutoff values and their gradients (nr-wide rows); the 3-body fingerprint
// and force kernels rebuild every triplet's angular descriptor and Jacobian from those rows in LDS.  HBM traffic of a
// call is positions and types in, forces out, and those nr-wide rows.  The MLP is the per-species Dense stack,
// evaluated on the GPU between the fingerprint and the force kernels (or on the host, staf_mlp.cpp, on request).
#include "staf_common.hpp"
#include "staf_reduce.hpp"
#include "staf_mlp_dev.hpp"
#include "staf_step.hpp"
#include "../../include/staf.h"
#include "../../include/staf_mlp.h"

#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <string>
#include <algorithm>
#include <vector>

namespace {

template <typename T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
  bool reserve(size_t want) {
    if (want <= n) return true;
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
    if (hipMalloc((void**)&p, want * sizeof(T)) != hipSuccess) return false;
    n = want;
    return true;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
};

// Pinned host staging (allocated pinned, never registered): one block for everything a call sends, one for what it
// brings back.  Kernels copy them (call_in_kernel, call_out_kernel).
template <typename T>
struct PinBuf {
  T* p = nullptr;
  T* dev = nullptr;   // the block as the device sees it
  size_t n = 0;
  bool reserve(size_t want) {
    if (want <= n) return true;
    release();
    want += want / 4;
    if (hipHostMalloc((void**)&p, want * sizeof(T), hipHostMallocDefault) != hipSuccess) {
      p = nullptr;
      return false;
    }
    if (hipHostGetDevicePointer((void**)&dev, p, 0) != hipSuccess) {
      release();
      return false;
    }
    n = want;
    return true;
  }
  void release() {
    if (p) (void)hipHostFree(p);
    p = dev = nullptr;
    n = 0;
  }
};

// A call's input block from the pinned host memory, and its results back.  Bound by latency: three copies by the runtime
// (input; results; error words) and the wait for the stream took 40 us of a 768-atom call and 44 of a 6144-atom one around
// an otherwise empty chain of kernels, the two kernels and flags that the host watches 19 and 24 (24576 atoms: 60 and 43).
// MD calls of 96, 768, 6144 and 24576 atoms: 90 -> 82, 136 -> 107, 417 -> 387 and 1340 -> 1313 us; with a caller's list,
// 1500 and 6144 atoms: 223 -> 213 and 553 -> 529.
// They also take the positions from the caller's order to the species-sorted slots and the forces back, and a changed order
// and species along, which the host did in loops over the atoms and with a copy of its own: calls of 768, 6144 and 24576
// atoms in an order that changes every time 101 -> 99, 386 -> 370 and 1299 -> 1245 us, with a caller's list, whose ghosts
// change species, 1500 and 6144 atoms 209 -> 170 and 533 -> 490.
constexpr int IO_THREADS = 256, IN_BLOCKS = 256, OUT_BLOCKS = 64;
// The first n3 doubles are positions in the caller's order and go to the atoms' slots; the rest is copied as it is.  new_order:
// the slots have changed; their numbers and the atoms' species lie in host memory too, and further workgroups keep them on
// the device for the calls that follow: order_d (and behind it the owned slots' atoms) and the slots' species.
struct CallOrder {
  const int* new_order;   // [slot of every atom nall | species of every atom nall] or null
  int *order_d, *type_map;
  int nall, nlocal, blocks;   // blocks: workgroups that copy the first part
};
__global__ __launch_bounds__(IO_THREADS) void call_in_kernel(const double2* __restrict__ host, double* __restrict__ dev, int n3,
                                                             int n, const CallOrder O) {
  if ((int)blockIdx.x < O.blocks) {
    const int* const slot_of = O.new_order ? O.new_order : O.order_d;
    for (int i = blockIdx.x * IO_THREADS + threadIdx.x; i < n; i += O.blocks * IO_THREADS) {
      const double2 v = host[i];
      const int e = 2 * i;
      dev[e < n3 ? 3 * slot_of[e / 3] + e % 3 : e] = v.x;
      dev[e + 1 < n3 ? 3 * slot_of[(e + 1) / 3] + (e + 1) % 3 : e + 1] = v.y;
    }
  } else {
    const int step = (gridDim.x - O.blocks) * IO_THREADS;
    for (int i = (blockIdx.x - O.blocks) * IO_THREADS + threadIdx.x; i < O.nall; i += step) {
      const int s = O.new_order[i], t = O.new_order[O.nall + i];
      O.order_d[i] = s;
      O.type_map[s] = t;
      if (i < O.nlocal) O.order_d[O.nall + s] = i;
    }
  }
}
// Forces in the caller's order, the rest as it is.
// The stream's error word goes along.  A workgroup's flag says that everything it copied has arrived: its threads' stores are released
// to the host before the flag is written.
__global__ __launch_bounds__(IO_THREADS) void call_out_kernel(const double* __restrict__ dev, double2* __restrict__ host,
                                                              const int* __restrict__ slot_of, int n3, int n, int* status,
                                                              int* status_h, unsigned* flags, unsigned call) {
  for (int i = blockIdx.x * IO_THREADS + threadIdx.x; i < n; i += gridDim.x * IO_THREADS) {
    double2 v;
    const int e = 2 * i;
    v.x = dev[e < n3 ? 3 * slot_of[e / 3] + e % 3 : e];
    v.y = dev[e + 1 < n3 ? 3 * slot_of[(e + 1) / 3] + (e + 1) % 3 : e + 1];
    host[i] = v;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0)
    *status_h = __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(&flags[blockIdx.x], call, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void add_into_kernel(double* dst, const double* src, int n) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) dst[e] += src[e];
}

// Host-to-device copy that is complete when it returns, on a stream of the model: a blocking hipMemcpy runs on the
// legacy default stream, and work on that stream while another host thread records a graph is refused by the runtime
// and spoils that thread's recording.
static bool upload_sync(void* dst, const void* src, size_t bytes, hipStream_t stream) {
  return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream) == hipSuccess &&
         hipStreamSynchronize(stream) == hipSuccess;
}

bool read_numbers(const std::string& path, std::vector<double>& out, int* rows) {
  FILE* f = fopen(path.c_str(), "r");
  if (!f) return false;
  out.clear();
  int nrows = 0;
  char line[1 << 16];
  while (fgets(line, sizeof(line), f)) {
    char* s = line;
    int got = 0;
    for (;;) {
      char* e;
      double v = strtod(s, &e);
      if (e == s) break;
      out.push_back(v);
      s = e;
      got++;
    }
    if (got) nrows++;
  }
  fclose(f);
  if (rows) *rows = nrows;
  return !out.empty();
}

}  // namespace

struct StafModel {
  StafOptions opt;
  std::string dir;
  StafMlp* mlp = nullptr;
  int nt = 0, ntc = 0, nr = 60, na = 1770;
  double Rc = 4.5, Ra = 4.5, Rs = 2.25;
  std::vector<int> Ar, Aa;
  std::vector<DevBuf<double>> alpha2b, alpha3b, emb2b, emb3b, table;
  staf::DescConfig<double> cfg;
  hipStream_t stream = nullptr;            // the call's stream
  // device buffers
  // in_d  = [pos nall*3 | box 6], with a caller's list behind them, in ints,
  //         [howmany nlocal | rows nlocal*pitch]
  //         (in_h the same with the positions in the caller's order, and a changed order, as in `order`, behind them)
  // out_d = [force nall*3 | rows of (virial 9, energy), sums over shares of the centres]  (out_h: forces in the caller's order)
  DevBuf<double> in_d, out_d, force_op, virial_op, af2, af3, g2, g3, e_atom, vpart;
  PinBuf<double> in_h, out_h;
  PinBuf<unsigned> done_h;   // [OUT_BLOCKS flags of call_out_kernel | the stream's error word]
  unsigned calls = 0;
  // The atoms' order: made for the types of a call and kept for the calls that follow with the same ones (in MD they change
  // when atoms migrate, not every step).  order_ready: a call that has sent them is through, and tipos_h, order and type_map are
  // those of types_seen.
  std::vector<int> types_seen, tipos_h;
  int nlocal_seen = 0;
  bool order_ready = false;
  std::vector<int> tipos_up;   // what the device's tipos holds
  bool actual_type_up = false;
  // device-resident MLP (default); false: the host evaluation of staf_mlp.cpp between the kernels
  bool dev_mlp = false;
  std::vector<staf::DevMlpNet> dnets;
  DevBuf<double> raddescr, des3bsupp, der2b, der3bsupp, unit;   // nr-wide rows per owned atom; unit = (u, 1/r)
  DevBuf<double> slotf, selff;   // slot forces [nlocal, nr, 3] and centres' own forces [nlocal, 3]
  DevBuf<int> intmap2b, numtriplet, type_map, tipos, actual_type;
  DevBuf<int> order;   // [slot of every atom nall | atom of every owned slot nlocal]
  // a caller's list transposed (atom -> the centres and slots that list it): counters, which read zero between builds (tr_clear:
  // they do), counts and keys
  DevBuf<int> tr_build, tr_cnt, tr_keys;
  bool tr_clear = false;
  // host staging
  std::vector<double> af_h, gr_h, tmp2, tmp3;
  std::vector<float> af_f, gr_f;
};

static bool load_species_params(StafModel* m) {
  const int nt = m->nt, ntc = m->ntc;
  m->Ar.assign(nt, 0);
  m->Aa.assign(nt, 0);
  m->alpha2b.resize(nt);
  m->alpha3b.resize(nt);
  m->emb2b.resize(nt);
  m->emb3b.resize(nt);
  m->table.resize(nt);
  for (int k = 0; k < nt; k++) {
    const std::string pre = m->dir + "/type" + std::to_string(k) + "_";
    std::vector<double> a2, a3, e2, e3;
    int rows = 0;
    if (!read_numbers(pre + "alpha_2body.dat", a2, &rows) || rows != nt || a2.size() % nt) return false;
    if (!read_numbers(pre + "alpha_3body.dat", a3, &rows) || rows != ntc || a3.size() % (3 * ntc)) return false;
    m->Ar[k] = (int)(a2.size() / nt);
    m->Aa[k] = (int)(a3.size() / (3 * ntc));
    // the kernels take the squared embeddings (what the reference's Python layers feed its ops)
    if (!read_numbers(pre + "type_emb_2b_sq.dat", e2, nullptr)) {
      if (!read_numbers(pre + "type_emb_2b.dat", e2, nullptr)) return false;
      for (double& v : e2) v *= v;
    }
    if (!read_numbers(pre + "type_emb_3b_sq.dat", e3, nullptr)) {
      if (!read_numbers(pre + "type_emb_3b.dat", e3, nullptr)) return false;
      for (double& v : e3) v *= v;
    }
    if ((int)e2.size() != nt * m->Ar[k] || (int)e3.size() != ntc * m->Aa[k]) return false;
    struct { DevBuf<double>* d; std::vector<double>* h; } up[4] = {
        {&m->alpha2b[k], &a2}, {&m->alpha3b[k], &a3}, {&m->emb2b[k], &e2}, {&m->emb3b[k], &e3}};
    for (auto& u : up) {
      if (!u.d->reserve(u.h->size())) return false;
      if (!upload_sync(u.d->p, u.h->data(), u.h->size() * sizeof(double), m->stream)) return false;
    }
    if (staf::rows_fits<double>(m->nr, m->na, nt, m->Ar[k], m->Aa[k])) {
      const std::vector<double> t = staf::step_table_host(a3.data(), e3.data(), nt, m->Aa[k]);
      if (t[0] == 0) continue;   // (exponents beyond its rows: the staged form is faster)
      if (!m->table[k].reserve(t.size()) || !upload_sync(m->table[k].p, t.data(), t.size() * sizeof(double), m->stream)) return false;
    }
  }
  return true;
}

// staf_jmd.cfg: "key = value" lines (test/test-lammps-smoke/staf_jmd.cfg); missing file or keys -> the defaults
// the reference writes into its auto-generated cfg (libstaf/src/staf_api.cpp:139-148).
static void read_cfg(StafModel* m) {
  FILE* f = fopen((m->dir + "/staf_jmd.cfg").c_str(), "r");
  if (!f) return;
  char line[4096];
  while (fgets(line, sizeof(line), f)) {
    char key[256];
    double v;
    if (sscanf(line, " %255[A-Za-z_] = %lf", key, &v) != 2) continue;
    if (!strcmp(key, "Buffer_radial_descriptors")) m->nr = (int)v;
    else if (!strcmp(key, "Buffer_angular_descriptors")) m->na = (int)v;
    else if (!strcmp(key, "Cutoff")) m->Rc = v;
    else if (!strcmp(key, "Cutoff_Angular")) m->Ra = v;
    else if (!strcmp(key, "Hardcore_Cutoff")) m->Rs = v;
    else if (!strcmp(key, "number_of_types")) m->nt = (int)v;
  }
  fclose(f);
}

extern "C" {

void staf_options_default(StafOptions* opt) {
  if (!opt) return;
  memset(opt, 0, sizeof(*opt));
  opt->mlp_backend = STAF_MLP_ORT;
  opt->device_id = 0;
  opt->precision = 0;
}

int staf_cuda_set_device(int device_id) {
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) {
    fprintf(stderr, "staf_cuda_set_device: no GPU\n");
    return -1;
  }
  if (device_id < 0) device_id = 0;
  device_id %= ndev;
  if (hipSetDevice(device_id) != hipSuccess) return -1;
  return device_id;
}

void staf_free(StafModel* m) {
  if (!m) return;
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  if (m->mlp) staf_mlp_destroy(m->mlp);
  for (auto& n : m->dnets) staf::dev_mlp_free(&n);
  for (auto* v : {&m->alpha2b, &m->alpha3b, &m->emb2b, &m->emb3b, &m->table})
    for (auto& b : *v) b.release();
  m->in_h.release();
  m->out_h.release();
  m->done_h.release();
  for (DevBuf<double>* b : {&m->in_d, &m->out_d, &m->force_op, &m->virial_op, &m->af2, &m->af3, &m->g2, &m->g3,
                            &m->e_atom, &m->vpart, &m->raddescr, &m->des3bsupp, &m->der2b, &m->der3bsupp, &m->unit,
                            &m->slotf, &m->selff})
    b->release();
  for (DevBuf<int>* b : {&m->intmap2b, &m->numtriplet, &m->type_map, &m->tipos, &m->actual_type, &m->order, &m->tr_build, &m->tr_cnt,
                         &m->tr_keys})
    b->release();
  delete m;
}

StafModel* staf_load(const char* model_dir, const StafOptions* opt) {
  if (!model_dir) return NULL;
  StafModel* m = new StafModel();
  staf_options_default(&m->opt);
  if (opt) m->opt = *opt;
  const int dev = staf_cuda_set_device(m->opt.device_id);
  if (dev < 0) { delete m; return NULL; }
  m->opt.device_id = dev;
  m->dir = model_dir;
  m->mlp = staf_mlp_create(m->opt.mlp_backend, model_dir, m->opt.precision, dev);
  if (!m->mlp) {
    fprintf(stderr, "staf_load: staf_mlp_create failed for %s\n", model_dir);
    staf_free(m);
    return NULL;
  }
  m->nt = staf_mlp_ntypes(m->mlp);
  read_cfg(m);
  if (m->nt != staf_mlp_ntypes(m->mlp) || m->nt < 1 || m->nt > staf::NT_MAX) {
    fprintf(stderr, "staf_load: %d species in staf_jmd.cfg, %d MLP files\n", m->nt, staf_mlp_ntypes(m->mlp));
    staf_free(m);
    return NULL;
  }
  m->ntc = m->nt * (m->nt + 1) / 2;
  // The model's stream (default priority; non-blocking: no implicit ordering with the legacy default stream).
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) {
    fprintf(stderr, "staf_load: cannot create the model's stream\n");
    staf_free(m);
    return NULL;
  }
  if (!load_species_params(m)) {
    fprintf(stderr, "staf_load: cannot read the type*_alpha_*.dat / type*_type_emb_*.dat files of %s\n", model_dir);
    staf_free(m);
    return NULL;
  }
  for (int k = 0; k < m->nt; k++)
    if (staf_mlp_n_af(m->mlp, k) != m->Ar[k] + m->Aa[k]) {
      fprintf(stderr, "staf_load: species %d: MLP input width %d != %d + %d fingerprints\n", k,
              staf_mlp_n_af(m->mlp, k), m->Ar[k], m->Aa[k]);
      staf_free(m);
      return NULL;
    }
  // The MLP runs on the GPU between the fingerprint and the force kernels unless the caller asks for the host
  // evaluation (StafOptions.reserved bit 1, or STAF_MLP_HOST=1 in the environment).
  if (!(m->opt.reserved & 2) && !getenv("STAF_MLP_HOST")) {
    m->dnets.resize(m->nt);
    m->dev_mlp = true;
    for (int k = 0; k < m->nt && m->dev_mlp; k++) m->dev_mlp = staf::dev_mlp_upload(m->mlp, k, &m->dnets[k], m->stream);
    if (!m->dev_mlp) {
      for (auto& n : m->dnets) staf::dev_mlp_free(&n);
      m->dnets.clear();
      fprintf(stderr, "staf_load: MLP not representable on the device path, evaluating it on the host\n");
    }
  }
  if (staf::desc_configure<double>(m->cfg, m->Rc, m->nr, m->na, m->Rs, m->Ra) != STAF_OK) {
    staf_free(m);
    return NULL;
  }
  return m;
}

// A GPU runtime failure: -20 to the caller; with STAF_DEBUG set in the environment, where it came from on stderr.
static int gpu_failure(int line, int code) {
  static const bool verbose = getenv("STAF_DEBUG") != nullptr;
  if (verbose) fprintf(stderr, "staf_compute: GPU runtime failure at staf_api.hip:%d (code %d)\n", line, code);
  return -20;
}
// A call from its first launch on.  One that returns before its results are there waits for what it has queued, which reads
// the pinned blocks that the next call writes, and the next call sends the order of the atoms again.
struct CallInFlight {
  StafModel* m;
  bool through = false;
  ~CallInFlight() {
    if (through) return;
    (void)hipStreamSynchronize(m->stream);
    m->order_ready = false;
  }
};
#define STAF_HIP_OK(x) do { const hipError_t e_ = (x); if (e_ != hipSuccess) return gpu_failure(__LINE__, (int)e_); } while (0)

int staf_compute(StafModel* m, int nlocal, int nghost, const double* x, const double* box, const int* type,
                 const int* howmany, const int* with, int maxneigh, double* e_rank, double* f, double* virial) {
  if (!m || !m->mlp) return -1;
  const bool ext = (howmany != NULL);
  const int nall = ext ? (nlocal + nghost) : nlocal;
  if (nlocal <= 0) return -3;
  if (!x || !box || (ext && !with)) return -1;
  if (box[0] == 0.0 || box[3] == 0.0 || box[5] == 0.0) return -7;
  if (hipSetDevice(m->opt.device_id) != hipSuccess) return gpu_failure(__LINE__, 0);
  const int nt = m->nt, nr = m->nr, na = m->na;

  // ---- owned atoms species-sorted into slots [0, nlocal), ghosts keep their order behind them
  const bool same_order = m->order_ready && m->nlocal_seen == nlocal && m->types_seen.size() == (size_t)nall &&
                          (type ? memcmp(type, m->types_seen.data(), (size_t)nall * sizeof(int)) == 0
                                : std::all_of(m->types_seen.begin(), m->types_seen.end(), [](int t) { return t == 0; }));
  if (!same_order) {
    m->order_ready = false;
    m->tipos_h.assign(nt, 0);
    int known = 0;
    for (int t = 0; t < nt; t++) {
      int n = 0;
      for (int i = 0; i < nlocal; i++) n += (type ? type[i] : 0) == t;
      m->tipos_h[t] = n;
      known += n;
    }
    if (known != nlocal) {
      int i = 0;
      while (type[i] >= 0 && type[i] < nt) i++;
      fprintf(stderr, "staf_compute: unsupported type %d at atom %d\n", type[i], i);
      return -8;
    }
    for (int i = nlocal; i < nall; i++)
      if (type && (type[i] < 0 || type[i] >= nt)) return -8;
    if (type) m->types_seen.assign(type, type + nall);
    else m->types_seen.assign(nall, 0);
    m->nlocal_seen = nlocal;
  }
  const std::vector<int>& tipos = m->tipos_h;
  // ---- the call's input block, written straight into pinned memory
  const size_t L = (size_t)nlocal;
  const size_t n_in_d = (size_t)nall * 3 + 6;                                 // doubles
  // A caller's list goes to the device in the caller's order, and the descriptor kernel looks the slots up: the host
  // copies and checks rows, both in vector instructions (looking 227 000 slots up on the host and clearing the padding was
  // 110 of the 620 us of a call of 6144 owned atoms, 25 of 240 for 1500).  Rows are as long as the longest one used.
  int pitch = 0;
  const int row_max = std::min(nr, maxneigh);   // truncated like the reference (staf_api.cpp:321-323)
  if (ext)
    for (int i = 0; i < nlocal; i++) pitch = std::max(pitch, std::min(howmany[i], row_max));
  const size_t n_in_i = ext ? L + L * pitch : 0;                              // ints behind them
  const size_t n_in = (n_in_d + (n_in_i + 1) / 2 + 1) & ~(size_t)1;           // (copied by twos)
  const int nparts = std::min(64, (nlocal + 255) / 256);   // shares of the centres' virial and energy sums
  const size_t n_out = ((size_t)nall * 3 + (size_t)nparts * 10 + 1) & ~(size_t)1;
  if (!m->in_h.reserve(n_in + (same_order ? 0 : (size_t)nall)) || !m->out_h.reserve(n_out)) return -1;
  if (!m->done_h.p) {
    if (!m->done_h.reserve(OUT_BLOCKS + 1)) return -1;
    memset(m->done_h.p, 0, (OUT_BLOCKS + 1) * sizeof(unsigned));
  }
  double* pos_h = m->in_h.p;
  int* how_h = (int*)(m->in_h.p + n_in_d);
  int* with_h = how_h + L;
  if (ext) {
    for (int i = 0; i < nlocal; i++) {
      const int nn = std::max(0, std::min(howmany[i], row_max));
      how_h[i] = nn;
      const int* from = with + (size_t)i * maxneigh;
      int* to = with_h + (size_t)i * pitch;
      unsigned outside = 0;   // bit 31: an entry is negative or at least nall
      for (int k = 0; k < nn; k++) {
        const unsigned j = (unsigned)from[k];
        outside |= j | ((unsigned)(nall - 1) - j);
        to[k] = (int)j;
      }
      if (outside >> 31) {
        for (int k = 0; k < nn; k++)
          if (from[k] < 0 || from[k] >= nall) {
            fprintf(stderr, "staf_compute: neighbor index %d out of range [0,%d)\n", from[k], nall);
            break;
          }
        return -9;
      }
    }
  }
  memcpy(pos_h, x, (size_t)nall * 3 * sizeof(double));
  memcpy(pos_h + (size_t)nall * 3, box, 6 * sizeof(double));
  if (!same_order) {
    // the slots, in the caller's order within a species.  With a table of running numbers an atom waits until the last one of
    // its species has stored its own: 24576 atoms in random order, 62 / 29 / 21 / 21 us for one / two / three / four species.
    // One running number, which one and two species need, stays in a register: 18.6.  (A pass over the atoms per species
    // mispredicts: 67 to 220 us for two, 143 to 249 for three.)
    int* const slot = (int*)(m->in_h.p + n_in);
    const int* const t = m->types_seen.data();
    if (nt <= 2) {
      int zeros = 0;
      const int n0 = tipos[0];
      for (int i = 0; i < nlocal; i++) {
        const int one = t[i];
        slot[i] = one ? n0 + i - zeros : zeros;
        zeros += 1 - one;
      }
    } else {
      std::vector<int> cursor(nt, 0);
      for (int k = 1; k < nt; k++) cursor[k] = cursor[k - 1] + tipos[k - 1];
      for (int i = 0; i < nlocal; i++) slot[i] = cursor[t[i]]++;
    }
    for (int i = nlocal; i < nall; i++) slot[i] = i;
    memcpy(slot + nall, t, (size_t)nall * sizeof(int));
  }

  // ---- device buffers
  int amax2 = 0, amax3 = 0;
  for (int k = 0; k < nt; k++) { amax2 = m->Ar[k] > amax2 ? m->Ar[k] : amax2; amax3 = m->Aa[k] > amax3 ? m->Aa[k] : amax3; }
  bool ok = m->in_d.reserve(n_in) && m->out_d.reserve(n_out) && m->af2.reserve(L * amax2) &&
            m->af3.reserve(L * amax3) && m->g2.reserve(L * amax2) && m->g3.reserve(L * amax3) &&
            m->raddescr.reserve(L * nr) && m->des3bsupp.reserve(L * nr) && m->der2b.reserve(L * 3 * nr) &&
            m->der3bsupp.reserve(L * 3 * nr) && m->unit.reserve(L * 4 * nr) && m->intmap2b.reserve(L * (nr + 1)) &&
            m->numtriplet.reserve(L) && m->type_map.reserve(nall) && m->tipos.reserve(nt) && m->actual_type.reserve(nt) &&
            m->order.reserve((size_t)nall + L);
  // Slot forces of both bodies and all species from one launch, or, for neighbour buffers and parameter rows that leave no
  // room for both bodies in a workgroup's LDS (three species: 250 slots), an op per body and species.
  bool one_force_launch = m->dev_mlp;
  for (int k = 0; k < nt; k++)
    if (tipos[k] > 0) one_force_launch = one_force_launch && staf::step_forces_fits<double>(nr, nt, m->Ar[k], m->Aa[k]);
  if (m->dev_mlp) ok = ok && m->e_atom.reserve(L);
  if (one_force_launch)
    ok = ok && m->slotf.reserve(L * nr * 3) && m->selff.reserve(L * 3) && m->vpart.reserve(L * 9);
  else
    ok = ok && m->force_op.reserve((size_t)nall * 3) && m->virial_op.reserve(9);
  const int tr_cap = 4 * nr;   // centres that may list an atom
  if (ext) {   // (the number of ghosts varies from call to call: room for a quarter more)
    auto room = [](DevBuf<int>& b, size_t want) { return want <= b.n || b.reserve(want + want / 4); };
    if ((size_t)nall > m->tr_build.n) m->tr_clear = false;
    ok = ok && room(m->tr_build, nall) && room(m->tr_cnt, nall) && room(m->tr_keys, (size_t)nall * tr_cap);
  }
  if (!ok) return -1;
  hipStream_t st = m->stream;
  double* const d_pos = m->in_d.p;
  double* const d_box = d_pos + (size_t)nall * 3;
  int* const d_how = (int*)(m->in_d.p + n_in_d);
  const staf::NeighList list = {d_how, d_how + L, m->order.p + nall, m->order.p, pitch};
  double* const d_force = m->out_d.p;
  double* const d_parts = d_force + (size_t)nall * 3;
  CallInFlight in_flight{m};
  {
    const int n = (int)(n_in / 2), blocks = std::min(IN_BLOCKS, (n + IO_THREADS - 1) / IO_THREADS);
    const CallOrder order = {same_order ? nullptr : (const int*)(m->in_h.dev + n_in), m->order.p, m->type_map.p, nall, nlocal,
                             blocks};
    const int more = same_order ? 0 : std::min(IN_BLOCKS, (nall + IO_THREADS - 1) / IO_THREADS);
    hipLaunchKernelGGL(call_in_kernel, dim3(blocks + more), dim3(IO_THREADS), 0, st, (const double2*)m->in_h.dev, m->in_d.p,
                       nall * 3, n, order);
    STAF_HIP_OK(hipGetLastError());
  }
  // atoms per species: sent when they differ from what the device holds; the blocking copies read host vectors that the next
  // lines may replace
  if (m->tipos_up != tipos) {
    if (!upload_sync(m->tipos.p, tipos.data(), nt * sizeof(int), st)) return gpu_failure(__LINE__, 0);
    m->tipos_up = tipos;
  }
  if (!m->actual_type_up) {
    std::vector<int> ats(nt);
    for (int k = 0; k < nt; k++) ats[k] = k;
    if (!upload_sync(m->actual_type.p, ats.data(), nt * sizeof(int), st)) return gpu_failure(__LINE__, 0);
    m->actual_type_up = true;
  }
  // No synchronisation here: the pinned input block outlives the call's final synchronisation.
  staf::DeferStatus defer;   // conditions the kernels detect are read once, after the last kernel

  // ---- descriptors (own minimum-image list, or the caller's list with explicit images)
  staf::TransposeRef tr;
  if (ext) {
    tr.build_cnt = m->tr_build.p; tr.cnt = m->tr_cnt.p; tr.keys = m->tr_keys.p; tr.cap = tr_cap;
  } else {
    tr.symmetric = 1; tr.full = m->intmap2b.p;
  }
  auto descriptors = [&]() -> int {
    if (ext && !m->tr_clear) staf::launch_fill_zero<int>(m->tr_build.p, (int)m->tr_build.n, st);
    if (ext) m->tr_clear = false;
    const int r = staf::desc_launch<double>(m->cfg, d_pos, d_box, 1, nlocal, nall, ext ? &list : nullptr, &tr, ext ? 1 : 0,
                                            m->raddescr.p, nullptr, m->des3bsupp.p, m->intmap2b.p, nullptr, m->der2b.p,
                                            nullptr, m->der3bsupp.p, m->numtriplet.p, m->unit.p, st);
    if (ext) m->tr_clear = r == STAF_OK;
    return r == STAF_OK ? 0 : -20;
  };
  int rc = 0;
  double energy = 0.0;
  double W[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  const int n3 = nall * 3;
  const bool want_w = virial != nullptr;
  const int skip_pbc = ext ? 1 : 0;   // the caller's neighbours are explicit periodic images
  // The force op of one body of species k, whose owned atoms start at o, added to the forces; its virial in virial_op.
  auto force_op = [&](int body, int k, size_t o, const double* g2, const double* g3, bool with_virial) -> int {
    double* const w = with_virial ? m->virial_op.p : nullptr;
    const double* const px = with_virial ? d_pos : nullptr;
    const double* const bx = with_virial ? d_box : nullptr;
    staf::TransposeRef known = tr;
    known.key_shift = (int)o;
    const int r = body == 2
        ? staf::force_doublets<double>(g2, m->raddescr.p + o * nr, m->der2b.p + o * 3 * nr, m->intmap2b.p + o * (nr + 1), nr,
                                       nall, 1, m->Ar[k], m->alpha2b[k].p, m->emb2b[k].p, nt, m->tipos.p,
                                       m->actual_type.p + k, m->force_op.p, m->type_map.p, tipos[k], w, px, bx, nlocal,
                                       skip_pbc, st, &known)
        : staf::force_tripl<double>(g3, m->des3bsupp.p + o * nr, nullptr, m->der3bsupp.p + o * 3 * nr, nullptr,
                                    m->unit.p + o * 4 * nr, m->intmap2b.p + o * (nr + 1), nullptr, nr, na, nall, 1, m->Aa[k],
                                    m->emb3b[k].p, nt, m->tipos.p, m->actual_type.p + k, m->force_op.p, m->numtriplet.p + o,
                                    m->alpha3b[k].p, m->type_map.p, tipos[k], w, px, bx, nlocal, skip_pbc, st, nullptr,
                                    nullptr, nullptr, &known);
    if (r == STAF_OK) hipLaunchKernelGGL(add_into_kernel, dim3((n3 + 255) / 256), dim3(256), 0, st, d_force, m->force_op.p, n3);
    return r;
  };
  // ---- everything stays on the device, between the copying kernels five launches one behind the other (six with a cell
  // list or a caller's list): descriptors -> fingerprints -> networks -> slot forces -> collection, each over the centres
  // of all species; one wait at the end of the call.  A chain per species on a stream of its own, with a launch per body, was
  // 17 to 31 launches, replayed as a recorded graph because the host could not issue them as fast as they ran, and a
  // small system's time was the gaps between them (96 atoms: 147 us a call, 100 now; 768: 168 and 140).  Five launches
  // are issued ahead of the GPU: a recorded graph of them is no faster (106 and 143 us), and costs its recording whenever
  // the number of atoms changes.
  auto device_sequence = [&]() -> int {
    if (descriptors() != 0) return gpu_failure(__LINE__, 0);
    std::vector<staf::StepSpecies<double>> sp;
    for (int k = 0, at = 0; k < nt; at += tipos[k], k++) {
      if (tipos[k] == 0) continue;
      const size_t o = (size_t)at;
      sp.push_back({at, tipos[k], m->Ar[k], m->Aa[k], m->alpha2b[k].p, m->alpha3b[k].p, m->emb2b[k].p, m->emb3b[k].p,
                    m->af2.p + o * amax2, m->af3.p + o * amax3, m->g2.p + o * amax2, m->g3.p + o * amax3, m->table[k].p});
    }
    const int ns = (int)sp.size();
    std::vector<staf::DevMlpCall<double>> nets;
    for (int c = 0, k = 0; c < ns; c++, k++) {
      while (tipos[k] == 0) k++;
      nets.push_back({&m->dnets[k], sp[c].af2, sp[c].af3, m->e_atom.p + sp[c].first, sp[c].g2, sp[c].g3, sp[c].Ar, sp[c].Aa,
                      sp[c].Nl});
    }
    const staf::StepRows<double> rows = {m->raddescr.p, m->des3bsupp.p, m->der2b.p, m->der3bsupp.p, m->unit.p, m->intmap2b.p,
                                         m->numtriplet.p, nr, na, 1, nlocal, tr};
    double* const vpart = want_w && one_force_launch ? m->vpart.p : nullptr;
    if ((rc = staf::step_fingerprints(sp.data(), ns, rows, m->type_map.p, nt, st)) != STAF_OK) return gpu_failure(__LINE__, rc);
    if ((rc = staf::dev_mlp_eval(nets.data(), ns, st)) != STAF_OK) return gpu_failure(__LINE__, rc);
    if (one_force_launch &&
        (rc = staf::step_forces(sp.data(), ns, rows, m->type_map.p, nt, m->slotf.p, m->selff.p, vpart, st)) != STAF_OK)
      return gpu_failure(__LINE__, rc);
    const staf::StepCollect<double> out = {m->slotf.p, m->selff.p, vpart, m->e_atom.p, one_force_launch ? d_force : nullptr,
                                           d_parts, nullptr, nullptr, nparts};
    if ((rc = staf::step_collect(sp.data(), ns, rows, nall, out, st)) != STAF_OK)
      return gpu_failure(__LINE__, rc);
    if (one_force_launch) return 0;
    // the virials go to the first share's row, which holds an energy sum and zeros
    staf::launch_fill_zero<double>(d_force, n3, st);
    for (int c = 0, k = 0; c < ns; c++, k++) {
      while (tipos[k] == 0) k++;
      const size_t o = (size_t)sp[c].first;
      for (int body = 2; body <= 3; body++) {
        if ((rc = force_op(body, k, o, sp[c].g2, sp[c].g3, want_w)) != STAF_OK) return gpu_failure(__LINE__, rc);
        if (want_w) hipLaunchKernelGGL(add_into_kernel, dim3(1), dim3(256), 0, st, d_parts, m->virial_op.p, 9);
      }
    }
    return hipGetLastError() == hipSuccess ? 0 : gpu_failure(__LINE__, 0);
  };
  if (m->dev_mlp) {
    if (device_sequence() != 0) return -20;
  } else {
    if (descriptors() != 0) return gpu_failure(__LINE__, 0);
    // ---- fingerprints of every species, packed rows [Ar+Aa] for the MLP
    size_t total = 0;
    for (int k = 0; k < nt; k++) total += (size_t)tipos[k] * (m->Ar[k] + m->Aa[k]);
    m->af_h.resize(total);
    m->gr_h.assign(total, 0.0);
    size_t off = 0;
    int shift = 0;
    for (int k = 0; k < nt; shift += tipos[k], k++) {
      const int Nl = tipos[k], Ar = m->Ar[k], Aa = m->Aa[k];
      if (Nl == 0) continue;
      const size_t o = (size_t)shift;
      rc = staf_op_radial_afs_f64(m->raddescr.p + o * nr, nr, m->alpha2b[k].p, Ar, m->af2.p, 1, Nl,
                                  m->intmap2b.p + o * (nr + 1), m->emb2b[k].p, m->type_map.p, nt, nlocal, st);
      if (rc == STAF_OK)
        rc = staf::angular_afs<double>(m->des3bsupp.p + o * nr, nullptr, m->unit.p + o * 4 * nr, nr, na, m->af3.p, 1, Nl,
                                       nullptr, m->intmap2b.p + o * (nr + 1), m->alpha3b[k].p, Aa, m->emb3b[k].p,
                                       m->type_map.p, m->numtriplet.p + o, nt, nlocal, st);
      if (rc != STAF_OK) return gpu_failure(__LINE__, rc);
      m->tmp2.resize((size_t)Nl * Ar);
      m->tmp3.resize((size_t)Nl * Aa);
      STAF_HIP_OK(hipMemcpyAsync(m->tmp2.data(), m->af2.p, m->tmp2.size() * sizeof(double), hipMemcpyDeviceToHost, st));
      STAF_HIP_OK(hipMemcpyAsync(m->tmp3.data(), m->af3.p, m->tmp3.size() * sizeof(double), hipMemcpyDeviceToHost, st));
      STAF_HIP_OK(hipStreamSynchronize(st));
      for (int a = 0; a < Nl; a++) {
        double* row = &m->af_h[off + (size_t)a * (Ar + Aa)];
        memcpy(row, &m->tmp2[(size_t)a * Ar], Ar * sizeof(double));
        memcpy(row + Ar, &m->tmp3[(size_t)a * Aa], Aa * sizeof(double));
      }
      off += (size_t)Nl * (Ar + Aa);
    }

    // ---- MLP on the host (libstaf/vendor/jmd/nn_nn_mlp.cu:657-768): float32 nets see float32 fingerprints
    std::vector<int> n_af(nt);
    for (int k = 0; k < nt; k++) n_af[k] = m->Ar[k] + m->Aa[k];
    StafMlpEval ev;
    memset(&ev, 0, sizeof(ev));
    ev.n_type = nt;
    ev.n_atoms = tipos.data();
    ev.n_af = n_af.data();
    energy = 0.0;
    if (staf_mlp_precision(m->mlp) == 0) {
      m->af_f.resize(total);
      m->gr_f.assign(total, 0.f);
      for (size_t i = 0; i < total; i++) m->af_f[i] = (float)m->af_h[i];
      float e_f = 0.f;
      ev.af_f32 = m->af_f.data();
      ev.energy_f32 = &e_f;
      ev.dE_daf_f32 = m->gr_f.data();
      if (staf_mlp_eval(m->mlp, &ev) != 0) return gpu_failure(__LINE__, 0);
      energy = (double)e_f;
      for (size_t i = 0; i < total; i++) m->gr_h[i] = (double)m->gr_f[i];
    } else {
      ev.af_f64 = m->af_h.data();
      ev.energy_f64 = &energy;
      ev.dE_daf_f64 = m->gr_h.data();
      if (staf_mlp_eval(m->mlp, &ev) != 0) return gpu_failure(__LINE__, 0);
    }
    if (!isfinite(energy))
      fprintf(stderr, "staf_compute: non-finite energy=%g nlocal=%d nghost=%d\n", energy, nlocal, nghost);

    // ---- forces: 2-body + 3-body of every centre species, with the virial
    staf::launch_fill_zero<double>(d_force, nall * 3, st);
    double Wk[9];
    off = 0;
    shift = 0;
    for (int k = 0; k < nt; shift += tipos[k], k++) {
      const int Nl = tipos[k], Ar = m->Ar[k], Aa = m->Aa[k];
      if (Nl == 0) continue;
      const size_t o = (size_t)shift;
      m->tmp2.resize((size_t)Nl * Ar);
      m->tmp3.resize((size_t)Nl * Aa);
      for (int a = 0; a < Nl; a++) {
        const double* row = &m->gr_h[off + (size_t)a * (Ar + Aa)];
        memcpy(&m->tmp2[(size_t)a * Ar], row, Ar * sizeof(double));
        memcpy(&m->tmp3[(size_t)a * Aa], row + Ar, Aa * sizeof(double));
      }
      off += (size_t)Nl * (Ar + Aa);
      STAF_HIP_OK(hipMemcpyAsync(m->g2.p, m->tmp2.data(), m->tmp2.size() * sizeof(double), hipMemcpyHostToDevice, st));
      STAF_HIP_OK(hipMemcpyAsync(m->g3.p, m->tmp3.data(), m->tmp3.size() * sizeof(double), hipMemcpyHostToDevice, st));
      STAF_HIP_OK(hipStreamSynchronize(st));
      for (int body = 2; body <= 3; body++) {
        if ((rc = force_op(body, k, o, m->g2.p, m->g3.p, true)) != STAF_OK) return gpu_failure(__LINE__, rc);
        STAF_HIP_OK(hipMemcpyAsync(Wk, m->virial_op.p, 9 * sizeof(double), hipMemcpyDeviceToHost, st));
        STAF_HIP_OK(hipStreamSynchronize(st));
        for (int c = 0; c < 9; c++) W[c] += Wk[c];
      }
    }
  }
  // forces, on the device path the virial and energy sums behind them, and the stream's error word
  staf::DeviceState* const state = staf::device_state(st);
  if (!state) return gpu_failure(__LINE__, 0);
  const unsigned call = ++m->calls ? m->calls : ++m->calls;   // (never what the flags start with)
  unsigned* const flags = m->done_h.p;
  int* const status_h = (int*)(m->done_h.p + OUT_BLOCKS);
  int out_blocks = 0;
  {
    const int n = (int)(((m->dev_mlp ? n_out : (size_t)n3) + 1) / 2);
    out_blocks = std::min(OUT_BLOCKS, (n + IO_THREADS - 1) / IO_THREADS);
    hipLaunchKernelGGL(call_out_kernel, dim3(out_blocks), dim3(IO_THREADS), 0, st, m->out_d.p, (double2*)m->out_h.dev,
                       m->order.p, n3, n, staf::status_word(state, st), (int*)(m->done_h.dev + OUT_BLOCKS), m->done_h.dev, call);
    STAF_HIP_OK(hipGetLastError());
  }
  const double* force_h = m->out_h.p;
  // the call's synchronisation: results are on the host, and so is what the kernels reported.  The host watches the flags for
  // the whole call, as a stream synchronisation does unless the program has asked for blocking waits on the device: then the
  // call sleeps in one (24576 atoms: 0.40 ms of host time in a call of 1.24 ms).  The stream is asked now and then, and ends
  // the wait where a kernel failed.
  unsigned device_flags = 0;
  STAF_HIP_OK(hipGetDeviceFlags(&device_flags));
  if ((device_flags & hipDeviceScheduleMask) == hipDeviceScheduleBlockingSync) STAF_HIP_OK(hipStreamSynchronize(st));
  for (unsigned round = 1; ; round++) {
    int b = 0;
    while (b < out_blocks && __atomic_load_n(&flags[b], __ATOMIC_ACQUIRE) == call) b++;
    if (b == out_blocks) break;
    if (round % 8192 == 0) {
      const hipError_t e = hipStreamQuery(st);
      if (e == hipErrorNotReady) continue;
      if (e != hipSuccess) return gpu_failure(__LINE__, (int)e);
      for (b = 0; b < out_blocks; b++)
        if (__atomic_load_n(&flags[b], __ATOMIC_ACQUIRE) != call) return gpu_failure(__LINE__, b);
      break;
    }
    __builtin_ia32_pause();
  }
  in_flight.through = m->order_ready = true;
  // What the results' kernel has read is what the call found; the conditions of other streams are left to them.
  rc = *status_h ? staf::take_status(state, st, *status_h) : STAF_OK;
  if (rc == STAF_E_RADIAL_OVERFLOW) return -10;
  if (rc == STAF_E_SCATTER_OVERFLOW) return -11;
  if (rc != STAF_OK) return gpu_failure(__LINE__, rc);
  if (m->dev_mlp) {
    const double* part = m->out_h.p + (size_t)n3;
    for (int p = 0; p < nparts; p++, part += 10) {   // (a fixed order)
      for (int c = 0; c < 9; c++) W[c] += part[c];
      energy += part[9];
    }
    energy *= 0.5;
    if (!isfinite(energy))
      fprintf(stderr, "staf_compute: non-finite energy=%g nlocal=%d nghost=%d\n", energy, nlocal, nghost);
  }

  if (e_rank) *e_rank = energy;
  if (f) memcpy(f, force_h, (size_t)n3 * sizeof(double));
  if (virial) {
    virial[0] = W[0];
    virial[1] = W[4];
    virial[2] = W[8];
    virial[3] = virial[4] = virial[5] = 0.0;   // the reference fills the diagonal only (staf_api.cpp:398-403)
    if (m->opt.reserved & 1) {
      virial[3] = 0.5 * (W[1] + W[3]);
      virial[4] = 0.5 * (W[2] + W[6]);
      virial[5] = 0.5 * (W[5] + W[7]);
    }
  }
  return 0;
}

}  // extern "C"
