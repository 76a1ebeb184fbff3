// The host side of staf_compute (csrc/staf_api.hip, csrc/staf_runtime.hip) over a runtime without a GPU: memory is the
// host's, a stream is a queue whose entries run when the host waits for it or asks it, and the stages between the copying
// kernels are replaced by one that writes a force per slot.  Conditions that a GPU gives only now and then -- a stage that
// cannot be launched while the call's first kernel has not run yet, another thread's poll between two lines -- are set here.
//
//   fake_gpu MODEL_DIR SCENARIO   prints "ok" or what is wrong
#include "../../alphanesgpu_amd/csrc/staf_common.hpp"
#include "../../alphanesgpu_amd/csrc/staf_mlp_dev.hpp"
#include "../../include/staf.h"

#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

#include <deque>
#include <functional>
#include <map>
#include <string>
#include <vector>

namespace {

std::deque<std::function<void()>> queue_;
std::map<const void*, std::string>& names() {   // (filled before this file's own objects are there)
  static std::map<const void*, std::string> n;
  return n;
}
std::function<void()> after_results_;   // runs between the results' kernel and what the host does next
int fail_descriptors_ = 0, raise_ = 0, queries_ = 0, waits_ = 0;
unsigned flags_ = hipDeviceScheduleAuto;

void run_queue() {
  while (!queue_.empty()) {
    auto f = queue_.front();
    queue_.pop_front();
    f();
  }
}
[[noreturn]] void wrong(const char* what) {
  printf("%s\n", what);
  fflush(stdout);
  _exit(1);
}

struct CallOrder {   // (as the copying kernel takes it)
  const int* new_order;
  int *order_d, *type_map;
  int nall, nlocal, blocks;
};
template <typename T>
T arg(void** args, int i) { return *(T*)args[i]; }

}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) { static void* module; return &module; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names()[host] = name;
}
static thread_local struct { dim3 grid, block; size_t lds; hipStream_t stream; } launch_;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) { launch_ = {g, b, lds, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  *g = launch_.grid; *b = launch_.block; *lds = launch_.lds; *s = launch_.stream;
  return hipSuccess;
}

hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t) {
  const std::string& name = names()[f];
  auto is = [&](const char* part) { return name.find(part) != std::string::npos; };
  if (is("call_in_kernel")) {
    const double* const host = arg<const double*>(args, 0);
    double* const dev = arg<double*>(args, 1);
    const int n3 = arg<int>(args, 2), n = arg<int>(args, 3);
    const CallOrder O = arg<CallOrder>(args, 4);
    queue_.push_back([=] {
      auto slot = [&](int i) {
        const int s = (O.new_order ? O.new_order : O.order_d)[i];
        if (s < 0 || s >= O.nall) wrong("a slot out of range");
        return s;
      };
      for (int e = 0; e < 2 * n; e++) memcpy(&dev[e < n3 ? 3 * slot(e / 3) + e % 3 : e], &host[e], sizeof(double));
      for (int i = 0; O.new_order && i < O.nall; i++) {
        O.type_map[slot(i)] = O.new_order[O.nall + i];
        if (i < O.nlocal) O.order_d[O.nall + slot(i)] = i;
      }
      if (O.new_order) memcpy(O.order_d, O.new_order, O.nall * sizeof(int));
    });
  } else if (is("call_out_kernel")) {
    const double* const dev = arg<const double*>(args, 0);
    double* const host = arg<double*>(args, 1);
    const int* const slot_of = arg<const int*>(args, 2);
    const int n3 = arg<int>(args, 3), n = arg<int>(args, 4), blocks = (int)grid.x;
    const int* const status = arg<const int*>(args, 5);
    int* const status_h = arg<int*>(args, 6);
    unsigned* const flags = arg<unsigned*>(args, 7);
    const unsigned call = arg<unsigned>(args, 8);
    queue_.push_back([=] {
      for (int e = 0; e < 2 * n; e++) host[e] = dev[e < n3 ? 3 * slot_of[e / 3] + e % 3 : e];
      status_h[0] = status[0];
      for (int b = 0; b < blocks; b++) flags[b] = call;
      if (after_results_) after_results_();
    });
  } else if (is("fill_zero_kernel")) {
    char* const p = arg<char*>(args, 0);
    const size_t bytes = arg<int>(args, 1) * (is("fill_zero_kernelIi") ? sizeof(int) : sizeof(double));
    queue_.push_back([=] { memset(p, 0, bytes); });
  } else if (is("status_clear_kernel")) {
    int* const word = arg<int*>(args, 0);
    struct Seen { int bits[staf::STATUS_WORDS]; };
    const Seen seen = arg<Seen>(args, 1);
    const int nw = arg<int>(args, 2);
    queue_.push_back([=] { for (int w = 0; w < nw; w++) word[w] &= ~seen.bits[w]; });
  } else {
    wrong(("unexpected kernel " + name).c_str());
  }
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceFlags(unsigned* f) { *f = flags_; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
// (blocks are filled, so that nothing is right by the zeroes of fresh memory; freeing waits, as the runtime's does)
hipError_t hipMalloc(void** p, size_t n) { *p = malloc(n); memset(*p, 0x7f, n); return hipSuccess; }
hipError_t hipFree(void* p) { run_queue(); free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipHostGetDevicePointer(void** d, void* p, unsigned) { *d = p; return hipSuccess; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
  queue_.push_back([=] { memcpy(dst, src, n); });
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) { memset(p, v, n); return hipSuccess; }
hipError_t hipDeviceSynchronize() { run_queue(); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { waits_++; run_queue(); return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { queries_++; run_queue(); return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { *s = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t*) { return hipErrorUnknown; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float*, hipEvent_t, hipEvent_t) { return hipErrorUnknown; }

int staf_op_radial_afs_f64(const double*, int, const double*, int, double*, int, int, const int*, const double*, const int*,
                           int, int, void*) { return STAF_E_HIP; }

}  // extern "C"

namespace staf {

static const double* positions_;   // what the descriptor stage of the call was given, in slots

template <> int desc_configure<double>(DescConfig<double>& c, double, int nr, int na, double, double) {
  c.ready = true; c.nr = nr; c.na = na;
  return STAF_OK;
}
template <> int desc_launch<double>(const DescConfig<double>&, const double* pos, const double*, int, int, int,
                                    const NeighList*, const TransposeRef*, int, double*, double*, double*, int*, int*, double*,
                                    double*, double*, int*, double*, hipStream_t stream) {
  if (fail_descriptors_) return STAF_E_HIP;
  positions_ = pos;
  if (const int bit = raise_) {
    int* const word = status_word(device_state(stream), stream);
    queue_.push_back([=] { *word |= bit; });
  }
  return STAF_OK;
}
bool dev_mlp_upload(const StafMlp*, int, DevMlpNet*, hipStream_t) { return true; }
void dev_mlp_free(DevMlpNet*) {}
template <> int dev_mlp_eval<double>(const DevMlpCall<double>*, int, hipStream_t) { return STAF_OK; }
template <> int step_fingerprints<double>(const StepSpecies<double>*, int, const StepRows<double>&, const int*, int,
                                          hipStream_t) { return STAF_OK; }
template <> bool step_forces_fits<double>(int, int, int, int) { return true; }
static const int* species_;
template <> int step_forces<double>(const StepSpecies<double>*, int, const StepRows<double>&, const int* type_map, int, double*,
                                    double*, double*, hipStream_t) {
  species_ = type_map;
  return STAF_OK;
}
// the force on a slot: its position times one more than its species
template <> int step_collect<double>(const StepSpecies<double>*, int, const StepRows<double>&, int nall,
                                     const StepCollect<double>& out, hipStream_t) {
  const double* const pos = positions_;
  const int* const species = species_;
  queue_.push_back([=] {
    for (int i = 0; i < 3 * nall; i++) out.force[i] = pos[i] * (1 + species[i / 3]);
    for (int i = 0; i < 10 * out.nparts; i++) out.parts[i] = 0;
  });
  return STAF_OK;
}
template <> int force_doublets<double>(const double*, const double*, const double*, const int*, int, int, int, int,
                                       const double*, const double*, int, const int*, const int*, double*, const int*, int,
                                       double*, const double*, const double*, int, int, void*, const TransposeRef*) {
  return STAF_E_HIP;
}
template <> int force_tripl<double>(const double*, const double*, const double*, const double*, const double*, const double*,
                                    const int*, const int*, int, int, int, int, int, const double*, int, const int*,
                                    const int*, double*, const int*, const double*, const int*, int, double*, const double*,
                                    const double*, int, int, void*, double*, double*, const Force2In<double>*,
                                    const TransposeRef*, int) { return STAF_E_HIP; }
template <> int angular_afs<double>(const double*, const double*, const double*, int, int, double*, int, int, const int*,
                                    const int*, const double*, int, const double*, const int*, const int*, int, int, void*,
                                    int, int) { return STAF_E_HIP; }

}  // namespace staf

// ------------------------------------------------------------------------------------------------------ scenarios

static const double BOX[6] = {1000, 0, 0, 1000, 0, 1000};

struct Call {
  int n, row;   // atoms, neighbours of each in a caller's list, or -1: no list
  std::vector<int> types;
  std::vector<double> x, f;
  // (as many atoms of a species whatever the order: other counts are sent with a wait of their own)
  Call(int n_, int row_, int order) : n(n_), row(row_), types(n_), x(3 * n_), f(3 * n_, -1.0) {
    for (int i = 0; i < n; i++) types[i] = (i + order) % 3 == 0;
    for (int i = 0; i < 3 * n; i++) x[i] = i + 0.25 * order;
  }
  int run(StafModel* m) {
    std::vector<int> how(n, row), with((size_t)n * std::max(row, 1));
    for (size_t i = 0; i < with.size(); i++) with[i] = (int)(i * 7 % n);
    double e;
    return staf_compute(m, n, 0, x.data(), BOX, types.data(), row < 0 ? nullptr : how.data(), row < 0 ? nullptr : with.data(),
                        std::max(row, 0), &e, f.data(), nullptr);
  }
  bool right() const {
    for (int i = 0; i < 3 * n; i++)
      if (f[i] != x[i] * (1 + types[i / 3])) return false;
    return true;
  }
};

int main(int argc, char** argv) {
  if (argc != 3) return 2;
  StafOptions opt;
  staf_options_default(&opt);
  opt.mlp_backend = STAF_MLP_NATIVE;
  opt.precision = 1;
  StafModel* m = staf_load(argv[1], &opt);
  if (!m) wrong("no model");
  const std::string scenario = argv[2];
  auto expect = [&](bool ok, const char* what) { if (!ok) wrong(what); };
  // (blocks as large as any call of a scenario needs, so that none is replaced on the way)
  Call first(300, 40, 0);
  expect(first.run(m) == 0 && first.right(), "first call");

  if (scenario == "failed_launch") {
    // a stage of a call with another order of the atoms cannot be launched
    Call failed(300, 2, 1);
    fail_descriptors_ = 1;
    expect(failed.run(m) == -20, "code of the failed call");
    fail_descriptors_ = 0;
    const bool drained = queue_.empty();
    // the same order again: the rows of this list are longer than the failed call's block
    Call next(300, 40, 1);
    expect(next.run(m) == 0, "call after the failed one");
    expect(next.right(), "forces after the failed call");
    expect(drained, "work in flight behind a failed call");
  } else if (scenario == "other_poll") {
    // another thread polls, and clears every word, between the results and what this call does next
    staf::DeviceState* const st = staf::device_state(nullptr);
    raise_ = 1;
    after_results_ = [=] { for (int w = 0; w < staf::STATUS_WORDS; w++) st->status_d[w] = 0; };
    Call c(300, -1, 1);
    expect(c.run(m) == -10, "a condition of the call that another poll has cleared");
    after_results_ = nullptr;
    expect(c.run(m) == -10, "a condition of the call");
    raise_ = 0;
    expect(c.run(m) == 0 && c.right(), "the call after it");
  } else if (scenario == "other_stream") {
    // a condition of another stream is pending
    staf::DeviceState* const st = staf::device_state(nullptr);
    int* const word = staf::status_word(st, (hipStream_t)&queue_);
    *word = 2;
    Call c(300, -1, 1);
    expect(c.run(m) == 0 && c.right(), "a call beside another stream's condition");
    raise_ = 1;
    expect(c.run(m) == -10, "a condition of the call");
    raise_ = 0;
    expect(*word == 2, "another stream's condition is gone");
    expect(staf_ops_poll_status(nullptr) == STAF_E_SCATTER_OVERFLOW, "the poll for it");
  } else if (scenario == "blocking_wait") {
    queries_ = waits_ = 0;
    Call c(300, -1, 0);
    expect(c.run(m) == 0 && c.right() && queries_ > 0, "a call that watches the flags");
    queries_ = waits_ = 0;
    flags_ = hipDeviceScheduleBlockingSync | hipDeviceMapHost;
    expect(c.run(m) == 0 && c.right(), "a call that blocks");
    expect(queries_ == 0 && waits_ > 0, "the stream is not waited for");
  } else {
    return 2;
  }
  staf_free(m);
  printf("ok\n");
  return 0;
}
