// Transpose of the neighbour map: for every receiving atom the (centre, slot) pairs that list it.
//
// The reference scatters pair forces with floating-point atomicAdd (STAF/src/force/rad/reforce.cu.cc:112-131,
// STAF/src/force/ang/reforce.cu.cc:206-231).  Here the force on an atom is gathered by the atom itself from the
// slots that point at it, which needs intmap2b transposed: receiver -> sorted list of keys (centre, slot).  A caller's
// list of the MD entry is transposed by the descriptor launch that reads it (pushes from its workgroups, one sort
// launch) into a block of the model.  A force op that is handed a map that is not remembered builds a transpose of its own
// first (push + sort launches).
//
// Building uses integer atomics only (the arrival order they leave is removed by the sort); every list ends up in
// ascending (centre, slot) order, so sums taken over it have a fixed order.
//
// None of this is needed for the maps the library's own neighbour search writes: those are symmetric, the centres
// that list an atom are the atom's own neighbours, and the slot is found by looking the atom up in the centre's row
// (slots_of below).  Sums then run in the order of the atom's own (distance-sorted) row.  The descriptor op remembers by its
// address that a tensor holds such a map, and every force op that is handed a view of that tensor finds it.
#pragma once
#include "staf_common.hpp"

namespace staf {

constexpr int KEY_SLOT_BITS = 10;   // key = centre << 10 | slot; slots < 1024 (the descriptor op's limit on nr)
constexpr int TR_BLOCK = 256;
constexpr int TR_WAVES = TR_BLOCK / WAVE;

__device__ inline int key_make(int centre, int slot) { return (centre << KEY_SLOT_BITS) | slot; }
__device__ inline int key_centre(int key) { return key >> KEY_SLOT_BITS; }
__device__ inline int key_slot(int key) { return key & ((1 << KEY_SLOT_BITS) - 1); }

// Registers slot `slot` of centre `centre` with receiving atom `recv` (index into [nf * Nrecv]).
__device__ inline void transpose_push(int* build_cnt, int* keys, int cap, size_t recv, int centre, int slot,
                                      int* status) {
  const int pos = atomicAdd(&build_cnt[recv], 1);
  if (pos < cap) keys[recv * cap + pos] = key_make(centre, slot);
  else atomicOr(status, 2);
}

// Checksum of a row of a map, order-free: the sum over its slots of row_hash(neighbour, slot), plus the count.  The
// descriptor op stores it for every row of a map it writes; a kernel that takes an atom's own row as the list of
// centres that list the atom recomputes it, so that other content at a remembered address (a caller's list copied
// there, a tensor of another call at a recycled address) is reported instead of read as symmetric.
__device__ inline unsigned row_hash(int neighbour, int slot) {
  return ((unsigned)neighbour + 1u) * (2u * (unsigned)slot + 1u) * 0x9E3779B1u;
}
// `partial`: the lane's share of the sum over the row's slots below `cnt`; the last lane holds the sum and reports.
__device__ inline void row_check(const TransposeRef& tr, size_t row, int cnt, unsigned partial, int lane, int* status) {
  if (!tr.rowsum) return;
  const unsigned h = wave_sum_to_last(partial) + (unsigned)cnt;
  if (lane == WAVE - 1 && h != tr.rowsum[row]) atomicOr(status, 4);
}

// Slots of atom `a` in the rows of its neighbours, all lanes of the wave calling: a lane with i >= 0 asks for the slot
// of `a` in the row of centre i of frame b of the symmetric map `full` [nf, N, nr+1] and gets it, or -1 (the map is
// not symmetric after all: reported by the caller); lanes with i < 0 get -1.
// The rows asked for are read by the wave together, 16 lanes to a row in 16-byte pieces, four rows a step and four
// steps in flight.  (A lane reading the whole row of its own neighbour asks the memory pipeline for 64 different lines
// with every instruction: force_total_kernel in double precision took 72.5 us for 24576 atoms and 18.2 us for 6144, with
// rows read together it takes 48.3 and 14.3; what is left is the traffic, each row and slot force from the L2 of eight
// XCDs.  For 96 atoms, where nothing but the chain of dependent reads counts, 7.5 and 7.9.)
struct __attribute__((packed, aligned(4))) Int4U { int x, y, z, w; };
struct SlotSearch {   // in LDS, one per wave
  int row[WAVE], lane[WAVE], found[WAVE];
};
__device__ inline int slots_of(const int* __restrict__ full, int b, int N, int nr, int i, int a, SlotSearch& w) {
  const int lane = lane_id();
  const unsigned long long asked = __ballot(i >= 0);
  const int n = __popcll(asked);
  w.found[lane] = -1;
  if (i >= 0) {
    const int at = __popcll(asked & ((1ull << lane) - 1ull));
    w.row[at] = i;
    w.lane[at] = lane;
  }
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
  const int* rows = full + (size_t)b * N * (nr + 1);
  const int part = lane >> 4, piece = lane & 15;
  for (int t0 = 0; t0 < n; t0 += 16) {
    const int* r[4];
    int who[4], cnt[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {   // (past the last row the last one is read again)
      const int t = t0 + 4 * u + part < n ? t0 + 4 * u + part : n - 1;
      r[u] = rows + (size_t)w.row[t] * (nr + 1);
      who[u] = w.lane[t];
      cnt[u] = r[u][0];   // (padded entries hold 0, which is also an atom: only slots below the count are neighbours)
    }
    if (nr >= 4) {
      for (int c0 = 0; c0 < nr; c0 += 64) {
        const int e = c0 + 4 * piece < nr - 4 ? c0 + 4 * piece : nr - 4;   // the row's end is read by several lanes
        Int4U v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = *(const Int4U*)(r[u] + 1 + e);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int top = cnt[u] < nr ? cnt[u] : nr;
          int s = -1;
          s = (v[u].x == a && e < top) ? e : s;
          s = (v[u].y == a && e + 1 < top) ? e + 1 : s;
          s = (v[u].z == a && e + 2 < top) ? e + 2 : s;
          s = (v[u].w == a && e + 3 < top) ? e + 3 : s;
          if (s >= 0) w.found[who[u]] = s;
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (piece < nr && piece < cnt[u] && r[u][1 + piece] == a) w.found[who[u]] = piece;
    }
  }
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
  const int s = w.found[lane];
  __builtin_amdgcn_wave_barrier();
  return s;
}

// One thread per (frame, centre, slot) of a map [nf, ld (Nl used), nr+1]: the push pass of a transpose built by a
// force op itself.  Centres are numbered from 0 at the first row of the view.
static __global__ __launch_bounds__(TR_BLOCK) void transpose_push_kernel(const int* __restrict__ im2, int* build_cnt,
                                                                         int* keys, int cap, int* status, int nf,
                                                                         int Nrecv, int Nl, int ld, int nr) {
  const int t = blockIdx.x * TR_BLOCK + threadIdx.x;
  const int total = nf * Nl * nr;
  if (t >= total) return;
  const int s = t % nr;
  const int atom = t / nr;
  const int b = atom / Nl, p = atom - b * Nl;
  const int* im = im2 + ((size_t)b * ld + p) * (nr + 1);
  int cnt = im[0];
  if (cnt > nr) cnt = nr;
  if (s >= cnt) return;
  const int nj = im[1 + s];
  if (nj < 0 || nj >= Nrecv) { atomicOr(status, 2); return; }
  transpose_push(build_cnt, keys, cap, (size_t)b * Nrecv + nj, p, s, status);
}

// One wave per receiving atom: its keys are put in ascending order in place, the final count goes to cnt and the
// build counter back to 0 for the next build.
static __global__ __launch_bounds__(TR_BLOCK) void transpose_sort_kernel(int* build_cnt, int* __restrict__ cnt,
                                                                         int* keys, int cap, int n_recv) {
  extern __shared__ __align__(16) unsigned char smem[];
  int* w_key = (int*)smem;   // [TR_WAVES][cap]
  const int wave = threadIdx.x / WAVE, lane = lane_id();
  int* key = w_key + wave * cap;
  const int recv = blockIdx.x * TR_WAVES + wave;
  if (recv >= n_recv) return;
  int L = uniform(build_cnt[recv]);
  if (L > cap) L = cap;
  int* mine = keys + (size_t)recv * cap;
  for (int e = lane; e < L; e += WAVE) key[e] = mine[e];
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
  if (lane == 0) {
    cnt[recv] = L;
    if (L > 0) build_cnt[recv] = 0;
  }
  for (int e = lane; e < L; e += WAVE) {
    const int ke = key[e];
    int rank = 0;
    for (int o = 0; o < L; o++) rank += (key[o] < ke) ? 1 : 0;   // keys of one receiver are distinct
    mine[rank] = ke;
  }
}

inline void launch_transpose_sort(const TransposeRef& t, int n_recv, hipStream_t stream) {
  hipLaunchKernelGGL(transpose_sort_kernel, dim3((n_recv + TR_WAVES - 1) / TR_WAVES), dim3(TR_BLOCK),
                     (size_t)TR_WAVES * t.cap * sizeof(int), stream, t.build_cnt, t.cnt, t.keys, t.cap, n_recv);
}

}  // namespace staf
