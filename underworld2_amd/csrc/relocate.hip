// Particle relocation after advection: new owners plus per-cell particle tables edited
// exactly as Swarm_UpdateAllParticleOwners does (LU/StgDomain/Swarm/src/SwarmClass.c:
// 947-1030): particles are visited in index order; a particle that changed cell is removed
// from its old table by swap-with-last (Swarm_RemoveParticleFromCell) and appended to its
// new one (Swarm_AddParticleToCell).  The edits that touch one cell are exactly that
// cell's removals and additions in particle-index order, so every cell replays its own
// events independently.  The removals are the table's own entries whose owner changed; the
// additions are gathered per cell with a counting pass (per-cell atomics whose order does not
// matter: the replay takes a cell's additions by increasing index).  A cell that gains more
// particles than that search is good for sends the call to a stable radix sort of the movers.
#include <algorithm>
#include <utility>

#include <hipcub/hipcub.hpp>

#include "uwg_geom.h"
#include "uwg_internal.h"

namespace uwg {

// additions per cell up to which the replay finds them in index order by scanning; above it
// the movers are sorted (one step of a 3D swarm at the CFL limit adds about a third of a
// cell's particles; the scan costs na^2 / 8 reads per cell, the sort 5-6 launches per step)
constexpr int kMaxScanAdd = 48;

struct RelocWork {
  long P, E;
  int* new_owner;
  int* rank;       // position of a mover among its new cell's additions (unordered)
  int* cnt;        // [2][E+2]: additions, removals per cell
  unsigned long long* off;  // [E+1]: start of a cell's new table (high word) and additions (low)
  int* add;        // movers grouped by new cell
  int* tmp;        // lists too long for LDS, [2 P]
  int* ptr;        // [E+1] the new tables, exchanged with the swarm's
  int* pid;        // [cap]
  int* stat;       // outside count, large-cell flag, caller's two counters
  // movers sorted by new cell (allocated on first use)
  int *ids = nullptr, *mv = nullptr, *key = nullptr, *key_s = nullptr;
  uint8_t* moved = nullptr;
  void* cub_tmp = nullptr;
  size_t cub_bytes = 0;
};

static inline unsigned nb(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

struct CellGrid {
  int res[3];
  double lo[3], hi[3];
  long E;
};

// Lanes of a wave that hold the same key as this one: *leader its lowest lane, *rank this lane's
// position among them, returned their number.  Neighbouring particles share cells, so a wave
// meets few distinct keys, and one atomic per key (all leaders at once) replaces up to 64
// serialised ones on one address: 0.74 ms -> 0.05 ms for the counts of 5.2 M particles.
__device__ __forceinline__ int same_key(bool on, int key, int* leader, int* rank) {
  const int lane = threadIdx.x & 63;
  const unsigned long long below = (1ull << lane) - 1ull;
  unsigned long long todo = __ballot(on);
  int n = 0;
  while (todo) {
    const int first = __ffsll((long long)todo) - 1;
    const int k = __builtin_amdgcn_readlane(key, first);
    const unsigned long long same = __ballot(on && key == k);
    if (on && key == k) {
      *leader = first;
      *rank = __popcll(same & below);
      n = __popcll(same);
    }
    todo &= ~same;
  }
  return n;
}

// New owner of every particle, additions and removals per cell, and each mover's position among
// its new cell's additions.  HBM-bound: coordinates and owner in, owner and rank out.
template <int DIM>
__global__ __launch_bounds__(256) void k_moves(CellGrid g, long P, const double* __restrict__ coords,
                                               const int* __restrict__ owner, int* __restrict__ new_owner,
                                               int* __restrict__ rank, int* __restrict__ cnt_a,
                                               int* __restrict__ cnt_r, int* __restrict__ stat) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = p < P;
  int nw = 0, old = 0;
  if (live) {
    double x[3];
    for (int d = 0; d < DIM; d++) x[d] = coords[p * DIM + d];
    nw = (int)cell_of<DIM>(g.res, g.lo, g.hi, x, g.E);
    old = owner[p];
    new_owner[p] = nw;
  }
  const int lane = threadIdx.x & 63;
  const unsigned long long out = __ballot(live && nw >= (int)g.E);
  if (out && lane == __ffsll((long long)out) - 1) atomicAdd(&stat[0], __popcll(out));
  const bool moved = live && nw != old;
  int leader = lane, r = 0;
  const int na = same_key(moved, nw, &leader, &r);
  int base = 0;
  if (moved && lane == leader) base = atomicAdd(&cnt_a[nw], na);
  base = __shfl(base, leader);
  if (moved) {
    rank[p] = base + r;
    if (base + r >= kMaxScanAdd && nw < (int)g.E) stat[1] = 1;
  }
  const bool leaves = moved && old < (int)g.E;
  const int nr = same_key(leaves, old, &leader, &r);
  if (leaves && lane == leader) atomicAdd(&cnt_r[old], nr);
}

// (new table size, additions) of a cell, scanned together
struct CellCounts {
  const int* ptr;
  const int* ca;
  const int* cr;
  int E;
  __host__ __device__ unsigned long long operator()(int e) const {
    if (e >= E) return 0ull;
    const int n = ptr[e + 1] - ptr[e] - cr[e] + ca[e];
    return ((unsigned long long)(unsigned)n << 32) | (unsigned)ca[e];
  }
};

__global__ void k_group(long P, int E, const int* __restrict__ owner, const int* __restrict__ new_owner,
                        const int* __restrict__ rank, const unsigned long long* __restrict__ off,
                        int* __restrict__ add) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  const int nw = new_owner[p];
  if (nw == owner[p] || nw >= E) return;
  add[(unsigned)off[nw] + rank[p]] = (int)p;
}

// Per cell, replay removals/additions in particle-index order.  Eight lanes per cell: they copy
// the table in (an entry whose owner changed carries the top bit), find the next removal and the
// next addition by a scan and a three-step minimum, and copy the table out; the edits themselves
// are sequential and made by the cell's first lane.  The list lives in LDS (global memory where
// it is longer).  Latency-bound on the dependent loads table -> owner.
constexpr int kReplayLanes = 8, kReplayBlock = 256, kReplayList = 96;
constexpr int kReplayCells = kReplayBlock / kReplayLanes;
constexpr unsigned kGone = 0x80000000u, kNone = 0x7fffffffu;
template <bool SORTED>
__global__ __launch_bounds__(kReplayBlock) void k_replay(int E, const int* __restrict__ ptr,
                                                         const int* __restrict__ pid,
                                                         const int* __restrict__ new_owner,
                                                         const unsigned long long* __restrict__ off,
                                                         const int* __restrict__ cnt_r, const int* __restrict__ add,
                                                         int* tmp, int* __restrict__ new_ptr,
                                                         int* __restrict__ new_pid, const int* __restrict__ stat) {
  __shared__ unsigned list[kReplayCells][kReplayList + 1];
  if (!SORTED && stat[1]) return;
  const int lane = threadIdx.x & (kReplayLanes - 1), c = threadIdx.x / kReplayLanes;
  const int e = blockIdx.x * kReplayCells + c;
  if (e >= E) return;  // whole groups of eight lanes; nothing below waits for other groups
  const int s0 = ptr[e], n = ptr[e + 1] - s0;
  const unsigned long long o0 = off[e], o1 = off[e + 1];
  const int a0 = (int)(unsigned)o0, na = (int)((unsigned)o1 - (unsigned)o0), q0 = (int)(o0 >> 32);
  const int nr = cnt_r[e];
  int* out = new_pid + q0;
  if (lane == 0) {
    new_ptr[e] = q0;
    if (e == E - 1) new_ptr[E] = (int)(o1 >> 32);
  }
  if (na == 0 && nr == 0) {
    for (int k = lane; k < n; k += kReplayLanes) out[k] = pid[s0 + k];
    return;
  }
  unsigned* L = n + na <= kReplayList ? list[c] : (unsigned*)tmp + s0 + a0;
  for (int k = lane; k < n; k += kReplayLanes) {
    const int p = pid[s0 + k];
    L[k] = (unsigned)p | (nr != 0 && new_owner[p] != e ? kGone : 0u);
  }
  __threadfence_block();
  const int* A = add + a0;
  auto group_min = [&](unsigned long long v) {
    for (int s = 1; s < kReplayLanes; s <<= 1) {
      const unsigned long long w = __shfl_xor(v, s, kReplayLanes);
      v = w < v ? w : v;
    }
    return v;
  };
  int m = n, left_r = nr, left_a = na;
  // (index, position) of the next removal; index of the next addition
  auto next_removal = [&]() {
    unsigned long long v = (unsigned long long)kNone << 32;
    if (left_r > 0) {
      for (int k = lane; k < m; k += kReplayLanes) {
        const unsigned w = L[k];
        if (w & kGone) {
          const unsigned long long t = ((unsigned long long)(w & ~kGone) << 32) | (unsigned)k;
          v = t < v ? t : v;
        }
      }
      v = group_min(v);
    }
    return v;
  };
  auto next_addition = [&](long long last) {
    if (left_a == 0) return kNone;
    if (SORTED) return (unsigned)A[na - left_a];
    unsigned long long v = kNone;
    for (int k = lane; k < na; k += kReplayLanes) {
      const unsigned a = (unsigned)A[k];
      if ((long long)a > last && a < v) v = a;
    }
    return (unsigned)group_min(v);
  };
  unsigned long long r = next_removal();
  unsigned a = next_addition(-1);
  while (left_r > 0 || left_a > 0) {
    if ((unsigned)(r >> 32) < a) {
      const int k = (int)(unsigned)r;
      m--;
      left_r--;
      const unsigned w = L[m];
      if (lane == 0) L[k] = w;
      __threadfence_block();
      r = next_removal();
    } else {
      if (a == kNone) break;  // tables and owners disagree (never for tables this code keeps)
      if (lane == 0) L[m] = a;
      __threadfence_block();
      m++;
      left_a--;
      a = next_addition((long long)a);
    }
  }
  const int room = (int)(o1 >> 32) - q0;
  for (int k = lane; k < m && k < room; k += kReplayLanes) out[k] = (int)(L[k] & ~kGone);
}

__global__ void k_iota_moved(long P, const int* __restrict__ oldo, const int* __restrict__ newo, int* __restrict__ ids,
                             uint8_t* __restrict__ moved) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  ids[p] = (int)p;
  moved[p] = oldo[p] != newo[p];
}
__global__ void k_keys(int n, const int* __restrict__ mv, const int* __restrict__ newo, int* __restrict__ key) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) key[i] = newo[mv[i]];
}

// P: particles; cap: capacity of the swarm's particle arrays (the tables are exchanged with them)
RelocWork* reloc_create(long P, long E, long cap) {
  RelocWork* w = new RelocWork();
  w->P = P;
  w->E = E;
  const long Pm = P > 0 ? P : 1;
  if (cap < Pm) cap = Pm;
  UWG_HIP(hipMalloc(&w->new_owner, sizeof(int) * cap));
  UWG_HIP(hipMalloc(&w->pid, sizeof(int) * cap));
  UWG_HIP(hipMalloc(&w->rank, sizeof(int) * Pm));
  UWG_HIP(hipMalloc(&w->add, sizeof(int) * Pm));
  UWG_HIP(hipMalloc(&w->tmp, sizeof(int) * 2 * Pm));
  UWG_HIP(hipMalloc(&w->cnt, sizeof(int) * (2 * (E + 2) + 4)));
  w->stat = w->cnt + 2 * (E + 2);
  UWG_HIP(hipMalloc(&w->off, sizeof(unsigned long long) * (E + 2)));
  UWG_HIP(hipMalloc(&w->ptr, sizeof(int) * (E + 1)));
  const CellCounts f{w->ptr, w->cnt, w->cnt, (int)E};
  hipcub::TransformInputIterator<unsigned long long, CellCounts, hipcub::CountingInputIterator<int>> in(
      hipcub::CountingInputIterator<int>(0), f);
  UWG_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, w->cub_bytes, in, w->off, (int)(E + 1)));
  UWG_HIP(hipMalloc(&w->cub_tmp, w->cub_bytes));
  return w;
}

void reloc_destroy(RelocWork* w) {
  if (!w) return;
  for (void* p : {(void*)w->new_owner, (void*)w->pid, (void*)w->rank, (void*)w->add, (void*)w->tmp, (void*)w->cnt,
                  (void*)w->off, (void*)w->ptr, (void*)w->ids, (void*)w->mv, (void*)w->key, (void*)w->key_s,
                  (void*)w->moved, w->cub_tmp})
    (void)hipFree(p);
  delete w;
}

// additions of every cell in index order: the movers, stably sorted by new cell
static void sort_movers(RelocWork* w, const int* owner, hipStream_t s) {
  const long P = w->P;
  if (!w->ids) {
    for (int** a : {&w->ids, &w->mv, &w->key, &w->key_s}) UWG_HIP(hipMalloc(a, sizeof(int) * P));
    UWG_HIP(hipMalloc(&w->moved, P));
    size_t b1 = 0, b2 = 0;
    UWG_HIP(hipcub::DeviceSelect::Flagged(nullptr, b1, w->ids, w->moved, w->mv, w->stat, (int)P));
    UWG_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, b2, w->key, w->key_s, w->mv, w->add, (int)P));
    const size_t need = std::max(b1, b2);
    if (need > w->cub_bytes) {
      UWG_HIP(hipFree(w->cub_tmp));
      w->cub_tmp = nullptr;
      UWG_HIP(hipMalloc(&w->cub_tmp, need));
      w->cub_bytes = need;
    }
  }
  hipLaunchKernelGGL(k_iota_moved, nb(P, 256), 256, 0, s, P, owner, w->new_owner, w->ids, w->moved);
  size_t bytes = w->cub_bytes;
  int* nmv = w->stat + 1;  // the flag has been read
  UWG_HIP(hipcub::DeviceSelect::Flagged(w->cub_tmp, bytes, w->ids, w->moved, w->mv, nmv, (int)P, s));
  int n = 0;
  UWG_HIP(hipMemcpyAsync(&n, nmv, sizeof(int), hipMemcpyDeviceToHost, s));
  UWG_HIP(hipStreamSynchronize(s));
  if (n == 0) return;
  int bits = 1;
  while ((1L << bits) <= w->E) bits++;
  hipLaunchKernelGGL(k_keys, nb(n, 256), 256, 0, s, n, w->mv, w->new_owner, w->key);
  bytes = w->cub_bytes;
  UWG_HIP(hipcub::DeviceRadixSort::SortPairs(w->cub_tmp, bytes, w->key, w->key_s, w->mv, w->add, n, 0, bits, s));
}

void reloc_begin(RelocWork* w, hipStream_t s) {
  UWG_HIP(hipMemsetAsync(w->cnt, 0, sizeof(int) * (2 * (w->E + 2) + 4), s));
}
int* reloc_counters(RelocWork* w) { return w->stat + 2; }

// The new tables are built beside the old ones and exchanged with them at the end; they are not
// when counters[0] (particles the caller could not move) is non-zero.
long relocate(const Geom& g, long P, const double* coords, int*& owner, int*& cell_ptr, int*& cell_pid, RelocWork* w,
              hipStream_t s, int* counters) {
  const int E = (int)g.E;
  if (P == 0) return 0;
  if (!counters) reloc_begin(w, s);
  CellGrid cg;
  for (int d = 0; d < 3; d++) {
    cg.res[d] = g.res[d];
    cg.lo[d] = g.lo[d];
    cg.hi[d] = g.hi[d];
  }
  cg.E = g.E;
  int *ca = w->cnt, *cr = w->cnt + E + 2;
  if (g.dim == 3)
    hipLaunchKernelGGL(k_moves<3>, nb(P, 256), 256, 0, s, cg, P, coords, owner, w->new_owner, w->rank, ca, cr, w->stat);
  else
    hipLaunchKernelGGL(k_moves<2>, nb(P, 256), 256, 0, s, cg, P, coords, owner, w->new_owner, w->rank, ca, cr, w->stat);
  const CellCounts f{cell_ptr, ca, cr, E};
  hipcub::TransformInputIterator<unsigned long long, CellCounts, hipcub::CountingInputIterator<int>> in(
      hipcub::CountingInputIterator<int>(0), f);
  size_t bytes = w->cub_bytes;
  UWG_HIP(hipcub::DeviceScan::ExclusiveSum(w->cub_tmp, bytes, in, w->off, E + 1, s));
  hipLaunchKernelGGL(k_group, nb(P, 256), 256, 0, s, P, E, owner, w->new_owner, w->rank, w->off, w->add);
  hipLaunchKernelGGL(k_replay<false>, nb(E, kReplayCells), kReplayBlock, 0, s, E, cell_ptr, cell_pid, w->new_owner,
                     w->off, cr, w->add, w->tmp, w->ptr, w->pid, w->stat);
  UWG_HIP(hipGetLastError());
  int h[4];
  UWG_HIP(hipMemcpyAsync(h, w->stat, sizeof(h), hipMemcpyDeviceToHost, s));
  UWG_HIP(hipStreamSynchronize(s));
  if (counters) {
    counters[0] = h[2];
    counters[1] = h[3];
    if (h[2] > 0) return 0;
  }
  if (h[1]) {
    sort_movers(w, owner, s);
    hipLaunchKernelGGL(k_replay<true>, nb(E, kReplayCells), kReplayBlock, 0, s, E, cell_ptr, cell_pid, w->new_owner,
                       w->off, cr, w->add, w->tmp, w->ptr, w->pid, w->stat);
    UWG_HIP(hipGetLastError());
  }
  std::swap(owner, w->new_owner);
  std::swap(cell_ptr, w->ptr);
  std::swap(cell_pid, w->pid);
  return h[0];
}

// Exclusive prefix sum of 0/1 flags into 64-bit counts (the particle layout's skip counts).
void scan_exclusive_flags(const int* flags, long long* out, long n, hipStream_t s) {
  size_t bytes = 0;
  UWG_HIP(hipcub::DeviceScan::ExclusiveScan(nullptr, bytes, flags, out, hipcub::Sum(), 0LL, (int)n, s));
  void* tmp = nullptr;
  UWG_HIP(hipMalloc(&tmp, bytes + 16));
  UWG_HIP(hipcub::DeviceScan::ExclusiveScan(tmp, bytes, flags, out, hipcub::Sum(), 0LL, (int)n, s));
  UWG_HIP(hipStreamSynchronize(s));
  UWG_HIP(hipFree(tmp));
}

}  // namespace uwg
