// The owner partition's lists on the device (op2h_owner_plan.cpp builds the
// same on the host): the target graph the patches are grown over, and, once
// the host has grown them, per block its owned targets, its instances and each
// owned target's increments, in the same order.
//
// What the host spends on these is random access: five passes over the
// elements' map rows and the lists they scatter into.  Here a pass is one
// kernel over all elements with atomics for the places, and one workgroup per
// block then puts its own lists in order in LDS.  Only the breadth-first growth
// itself, a serial walk, stays on the host, and the prefix sums over blocks and
// targets, which it needs there.  720,000
// cells, 128-cell patches: a plan in 14 ms instead of 38, 2.88 million: 71
// instead of 238.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "op2h_plan_build.h"

#define OGCHECK(x)                                                           \
  do {                                                                       \
    hipError_t e_ = (x);                                                     \
    if (e_ != hipSuccess) {                                                  \
      printf("op2hip: %s failed at %s:%d: %s\n", #x, __FILE__, __LINE__,     \
             hipGetErrorString(e_));                                         \
      exit(-1);                                                              \
    }                                                                        \
  } while (0)

namespace op2h {
namespace {

constexpr int kSortMax = 4096;   // a block's targets or instances, sorted in LDS
constexpr int kListMax = 64;     // increments of one target, sorted by a thread
constexpr int kMaxInc = 8;       // increment args

struct Map {
  const int *row;  // device table [nel][dim]
  int nel, dim, ninc, nto;
  int idx[kMaxInc];
};

__device__ __forceinline__ int target(const Map &m, int e, int k) {
  return m.row[(size_t)e * m.dim + m.idx[k]];
}

// Per target how many neighbours it has (the other targets of its elements,
// once per element and position) and whether any element names it; the widest
// spread of one element's targets.
__global__ void k_degrees(Map m, int *__restrict deg, unsigned char *__restrict used,
                          int *width) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  int w = 0;
  if (e < m.nel) {
    int t[kMaxInc], lo = INT_MAX, hi = -1;
    for (int k = 0; k < m.ninc; ++k) {
      t[k] = target(m, e, k);
      lo = min(lo, t[k]);
      hi = max(hi, t[k]);
    }
    w = hi - lo;
    for (int k = 0; k < m.ninc; ++k) {
      int n = 0;
      for (int l = 0; l < m.ninc; ++l) n += l != k && t[l] != t[k];
      used[t[k]] = 1;
      if (n) atomicAdd(&deg[t[k]], n);
    }
  }
  for (int o = 32; o > 0; o >>= 1) w = max(w, __shfl_xor(w, o));
  if ((threadIdx.x & 63) == 0 && w > 0) atomicMax(width, w);
}

// Each neighbour as {element, its position among the element's increments} at
// the target's place: in any order within a target.
__global__ void k_neighbours(Map m, const int *__restrict off, int *__restrict fill,
                             unsigned long long *__restrict adj) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m.nel) return;
  for (int k = 0; k < m.ninc; ++k) {
    const int t = target(m, e, k);
    for (int l = 0; l < m.ninc; ++l)
      if (l != k && target(m, e, l) != t)
        adj[off[t] + atomicAdd(&fill[t], 1)] =
            ((unsigned long long)(unsigned)e << 32) | (unsigned)(k * m.ninc + l);
  }
}

// Each target's neighbours (at most kListMax (ninc - 1)) in element order, as
// targets.
__global__ void k_order_neighbours(Map m, const int *__restrict off,
                                   unsigned long long *__restrict adj, int *__restrict out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= m.nto) return;
  const int a = off[t], b = off[t + 1];
  for (int i = a + 1; i < b; ++i) {
    const unsigned long long v = adj[i];
    int j = i;
    for (; j > a && adj[j - 1] > v; --j) adj[j] = adj[j - 1];
    adj[j] = v;
  }
  for (int i = a; i < b; ++i)
    out[i] = target(m, (int)(adj[i] >> 32), (int)((unsigned)adj[i] % m.ninc));
}

// Position of element e's k-th target's block among the element's distinct
// blocks: true when no earlier position names the same block.
__device__ __forceinline__ bool first_of_block(const int *b, int k) {
  for (int l = 0; l < k; ++l)
    if (b[l] == b[k]) return false;
  return true;
}

// cnt: [3][nb], per block its targets, instances and increments.
__global__ void k_block_counts(Map m, const int *__restrict block_of, int nb,
                               int *__restrict cnt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m.nto && block_of[i] >= 0) atomicAdd(&cnt[block_of[i]], 1);
  if (i >= m.nel) return;
  int b[kMaxInc];
  for (int k = 0; k < m.ninc; ++k) {
    b[k] = block_of[target(m, i, k)];
    atomicAdd(&cnt[2 * nb + b[k]], 1);
    if (first_of_block(b, k)) atomicAdd(&cnt[nb + b[k]], 1);
  }
}

// Targets and instances to their blocks, in any order within one (fill: [2][nb]).
__global__ void k_block_fill(Map m, const int *__restrict block_of, int nb,
                             const int *__restrict owned_offs, const int *__restrict elem_offs,
                             int *__restrict fill, int *__restrict owned,
                             int *__restrict elems) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m.nto && block_of[i] >= 0) {
    const int b = block_of[i];
    owned[owned_offs[b] + atomicAdd(&fill[b], 1)] = i;
  }
  if (i >= m.nel) return;
  int b[kMaxInc];
  for (int k = 0; k < m.ninc; ++k) {
    b[k] = block_of[target(m, i, k)];
    if (first_of_block(b, k)) elems[elem_offs[b[k]] + atomicAdd(&fill[nb + b[k]], 1)] = i;
  }
}

// list[a, b) in ascending {key, value} order (key null: the value), through
// `s` (LDS, kSortMax); bitonic, the whole workgroup.
__device__ void sort_list(int *list, int a, int b, const int *key, unsigned long long *s) {
  const int n = b - a;
  int p = 1;
  while (p < n) p <<= 1;
  for (int i = threadIdx.x; i < p; i += blockDim.x)
    s[i] = i < n ? ((unsigned long long)(unsigned)(key ? key[list[a + i]] : list[a + i]) << 32) |
                       (unsigned)list[a + i]
                 : ~0ull;
  __syncthreads();
  for (int k = 2; k <= p; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < p; i += blockDim.x) {
        const int l = i ^ j;
        if (l > i) {
          const unsigned long long x = s[i], y = s[l];
          if ((x > y) == ((i & k) == 0)) {
            s[i] = y;
            s[l] = x;
          }
        }
      }
      __syncthreads();
    }
  for (int i = threadIdx.x; i < n; i += blockDim.x) list[a + i] = (int)(unsigned)s[i];
  __syncthreads();
}

// One workgroup per block: its targets ascending, its instances in element (or
// key) order, and where each of its targets sits in the owned list.
__global__ void __launch_bounds__(256)
    k_block_order(const int *__restrict owned_offs, int *owned,
                  const int *__restrict elem_offs, int *elems, const int *__restrict key,
                  int *__restrict pos) {
  __shared__ unsigned long long s[kSortMax];
  const int b = blockIdx.x;
  sort_list(owned, owned_offs[b], owned_offs[b + 1], nullptr, s);
  sort_list(elems, elem_offs[b], elem_offs[b + 1], key, s);
  for (int i = owned_offs[b] + threadIdx.x; i < owned_offs[b + 1]; i += blockDim.x)
    pos[owned[i]] = i;
}

// One workgroup per block: its targets' increments as (local instance * ninc +
// k) entries in (element or key, k) order, and their offsets.  longest: the
// most of one target; nothing is written for blocks with a longer list than
// kListMax.
__global__ void __launch_bounds__(256)
    k_block_increments(Map m, const int *__restrict block_of,
                       const int *__restrict owned_offs, const int *__restrict elem_offs,
                       const int *__restrict elems, const int *__restrict inc_offs,
                       const int *__restrict pos, const int *__restrict key,
                       int *__restrict csr_offs, unsigned short *csr, int *longest) {
  __shared__ int cnt[kSortMax], start[kSortMax], part[256];
  const int b = blockIdx.x, t = threadIdx.x;
  const int o0 = owned_offs[b], no = owned_offs[b + 1] - o0;
  const int e0 = elem_offs[b], ne = elem_offs[b + 1] - e0;
  for (int i = t; i < no; i += 256) cnt[i] = 0;
  __syncthreads();
  for (int j = t; j < ne; j += 256)
    for (int k = 0; k < m.ninc; ++k) {
      const int u = target(m, elems[e0 + j], k);
      if (block_of[u] == b) atomicAdd(&cnt[pos[u] - o0], 1);
    }
  __syncthreads();
  // exclusive sums: each thread a run of targets, then the threads
  const int per = (no + 255) / 256, lo = min(no, t * per), hi = min(no, lo + per);
  int sum = 0, most = 0;
  for (int i = lo; i < hi; ++i) {
    sum += cnt[i];
    most = max(most, cnt[i]);
  }
  part[t] = sum;
  for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o));
  if ((t & 63) == 0) atomicMax(longest, most);
  __syncthreads();
  int at = inc_offs[b];
  for (int i = 0; i < t; ++i) at += part[i];
  for (int i = lo; i < hi; ++i) {
    start[i] = at;
    csr_offs[o0 + i] = at;
    at += cnt[i];
    cnt[i] = 0;
  }
  __syncthreads();
  for (int j = t; j < ne; j += 256)
    for (int k = 0; k < m.ninc; ++k) {
      const int u = target(m, elems[e0 + j], k);
      if (block_of[u] == b) {
        const int i = pos[u] - o0;
        csr[start[i] + atomicAdd(&cnt[i], 1)] = (unsigned short)(j * m.ninc + k);
      }
    }
  __syncthreads();
  for (int i = t; i < no; i += 256) {
    unsigned short *l = csr + start[i];
    const int n = cnt[i];
    if (n > kListMax) continue;
    auto before = [&](unsigned short x, unsigned short y) {
      if (!key) return x < y;
      const int kx = key[elems[e0 + x / m.ninc]], ky = key[elems[e0 + y / m.ninc]];
      return kx != ky ? kx < ky : x % m.ninc < y % m.ninc;
    };
    for (int p = 1; p < n; ++p) {
      const unsigned short v = l[p];
      int q = p;
      for (; q > 0 && before(v, l[q - 1]); --q) l[q] = l[q - 1];
      l[q] = v;
    }
  }
}

// Fixed-width lists (at most four increments), 0xFFFF past the last.
__global__ void k_csr4(const int *__restrict csr_offs, const unsigned short *__restrict csr, int n,
                       ushort4 *__restrict out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int a = csr_offs[i], c = csr_offs[i + 1] - a;
  out[i] = make_ushort4(c > 0 ? csr[a] : 0xFFFF, c > 1 ? csr[a + 1] : 0xFFFF,
                        c > 2 ? csr[a + 2] : 0xFFFF, c > 3 ? csr[a + 3] : 0xFFFF);
}

int grid(size_t n) { return (int)((n + 255) / 256); }

// Device scratch of one build, freed at its end.  full: the device had no room
// for some of it (null), and the host builds the plan.
struct Scratch {
  std::vector<void *> ptrs;
  bool full = false;
  template <class T> T *get(size_t n, bool zero, hipStream_t st) {
    const size_t bytes = (std::max<size_t>(n, 1) * sizeof(T) + 3) / 4 * 4;
    void *p = full ? nullptr : op2h_extra_alloc(bytes);
    if (!p) {
      full = true;
      return nullptr;
    }
    if (zero) OGCHECK(hipMemsetAsync(p, 0, bytes, st));
    ptrs.push_back(p);
    return (T *)p;
  }
  ~Scratch() {
    for (void *p : ptrs) (void)hipFree(p);
  }
};

Map map_of(int nto, int nel, int dim, const int *map_d, int ninc, const int *inc_idx) {
  Map m{map_d, nel, dim, ninc, nto, {}};
  for (int k = 0; k < ninc; ++k) m.idx[k] = inc_idx[k];
  return m;
}

}  // namespace

bool gpu_owner_fits(int nto, int nel, int ninc) {
  return ninc <= kMaxInc && (long long)nel * ninc * ninc <= INT_MAX && nto > 0;
}

bool gpu_target_graph(int nto, int nel, int dim, const int *map_d, int ninc, const int *inc_idx,
                      hipStream_t st, TargetGraph &g) {
  Scratch S;
  const Map m = map_of(nto, nel, dim, map_d, ninc, inc_idx);
  int *deg = S.get<int>((size_t)nto + 1, true, st), *width = S.get<int>(1, true, st);
  unsigned char *used = S.get<unsigned char>(nto, true, st);
  if (S.full) return false;
  k_degrees<<<grid(nel), 256, 0, st>>>(m, deg, used, width);
  g.off.resize((size_t)nto + 1);
  g.used.resize(nto);
  int w = 0;
  OGCHECK(hipMemcpyAsync(g.off.data() + 1, deg, sizeof(int) * nto, hipMemcpyDeviceToHost, st));
  OGCHECK(hipMemcpyAsync(g.used.data(), used, nto, hipMemcpyDeviceToHost, st));
  OGCHECK(hipMemcpyAsync(&w, width, sizeof w, hipMemcpyDeviceToHost, st));
  OGCHECK(hipStreamSynchronize(st));
  g.width = w;
  // a target that so many elements name has more increments than its list here
  // may hold, and ordering its neighbours would be one thread's work
  for (int t = 0; t < nto; ++t)
    if (g.off[t + 1] > kListMax * (ninc - 1)) return false;
  g.off[0] = 0;
  for (int t = 0; t < nto; ++t) g.off[t + 1] += g.off[t];
  const size_t n = g.off[nto];
  g.adj.resize(n);
  if (!n) return true;
  int *off = S.get<int>((size_t)nto + 1, false, st), *out = S.get<int>(n, false, st);
  unsigned long long *adj = S.get<unsigned long long>(n, false, st);
  if (S.full) return false;
  OGCHECK(hipMemcpyAsync(off, g.off.data(), sizeof(int) * ((size_t)nto + 1),
                         hipMemcpyHostToDevice, st));
  OGCHECK(hipMemsetAsync(deg, 0, sizeof(int) * nto, st));
  k_neighbours<<<grid(nel), 256, 0, st>>>(m, off, deg, adj);
  k_order_neighbours<<<grid(nto), 256, 0, st>>>(m, off, adj, out);
  OGCHECK(hipGetLastError());
  OGCHECK(hipMemcpyAsync(g.adj.data(), out, sizeof(int) * n, hipMemcpyDeviceToHost, st));
  OGCHECK(hipStreamSynchronize(st));
  return true;
}

bool gpu_owner_lists(int nto, int nel, int dim, const int *map_d, int ninc, const int *inc_idx,
                     int nb, const std::vector<int> &block_of, const int *elem_key,
                     bool key_instances, hipStream_t st, OwnerPlanRec &rec) {
  Scratch S;
  op2h_owner_plan &P = rec.plan;
  const Map m = map_of(nto, nel, dim, map_d, ninc, inc_idx);
  int *blk = S.get<int>(nto, false, st), *cnt = S.get<int>(3 * (size_t)nb, true, st);
  int *inc_offs = S.get<int>((size_t)nb + 1, false, st);
  int *key = elem_key ? S.get<int>(nel, false, st) : nullptr;
  int *pos = S.get<int>(nto, false, st), *longest = S.get<int>(1, true, st);
  if (S.full) return false;
  OGCHECK(hipMemcpyAsync(blk, block_of.data(), sizeof(int) * nto, hipMemcpyHostToDevice, st));
  const int g = grid(std::max(nto, nel));
  k_block_counts<<<g, 256, 0, st>>>(m, blk, nb, cnt);
  // offsets of the blocks' targets, instances and increments
  std::vector<int> c(3 * (size_t)nb), offs[3];
  OGCHECK(hipMemcpyAsync(c.data(), cnt, sizeof(int) * c.size(), hipMemcpyDeviceToHost, st));
  OGCHECK(hipStreamSynchronize(st));
  int most[3] = {0, 0, 0};
  for (int a = 0; a < 3; ++a) {
    offs[a].assign((size_t)nb + 1, 0);
    for (int b = 0; b < nb; ++b) {
      const int n = c[(size_t)a * nb + b];
      offs[a][b + 1] = offs[a][b] + n;
      most[a] = std::max(most[a], n);
    }
  }
  if (most[0] > kSortMax || most[1] > kSortMax || (long long)most[1] * ninc > 65535) return false;
  const int n_owned = offs[0][nb], total = offs[1][nb], n_csr = offs[2][nb];
  int *owned_offs = rec.mem.upload(offs[0], st), *elem_offs = rec.mem.upload(offs[1], st);
  OGCHECK(hipMemcpyAsync(inc_offs, offs[2].data(), sizeof(int) * ((size_t)nb + 1),
                         hipMemcpyHostToDevice, st));
  if (key) OGCHECK(hipMemcpyAsync(key, elem_key, sizeof(int) * nel, hipMemcpyHostToDevice, st));
  int *owned = rec.mem.alloc<int>(n_owned), *elems = rec.mem.alloc<int>(total);
  int *csr_offs = rec.mem.alloc<int>((size_t)n_owned + 1);
  unsigned short *csr = rec.mem.alloc<unsigned short>(n_csr);
  OGCHECK(hipMemsetAsync(cnt, 0, sizeof(int) * 2 * (size_t)nb, st));
  k_block_fill<<<g, 256, 0, st>>>(m, blk, nb, owned_offs, elem_offs, cnt, owned, elems);
  k_block_order<<<nb, 256, 0, st>>>(owned_offs, owned, elem_offs, elems,
                                    key_instances ? key : nullptr, pos);
  k_block_increments<<<nb, 256, 0, st>>>(m, blk, owned_offs, elem_offs, elems, inc_offs, pos, key,
                                         csr_offs, csr, longest);
  OGCHECK(hipGetLastError());
  OGCHECK(hipMemcpyAsync(csr_offs + n_owned, &n_csr, sizeof(int), hipMemcpyHostToDevice, st));
  int ml = 0;
  OGCHECK(hipMemcpyAsync(&ml, longest, sizeof ml, hipMemcpyDeviceToHost, st));
  OGCHECK(hipStreamSynchronize(st));
  if (ml > kListMax) return false;
  P.nblocks = nb;
  P.total = total;
  P.max_elems = most[1];
  P.max_owned = most[0];
  P.owned_offs = owned_offs;
  P.owned = owned;
  P.elem_offs = elem_offs;
  P.elems = elems;
  P.csr_offs = csr_offs;
  P.csr = csr;
  P.n_owned = rec.n_owned = n_owned;
  rec.n_csr = n_csr;
  P.max_incs = ml;
  P.csr4 = nullptr;
  if (ml <= 4) {
    unsigned short *c4 = rec.mem.alloc<unsigned short>(4 * (size_t)std::max(n_owned, 1));
    k_csr4<<<grid(n_owned), 256, 0, st>>>(csr_offs, csr, n_owned, (ushort4 *)c4);
    OGCHECK(hipGetLastError());
    P.csr4 = c4;
  }
  OGCHECK(hipStreamSynchronize(st));
  return true;
}

}  // namespace op2h
