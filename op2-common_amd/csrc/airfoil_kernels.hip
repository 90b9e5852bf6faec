// airfoil_kernels.hip — the HIP-only target's output for the airfoil
// application (apps/c/airfoil/airfoil_plain/dp/airfoil.cpp:225-277): one
// op_par_loop_airfoil_<i>_<kernel> stub per loop, its gfx950 kernels and the
// application's device constants.
//
// User kernels (save_soln.h, adt_calc.h, res_calc.h, bres_calc.h, update.h) are
// device functions with the reference's expression trees; the whole library is
// compiled with -ffp-contract=off, so each multiply and add rounds as in the
// reference's host build.  Loops with indirect increments (res_calc,
// bres_calc) have five plans:
//   ATOMIC  one thread per edge, FP64 atomics on res;
//   COLOR   flat colouring, one launch per colour, plain read-modify-write;
//   STAGED  plan blocks staged in LDS, increments applied colour by colour
//           inside the block, blocks launched colour by colour;
//   GATHER  one thread per cell, the edges of the cell visited in edge order
//           and res accumulated in registers — the sequential executor's
//           summation order, so results match it bit for bit;
//   OWNER   one workgroup per patch of cells, each edge's flux once per patch
//           into LDS, each cell summing its own in edge order: the same bits.
// Inside a captured graph whole half steps run as one launch each
// (airfoil_patch.h).
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include <algorithm>
#include <cmath>
#include <climits>
#include <cstdio>
#include <cstring>

#include <map>
#include <vector>

#include "op2_hip_airfoil.h"
#include "op2_hip_rt.h"
#include "op2h_plan_build.h"
#include "airfoil_device.h"
#include "airfoil_patch.h"
#include "op2h_reduce.h"

#define KCHECK(x)                                                            \
  do {                                                                       \
    hipError_t e_ = (x);                                                     \
    if (e_ != hipSuccess) {                                                  \
      printf("op2hip: %s failed at %s:%d: %s\n", #x, __FILE__, __LINE__,     \
             hipGetErrorString(e_));                                         \
      exit(-1);                                                              \
    }                                                                        \
  } while (0)

// The airfoil constants (airfoil.cpp:149-164), offered by op_decl_const_char.
static int airfoil_consts(int dim, char const *type, int size, const char *dat,
                          char const *name) {
  (void)type;
  size_t bytes = (size_t)dim * size;
  if (!strcmp(name, "gam")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(gam_d), dat, bytes));
  else if (!strcmp(name, "gm1")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(gm1_d), dat, bytes));
  else if (!strcmp(name, "cfl")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(cfl_d), dat, bytes));
  else if (!strcmp(name, "eps")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(eps_d), dat, bytes));
  else if (!strcmp(name, "mach")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(mach_d), dat, bytes));
  else if (!strcmp(name, "alpha")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(alpha_d), dat, bytes));
  else if (!strcmp(name, "qinf")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(qinf_d), dat, bytes));
  else return 0;
  // FP32 copies of the flux constants, rounded once on the host
  float f[4];
  for (int i = 0; i < dim && i < 4; ++i)
    f[i] = size == 8 ? (float)((const double *)dat)[i] : ((const float *)dat)[i];
  if (!strcmp(name, "gam")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(gam_f), f, sizeof(float)));
  else if (!strcmp(name, "gm1")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(gm1_f), f, sizeof(float)));
  else if (!strcmp(name, "cfl")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(cfl_f), f, sizeof(float)));
  else if (!strcmp(name, "eps")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(eps_f), f, sizeof(float)));
  else if (!strcmp(name, "qinf")) KCHECK(hipMemcpyToSymbol(HIP_SYMBOL(qinf_f), f, 4 * sizeof(float)));
  return 1;
}

// Arithmetic per element of each loop's kernel in multiply-add equivalents
// (a division or square root counted as ten), the cost model's measure of a
// loop's compute: save_soln copies; adt_calc has a division, five square
// roots and ~50 operations; res_calc two divisions and ~75 operations;
// bres_calc ~40; update a division and ~12.
static const struct AirfoilConstHook {
  AirfoilConstHook() {
    op2h_register_const_hook(airfoil_consts);
    op2h_set_loop_arith("save_soln", 4);
    op2h_set_loop_arith("adt_calc", 64);
    op2h_set_loop_arith("res_calc", 60);
    op2h_set_loop_arith("bres_calc", 40);
    op2h_set_loop_arith("update", 20);
  }
} airfoil_const_hook;


namespace {
using namespace op2_dev;

// Launch with the kernel's declared argument types; with timing events
// (op2h_kernel_timer_events) through hipExtLaunchKernel, which stamps `e0` at
// the kernel's start and `e1` at its end (either may be NULL).
template <class Tuple, std::size_t... I>
void arg_ptrs(Tuple &t, void **p, std::index_sequence<I...>) {
  ((p[I] = (void *)&std::get<I>(t)), ...);
}

template <typename... KArgs, typename... Args>
void launch_k(bool ext, void *e0, void *e1, void (*kernel)(KArgs...), dim3 grid,
              dim3 block, size_t lds, hipStream_t st, Args... args) {
  static_assert(sizeof...(KArgs) == sizeof...(Args), "kernel argument count");
  std::tuple<KArgs...> t{static_cast<KArgs>(args)...};
  void *p[sizeof...(KArgs) > 0 ? sizeof...(KArgs) : 1];
  arg_ptrs(t, p, std::index_sequence_for<KArgs...>{});
  if (ext)
    KCHECK(hipExtLaunchKernel((const void *)kernel, grid, block, p, lds, st,
                              (hipEvent_t)e0, (hipEvent_t)e1, 0));
  else
    KCHECK(hipLaunchKernel((const void *)kernel, grid, block, p, lds, st));
}

// Timing for a loop launched with launch_k: kernel-attached events when
// timing is on, the event-pair timer (or the autotuner's) otherwise.
struct LoopTimer {
  op2h_loop_ctx *ctx;
  void *e0 = nullptr, *e1 = nullptr;
  bool ext = false;
  explicit LoopTimer(op2h_loop_ctx *c) : ctx(c) {
    ext = op2h_kernel_timer_events(c, &e0, &e1) != 0;
    if (!ext) op2h_kernel_timer_start(c);
  }
  void done() {
    if (!ext) op2h_kernel_timer_stop(ctx);
  }
};

// ---------------------------------------------------------------------------
// save_soln: qold = q over the whole dat, 16-byte vectors (direct copy)
// ---------------------------------------------------------------------------
__global__ void k_save_soln(const double2 *__restrict q, double2 *__restrict qold,
                            int n2) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n2) qold[i] = q[i];
}

// ---------------------------------------------------------------------------
// adt_calc: one thread per cell, nodes gathered through pcell.  NT: the
// cell's own streams (its pcell row, q, adt) non-temporal, the gathered
// nodes (shared with the neighbouring cells) cached as usual.
// ---------------------------------------------------------------------------
template <bool SOA, bool NT>
__global__ void k_adt_calc(const double *__restrict x, const double *__restrict q,
                           double *__restrict adt, const int *__restrict pcell,
                           int n, int sx, int sq) {
  int c = xcd_block(kXcds) * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const int4 cn = NT ? ld_int4_nt(pcell, c) : reinterpret_cast<const int4 *>(pcell)[c];
  double x1[2], x2[2], x3[2], x4[2], qc[4], a;
  if (NT) ld4_nt<SOA>(q, c, sq, qc);
  else ld4<SOA>(q, c, sq, qc);
  ld2<SOA>(x, cn.x, sx, x1);
  ld2<SOA>(x, cn.y, sx, x2);
  ld2<SOA>(x, cn.z, sx, x3);
  ld2<SOA>(x, cn.w, sx, x4);
  op2_k::adt_calc(x1, x2, x3, x4, qc, &a);
  if (NT) __builtin_nontemporal_store(a, adt + c);
  else adt[c] = a;
}

// ---------------------------------------------------------------------------
// res_calc
// ---------------------------------------------------------------------------
template <bool SOA>
__device__ __forceinline__ void res_edge(const double *__restrict x,
                                         const double *__restrict q,
                                         const double *__restrict adt,
                                         int2 en, int2 ec, int sx, int sq,
                                         double *r1, double *r2) {
  double x1[2], x2[2], q1[4], q2[4];
  ld2<SOA>(x, en.x, sx, x1);
  ld2<SOA>(x, en.y, sx, x2);
  ld4<SOA>(q, ec.x, sq, q1);
  ld4<SOA>(q, ec.y, sq, q2);
  double a1 = adt[ec.x], a2 = adt[ec.y];
  for (int d = 0; d < 4; ++d) {
    r1[d] = 0.0;
    r2[d] = 0.0;
  }
  op2_k::res_calc(x1, x2, q1, q2, &a1, &a2, r1, r2);
}

template <bool SOA>
__global__ void k_res_atomic(const double *__restrict x, const double *__restrict q,
                             const double *__restrict adt, double *res,
                             const int2 *__restrict pedge,
                             const int2 *__restrict pecell, int n, int sx, int sq) {
  int e = xcd_block(kXcds) * blockDim.x + threadIdx.x;
  if (e >= n) return;
  int2 en = pedge[e], ec = pecell[e];
  double r1[4], r2[4];
  res_edge<SOA>(x, q, adt, en, ec, sx, sq, r1, r2);
  atomic_add4<SOA>(res, ec.x, sq, r1);
  atomic_add4<SOA>(res, ec.y, sq, r2);
}

template <bool SOA>
__global__ void k_res_color(const double *__restrict x, const double *__restrict q,
                            const double *__restrict adt, double *res,
                            const int2 *__restrict pedge,
                            const int2 *__restrict pecell,
                            const int *__restrict col_reord, int start, int end,
                            int sx, int sq) {
  int i = start + blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= end) return;
  int e = col_reord[i];
  int2 en = pedge[e], ec = pecell[e];
  double r1[4], r2[4];
  res_edge<SOA>(x, q, adt, en, ec, sx, sq, r1, r2);
  add4<SOA>(res, ec.x, sq, r1);
  add4<SOA>(res, ec.y, sq, r2);
}

// Owner-compute: one thread per cell; entries are edge*2+slot in edge order.
template <bool SOA>
__global__ void k_res_gather(const double *__restrict x, const double *__restrict q,
                             const double *__restrict adt, double *res,
                             const int2 *__restrict pedge,
                             const int2 *__restrict pecell,
                             const int *__restrict offsets,
                             const int *__restrict entries,
                             const int *__restrict targets, int ntargets, int sx,
                             int sq) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntargets) return;
  int cell = targets[t];
  double acc[4];
  ld4<SOA>(res, cell, sq, acc);
  int k0 = offsets[t], k1 = offsets[t + 1];
  for (int k = k0; k < k1; ++k) {
    int ent = entries[k];
    int e = ent >> 1;
    int2 en = pedge[e], ec = pecell[e];
    double r1[4], r2[4];
    res_edge<SOA>(x, q, adt, en, ec, sx, sq, r1, r2);
    const double *r = (ent & 1) ? r2 : r1;
    acc[0] += r[0];
    acc[1] += r[1];
    acc[2] += r[2];
    acc[3] += r[3];
  }
  st4<SOA>(res, cell, sq, acc);
}

// Owner-compute with K lanes per cell: lane k of a cell's group computes the
// flux of the cell's k-th edge (in edge order); the group's first lane adds
// the K results to res in edge order, so the sum is the sequential
// executor's.  Every lane of a wave reaches every shuffle.
template <bool SOA, int K>
__global__ void __launch_bounds__(1024)
    k_res_gather_lanes(const double *__restrict x, const double *__restrict q,
                       const double *__restrict adt, double *res,
                       const int2 *__restrict pedge, const int2 *__restrict pecell,
                       const int *__restrict offsets, const int *__restrict entries,
                       const int *__restrict targets, int ntargets, int sx, int sq) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  const int t = g / K, k = g & (K - 1);
  const bool valid = t < ntargets;
  int k0 = 0, cnt = 0;
  if (valid) {
    k0 = offsets[t];
    cnt = offsets[t + 1] - k0;
  }
  double r[4] = {0.0, 0.0, 0.0, 0.0};
  if (k < cnt) {
    int ent = entries[k0 + k];
    int e = ent >> 1;
    double r1[4], r2[4];
    res_edge<SOA>(x, q, adt, pedge[e], pecell[e], sx, sq, r1, r2);
    for (int d = 0; d < 4; ++d) r[d] = (ent & 1) ? r2[d] : r1[d];
  }
  const int lead = (threadIdx.x & 63) & ~(K - 1);
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  int cell = 0;
  if (k == 0 && valid) {
    cell = targets[t];
    ld4<SOA>(res, cell, sq, acc);
  }
  for (int j = 0; j < K; ++j) {
    double v[4];
    for (int d = 0; d < 4; ++d) v[d] = __shfl(r[d], lead + j, 64);
    if (j < cnt)
      for (int d = 0; d < 4; ++d) acc[d] += v[d];
  }
  if (k == 0 && valid) st4<SOA>(res, cell, sq, acc);
}

// Gather with a packed table: rec[t*K + k] = {n0, n1, other cell, slot} of
// the k-th edge of target t in edge order, {-1, -1, -1, 0} past its last edge.
template <int K>
__global__ void k_pack_res_gather(const int2 *__restrict pedge,
                                  const int2 *__restrict pecell,
                                  const int *__restrict offsets,
                                  const int *__restrict entries, int ntargets,
                                  int4 *__restrict rec) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)ntargets * K) return;
  int t = (int)(i / K), k = (int)(i % K);
  int k0 = offsets[t], cnt = offsets[t + 1] - k0;
  int4 r = make_int4(-1, -1, -1, 0);
  if (k < cnt) {
    int ent = entries[k0 + k];
    int e = ent >> 1, slot = ent & 1;
    int2 en = pedge[e], ec = pecell[e];
    r = make_int4(en.x, en.y, slot ? ec.x : ec.y, slot);
  }
  rec[i] = r;
}

template <bool SOA, int K>
__global__ void __launch_bounds__(1024)
    k_res_gather_packed(const double *__restrict x, const double *__restrict q,
                        const double *__restrict adt, double *res,
                        const int4 *__restrict rec, const int *__restrict targets,
                        int ntargets, int sx, int sq) {
  const int g = xcd_block(kXcds) * blockDim.x + threadIdx.x;
  const int t = g / K, k = g & (K - 1);
  const bool valid = t < ntargets;
  const int cell = valid ? targets[t] : 0;
  const int4 rr = valid ? rec[g] : make_int4(-1, -1, -1, 0);
  double r[4] = {0.0, 0.0, 0.0, 0.0};
  const int has = rr.x >= 0;
  if (has) {
    double x1[2], x2[2], qa[4], qb[4];
    ld2<SOA>(x, rr.x, sx, x1);
    ld2<SOA>(x, rr.y, sx, x2);
    ld4<SOA>(q, cell, sq, qa);
    ld4<SOA>(q, rr.z, sq, qb);
    // the edge's ecell[0] side is q1 whichever side this lane's cell is:
    // operands are selected, not branched on, so the wave evaluates one flux
    const bool second = rr.w != 0;
    double q1[4], q2[4];
    for (int d = 0; d < 4; ++d) {
      q1[d] = second ? qb[d] : qa[d];
      q2[d] = second ? qa[d] : qb[d];
    }
    const double aa = adt[cell], ab = adt[rr.z];
    double a1 = second ? ab : aa, a2 = second ? aa : ab;
    double r1[4] = {0.0, 0.0, 0.0, 0.0}, r2[4] = {0.0, 0.0, 0.0, 0.0};
    op2_k::res_calc(x1, x2, q1, q2, &a1, &a2, r1, r2);
    for (int d = 0; d < 4; ++d) r[d] = second ? r2[d] : r1[d];
  }
  static_assert(K == 4, "quad broadcasts assume four lanes per cell");
  // the quad's increments in edge order (lane 0 first), added to res
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  if (k == 0 && valid) ld4<SOA>(res, cell, sq, acc);
  double v[4][4];
  int hv[4];
  for (int d = 0; d < 4; ++d) {
    v[0][d] = quad_bcast<0>(r[d]);
    v[1][d] = quad_bcast<1>(r[d]);
    v[2][d] = quad_bcast<2>(r[d]);
    v[3][d] = quad_bcast<3>(r[d]);
  }
  hv[0] = quad_bcast<0>(has);
  hv[1] = quad_bcast<1>(has);
  hv[2] = quad_bcast<2>(has);
  hv[3] = quad_bcast<3>(has);
  for (int j = 0; j < 4; ++j)
    if (hv[j])
      for (int d = 0; d < 4; ++d) acc[d] += v[j][d];
  if (k == 0 && valid) st4<SOA>(res, cell, sq, acc);
}

struct StagedArgs {
  const int *blkmap, *offset, *nelems, *nthrcol;
  const unsigned char *thrcol;
  const int *ind_offs_n, *ind_sizes_n, *ind_map_n;  // node map slot
  const int *ind_offs_c, *ind_sizes_c, *ind_map_c;  // cell map slot
  const unsigned short *loc_n0, *loc_n1, *loc_c0, *loc_c1;
  int max_n, max_c;
};

// Two-level coloured, LDS-staged res_calc: one workgroup per plan block.
// LDS: x of the block's nodes [max_n][2], q [max_c][4], adt [max_c],
// res increments [max_c][4].
template <bool SOA>
__global__ void __launch_bounds__(1024)
    k_res_staged(const double *__restrict x, const double *__restrict q,
                 const double *__restrict adt, double *__restrict res,
                 StagedArgs P, int block_offset, int sx, int sq) {
  extern __shared__ double lds[];
  const int b = P.blkmap[blockIdx.x + block_offset];
  const int off = P.offset[b], nel = P.nelems[b];
  const int nn = P.ind_sizes_n[b], nbase = P.ind_offs_n[b];
  const int nc = P.ind_sizes_c[b], cbase = P.ind_offs_c[b];
  double *lx = lds;
  double *lq = lx + 2 * P.max_n;
  double *la = lq + 4 * P.max_c;
  double *lr = la + P.max_c;
  for (int k = threadIdx.x; k < nn; k += blockDim.x) {
    double v[2];
    ld2<SOA>(x, P.ind_map_n[nbase + k], sx, v);
    lx[2 * k] = v[0];
    lx[2 * k + 1] = v[1];
  }
  for (int k = threadIdx.x; k < nc; k += blockDim.x) {
    int cell = P.ind_map_c[cbase + k];
    double v[4];
    ld4<SOA>(q, cell, sq, v);
    lq[4 * k] = v[0];
    lq[4 * k + 1] = v[1];
    lq[4 * k + 2] = v[2];
    lq[4 * k + 3] = v[3];
    la[k] = adt[cell];
    lr[4 * k] = 0.0;
    lr[4 * k + 1] = 0.0;
    lr[4 * k + 2] = 0.0;
    lr[4 * k + 3] = 0.0;
  }
  __syncthreads();
  double r1[4] = {0.0, 0.0, 0.0, 0.0}, r2[4] = {0.0, 0.0, 0.0, 0.0};
  int col = -1, l0 = 0, l1 = 0;
  if ((int)threadIdx.x < nel) {
    const int e = off + threadIdx.x;
    const int a0 = P.loc_n0[e], a1 = P.loc_n1[e];
    l0 = P.loc_c0[e];
    l1 = P.loc_c1[e];
    op2_k::res_calc(lx + 2 * a0, lx + 2 * a1, lq + 4 * l0, lq + 4 * l1, la + l0,
                    la + l1, r1, r2);
    col = P.thrcol[e];
  }
  const int ncol = P.nthrcol[b];
  for (int c = 0; c < ncol; ++c) {
    if (col == c) {
      for (int d = 0; d < 4; ++d) {
        lr[4 * l0 + d] += r1[d];
        lr[4 * l1 + d] += r2[d];
      }
    }
    __syncthreads();
  }
  for (int k = threadIdx.x; k < nc; k += blockDim.x)
    add4<SOA>(res, P.ind_map_c[cbase + k], sq, lr + 4 * k);
}


// Per-instance records of res_calc's owner plan: {pedge[e], pecell[e]}.
__global__ void k_pack_owner_res(const int2 *__restrict pedge,
                                 const int2 *__restrict pecell,
                                 const int *__restrict elems, int total,
                                 int4 *__restrict inst) {
  int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= total) return;
  int e = elems[j];
  int2 n = pedge[e], c = pecell[e];
  inst[j] = make_int4(n.x, n.y, c.x, c.y);
}

// Compact records, one workgroup per block: the lowest cell and node its
// instances touch, and when every cell and node lies within 65535 of those,
// 8-byte records of 16-bit offsets (else the block keeps the 16-byte ones).
__global__ void __launch_bounds__(256)
    k_pack_owner_res8(const int4 *__restrict inst, const int *__restrict elem_offs,
                      int2 *__restrict base, uint2 *__restrict inst8) {
  __shared__ int s_min[2][4], s_max[2][4];
  const int b = blockIdx.x, t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int e0 = elem_offs[b], e1 = elem_offs[b + 1];
  int cmin = INT_MAX, nmin = INT_MAX, cmax = -1, nmax = -1;
  for (int j = e0 + t; j < e1; j += blockDim.x) {
    const int4 r = inst[j];
    nmin = min(nmin, min(r.x, r.y));
    nmax = max(nmax, max(r.x, r.y));
    cmin = min(cmin, min(r.z, r.w));
    cmax = max(cmax, max(r.z, r.w));
  }
  for (int o = 32; o > 0; o >>= 1) {
    cmin = min(cmin, __shfl_xor(cmin, o));
    nmin = min(nmin, __shfl_xor(nmin, o));
    cmax = max(cmax, __shfl_xor(cmax, o));
    nmax = max(nmax, __shfl_xor(nmax, o));
  }
  if (lane == 0) {
    s_min[0][w] = cmin;
    s_min[1][w] = nmin;
    s_max[0][w] = cmax;
    s_max[1][w] = nmax;
  }
  __syncthreads();
  for (int k = 0; k < 4; ++k) {
    cmin = min(cmin, s_min[0][k]);
    nmin = min(nmin, s_min[1][k]);
    cmax = max(cmax, s_max[0][k]);
    nmax = max(nmax, s_max[1][k]);
  }
  const bool fits = e1 > e0 && cmax - cmin <= 0xFFFF && nmax - nmin <= 0xFFFF;
  if (t == 0) base[b] = fits ? make_int2(cmin, nmin) : make_int2(0, -1);
  if (!fits) return;
  for (int j = e0 + t; j < e1; j += blockDim.x) {
    const int4 r = inst[j];
    inst8[j] = make_uint2((unsigned)(r.x - nmin) | ((unsigned)(r.y - nmin) << 16),
                          (unsigned)(r.z - cmin) | ((unsigned)(r.w - cmin) << 16));
  }
}

// Owner plan for res_calc's args (res incremented via pecell 0 (+f) and 1
// (-f)), with its instance records packed once per plan; a NULL plan or an
// unexpected shape is fatal, as the reference's plan errors are.
static OwnerArgs owner_args_res(const op2h_owner_plan *p, const op_arg *args,
                                hipStream_t st) {
  if (!p) exit(-1);
  if (p->inc_of_arg[6] != 0 || p->inc_of_arg[7] != 1 || p->ninc != 2) {
    printf("op2hip: res_calc owner plan expects res via ecell[0], ecell[1]\n");
    exit(-1);
  }
  // packed once per plan (the plan pins the set, the maps and the block size)
  char key[96];
  snprintf(key, sizeof key, "res_calc.owner.%p", (const void *)p);
  int fresh = 0;
  int4 *inst = (int4 *)op2h_plan_user(key, sizeof(int4) * (size_t)p->total, &fresh);
  if (fresh && p->total)
    k_pack_owner_res<<<grid_for(p->total, 256), 256, 0, st>>>(
        (const int2 *)args[0].map->map_d, (const int2 *)args[2].map->map_d, p->elems,
        p->total, inst);
  // compact records: blocks per launch are at most a few hundred thousand, so
  // one workgroup per block
  snprintf(key, sizeof key, "res_calc.owner8.%p", (const void *)p);
  const size_t base_bytes = (sizeof(int2) * (size_t)p->nblocks + 255) / 256 * 256;
  char *c8 = (char *)op2h_plan_user(key, base_bytes + sizeof(uint2) * (size_t)p->total, &fresh);
  if (fresh && p->nblocks)
    k_pack_owner_res8<<<p->nblocks, 256, 0, st>>>(inst, p->elem_offs, (int2 *)c8,
                                                  (uint2 *)(c8 + base_bytes));
  OwnerArgs A;
  A.inst = inst;
  A.base = (const int2 *)c8;
  A.inst8 = (const uint2 *)(c8 + base_bytes);
  A.elem_offs = p->elem_offs;
  A.owned_offs = p->owned_offs;
  A.owned = p->owned;
  A.csr_offs = p->csr_offs;
  A.csr = p->csr;
  // the plan's fixed-width increment lists (quadrilateral cells: at most
  // four edges each): one 8-byte load per owned cell
  A.csr4 = (const ushort4 *)p->csr4;
  A.max_e = p->max_elems;
  return A;
}

// Owner-compute res_calc (op2_dev::owner_res_block), one workgroup per block
// of owned cells, blocks in XCD order.  R: the type of adt and res (float:
// mixed mode, SP fluxes from x and q rounded).  LDS: fluxes [max_e][4].
template <class R, bool SOA, bool C4>
__global__ void __launch_bounds__(1024)
    k_res_owner(const double *__restrict x, const double *__restrict q,
                const R *__restrict adt, R *__restrict res, OwnerArgs P, int sx, int sq,
                int zero_acc) {
  extern __shared__ double lf[];
  owner_res_block<R, SOA, C4>(xcd_block(kXcds), x, q, adt, res, P, sx, sq, (R *)lf,
                              zero_acc != 0);
}

// ---------------------------------------------------------------------------
// bres_calc
// ---------------------------------------------------------------------------
template <bool SOA>
__device__ __forceinline__ void bres_edge(const double *__restrict x,
                                          const double *__restrict q,
                                          const double *__restrict adt,
                                          int2 bn, int cell, int bound, int sx,
                                          int sq, double *r) {
  double x1[2], x2[2], q1[4];
  ld2<SOA>(x, bn.x, sx, x1);
  ld2<SOA>(x, bn.y, sx, x2);
  ld4<SOA>(q, cell, sq, q1);
  double a1 = adt[cell];
  for (int d = 0; d < 4; ++d) r[d] = 0.0;
  op2_k::bres_calc(x1, x2, q1, &a1, r, &bound);
}

template <bool SOA>
__global__ void k_bres_atomic(const double *__restrict x, const double *__restrict q,
                              const double *__restrict adt, double *res,
                              const int2 *__restrict pbedge,
                              const int *__restrict pbecell,
                              const int *__restrict bound, int n, int sx, int sq) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  int cell = pbecell[e];
  double r[4];
  bres_edge<SOA>(x, q, adt, pbedge[e], cell, bound[e], sx, sq, r);
  atomic_add4<SOA>(res, cell, sq, r);
}

template <bool SOA>
__global__ void k_bres_color(const double *__restrict x, const double *__restrict q,
                             const double *__restrict adt, double *res,
                             const int2 *__restrict pbedge,
                             const int *__restrict pbecell,
                             const int *__restrict bound,
                             const int *__restrict col_reord, int start, int end,
                             int sx, int sq) {
  int i = start + blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= end) return;
  int e = col_reord[i];
  int cell = pbecell[e];
  double r[4];
  bres_edge<SOA>(x, q, adt, pbedge[e], cell, bound[e], sx, sq, r);
  add4<SOA>(res, cell, sq, r);
}

template <bool SOA>
__global__ void k_bres_gather(const double *__restrict x, const double *__restrict q,
                              const double *__restrict adt, double *res,
                              const int2 *__restrict pbedge,
                              const int *__restrict bound,
                              const int *__restrict offsets,
                              const int *__restrict entries,
                              const int *__restrict targets, int ntargets, int sx,
                              int sq) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntargets) return;
  int cell = targets[t];
  double acc[4];
  ld4<SOA>(res, cell, sq, acc);
  for (int k = offsets[t]; k < offsets[t + 1]; ++k) {
    int e = entries[k];  // map dim 1: entry = bedge
    double r[4];
    bres_edge<SOA>(x, q, adt, pbedge[e], cell, bound[e], sx, sq, r);
    acc[0] += r[0];
    acc[1] += r[1];
    acc[2] += r[2];
    acc[3] += r[3];
  }
  st4<SOA>(res, cell, sq, acc);
}

struct BStagedArgs {
  const int *blkmap, *offset, *nelems, *nthrcol;
  const unsigned char *thrcol;
  const int *ind_offs_n, *ind_sizes_n, *ind_map_n;
  const int *ind_offs_c, *ind_sizes_c, *ind_map_c;
  const unsigned short *loc_n0, *loc_n1, *loc_c0;
  int max_n, max_c;
};

template <bool SOA>
__global__ void __launch_bounds__(1024)
    k_bres_staged(const double *__restrict x, const double *__restrict q,
                  const double *__restrict adt, double *__restrict res,
                  const int *__restrict bound, BStagedArgs P, int block_offset,
                  int sx, int sq) {
  extern __shared__ double lds[];
  const int b = P.blkmap[blockIdx.x + block_offset];
  const int off = P.offset[b], nel = P.nelems[b];
  const int nn = P.ind_sizes_n[b], nbase = P.ind_offs_n[b];
  const int nc = P.ind_sizes_c[b], cbase = P.ind_offs_c[b];
  double *lx = lds;
  double *lq = lx + 2 * P.max_n;
  double *la = lq + 4 * P.max_c;
  double *lr = la + P.max_c;
  for (int k = threadIdx.x; k < nn; k += blockDim.x) {
    double v[2];
    ld2<SOA>(x, P.ind_map_n[nbase + k], sx, v);
    lx[2 * k] = v[0];
    lx[2 * k + 1] = v[1];
  }
  for (int k = threadIdx.x; k < nc; k += blockDim.x) {
    int cell = P.ind_map_c[cbase + k];
    double v[4];
    ld4<SOA>(q, cell, sq, v);
    for (int d = 0; d < 4; ++d) {
      lq[4 * k + d] = v[d];
      lr[4 * k + d] = 0.0;
    }
    la[k] = adt[cell];
  }
  __syncthreads();
  double r[4] = {0.0, 0.0, 0.0, 0.0};
  int col = -1, l0 = 0;
  if ((int)threadIdx.x < nel) {
    const int e = off + threadIdx.x;
    const int a0 = P.loc_n0[e], a1 = P.loc_n1[e];
    l0 = P.loc_c0[e];
    int bd = bound[e];
    op2_k::bres_calc(lx + 2 * a0, lx + 2 * a1, lq + 4 * l0, la + l0, r, &bd);
    col = P.thrcol[e];
  }
  const int ncol = P.nthrcol[b];
  for (int c = 0; c < ncol; ++c) {
    if (col == c)
      for (int d = 0; d < 4; ++d) lr[4 * l0 + d] += r[d];
    __syncthreads();
  }
  for (int k = threadIdx.x; k < nc; k += blockDim.x)
    add4<SOA>(res, P.ind_map_c[cbase + k], sq, lr + 4 * k);
}

// ---------------------------------------------------------------------------
// update, with the rms (INC) and maxerr (MAX, errloc argmax) reductions.
// Each workgroup reduces its elements (waves by shuffles, then LDS) and writes
// one partial; a one-workgroup kernel then combines the partials in
// workgroup order and writes the result slots.  The kernel boundary makes the
// partials visible across XCDs, so no device-scope fence is needed inside the
// streaming kernel (on a multi-XCD gfx950 such a fence writes back L2).
// ---------------------------------------------------------------------------
using op2h_red::MaxLoc;
using op2h_red::UpdateAcc;
using op2h_red::UpdateParts;

// The cells a workgroup of the update (or of a direct chain fused with it)
// takes, and the partial it writes: with chunk > 0 the contiguous cells
// [L chunk, (L+1) chunk) of the workgroup the XCD-ordered id L names, its
// threads striding by the workgroup size; with chunk 0 a grid-stride sweep
// from the workgroup's own id.  The same cells in the same order per
// partial, so every kernel launched with one shape reduces the same bits.
struct CellRange {
  int L, c, end, step;
};
__device__ __forceinline__ CellRange cell_range(int n, int chunk) {
  if (chunk > 0) {
    const int L = xcd_block(kXcds);
    return {L, L * chunk + (int)threadIdx.x, min(n, (L + 1) * chunk), (int)blockDim.x};
  }
  return {(int)blockIdx.x, (int)(blockIdx.x * blockDim.x + threadIdx.x), n,
          (int)(gridDim.x * blockDim.x)};
}

// R: the type of res and adt (float: mixed mode, the update in FP64 from them).
template <class R, bool SOA>
__global__ void __launch_bounds__(1024)
    k_update(const double *__restrict qold, double *__restrict q, R *__restrict res,
             const R *__restrict adt, int n, int s, UpdateParts parts,
             const int *__restrict oldidx, int chunk) {
  UpdateAcc acc;
  const CellRange cr = cell_range(n, chunk);
  for (int c = cr.c; c < cr.end; c += cr.step) {
    double qo[4], qn[4], r[4], cs = 0.0;
    R rr[4];
    const double a = (double)adt[c];
    ld4<SOA>(qold, c, s, qo);
    ld4r<SOA>(res, c, s, rr);
    for (int d = 0; d < 4; ++d) r[d] = (double)rr[d];
    // op_arg_idx: the application's element index (transparent renumbering)
    const int ci = oldidx ? oldidx[c] : c;
    double mx = -INFINITY;
    int at;
    op2_k::update(qo, qn, r, &a, &cs, &mx, &ci, &at);
    op2h_red::add_cell(acc, cs, mx, ci);
    st4<SOA>(q, c, s, qn);
    const R z[4] = {0, 0, 0, 0};
    st4r<SOA>(res, c, s, z);
  }
  op2h_red::write_partial(acc, parts, cr.L);
}

// Two groups of 256 threads: group 0 finishes rms (sum), group 1 maxerr and
// errloc (max, lowest element on ties), both with op2h_red::group_reduce, the
// reduction the graph's history kernel applies to deferred partials.
constexpr int kFinishThreads = 2 * op2h_red::kRedThreads;

__global__ void __launch_bounds__(kFinishThreads)
    k_update_finish(UpdateParts parts, int nparts, double *__restrict slot_rms,
                    double *__restrict slot_max) {
  __shared__ double s_v[2][op2h_red::kRedThreads / 64], s_lo[2][op2h_red::kRedThreads / 64];
  __shared__ int s_l[2][op2h_red::kRedThreads / 64];
  const int grp = threadIdx.x / op2h_red::kRedThreads;
  const int t = threadIdx.x % op2h_red::kRedThreads;
  // one call site for both groups (the reduction holds a workgroup barrier)
  const op2h_red::ValLoc r = op2h_red::group_reduce(
      grp == 0 ? parts.hi : parts.mx, grp == 0 ? nullptr : parts.loc,
      grp == 0 ? parts.lo : nullptr, nparts, grp == 0 ? 4 : 2, t, s_v[grp], s_l[grp], s_lo[grp]);
  if (t == 0) {
    if (grp == 0) {
      slot_rms[0] = r.v;
    } else {
      slot_max[0] = r.v;
      reinterpret_cast<int *>(slot_max + 1)[0] = r.loc;
    }
  }
}

// ---------------------------------------------------------------------------
// Mixed precision: adt and res stored in FP32, fluxes and adt computed in FP32
// from FP32 copies of q and x; q, qold, the update and the rms/maxerr
// reductions stay FP64.
// ---------------------------------------------------------------------------
template <bool SOA>
__device__ __forceinline__ void atomic_add4s(float *p, int n, int s, const float *v) {
  size_t st = SOA ? (size_t)s : 1, base = SOA ? (size_t)n : 4 * (size_t)n;
  for (int d = 0; d < 4; ++d) unsafeAtomicAdd(p + base + d * st, v[d]);
}

template <bool SOA>
__global__ void k_adt_calc_mixed(const double *__restrict x, const double *__restrict q,
                                 float *__restrict adt, const int *__restrict pcell,
                                 int n, int sx, int sq) {
  int c = xcd_block(kXcds) * blockDim.x + threadIdx.x;
  if (c >= n) return;
  int4 cn = reinterpret_cast<const int4 *>(pcell)[c];
  float x1[2], x2[2], x3[2], x4[2], qc[4], a;
  ld2r<SOA>(x, cn.x, sx, x1);
  ld2r<SOA>(x, cn.y, sx, x2);
  ld2r<SOA>(x, cn.z, sx, x3);
  ld2r<SOA>(x, cn.w, sx, x4);
  ld4r<SOA>(q, c, sq, qc);
  op2_kf::adt_calc(x1, x2, x3, x4, qc, &a);
  adt[c] = a;
}

template <bool SOA>
__global__ void k_res_atomic_mixed(const double *__restrict x, const double *__restrict q,
                                   const float *__restrict adt, float *res,
                                   const int2 *__restrict pedge,
                                   const int2 *__restrict pecell, int n, int sx, int sq) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  int2 en = pedge[e], ec = pecell[e];
  float x1[2], x2[2], q1[4], q2[4];
  ld2r<SOA>(x, en.x, sx, x1);
  ld2r<SOA>(x, en.y, sx, x2);
  ld4r<SOA>(q, ec.x, sq, q1);
  ld4r<SOA>(q, ec.y, sq, q2);
  float a1 = adt[ec.x], a2 = adt[ec.y];
  float r1[4] = {0.f, 0.f, 0.f, 0.f}, r2[4] = {0.f, 0.f, 0.f, 0.f};
  op2_kf::res_calc(x1, x2, q1, q2, &a1, &a2, r1, r2);
  atomic_add4s<SOA>(res, ec.x, sq, r1);
  atomic_add4s<SOA>(res, ec.y, sq, r2);
}

template <bool SOA, int K>
__global__ void __launch_bounds__(1024)
    k_res_gather_packed_mixed(const double *__restrict x, const double *__restrict q,
                              const float *__restrict adt, float *res,
                              const int4 *__restrict rec, const int *__restrict targets,
                              int ntargets, int sx, int sq) {
  const int g = xcd_block(kXcds) * blockDim.x + threadIdx.x;
  const int t = g / K, k = g & (K - 1);
  const bool valid = t < ntargets;
  const int cell = valid ? targets[t] : 0;
  const int4 rr = valid ? rec[g] : make_int4(-1, -1, -1, 0);
  float r[4] = {0.f, 0.f, 0.f, 0.f};
  const int has = rr.x >= 0;
  if (has) {
    float x1[2], x2[2], qa[4], qb[4];
    ld2r<SOA>(x, rr.x, sx, x1);
    ld2r<SOA>(x, rr.y, sx, x2);
    ld4r<SOA>(q, cell, sq, qa);
    ld4r<SOA>(q, rr.z, sq, qb);
    const bool second = rr.w != 0;
    float q1[4], q2[4];
    for (int d = 0; d < 4; ++d) {
      q1[d] = second ? qb[d] : qa[d];
      q2[d] = second ? qa[d] : qb[d];
    }
    const float aa = adt[cell], ab = adt[rr.z];
    float a1 = second ? ab : aa, a2 = second ? aa : ab;
    float r1[4] = {0.f, 0.f, 0.f, 0.f}, r2[4] = {0.f, 0.f, 0.f, 0.f};
    op2_kf::res_calc(x1, x2, q1, q2, &a1, &a2, r1, r2);
    for (int d = 0; d < 4; ++d) r[d] = second ? r2[d] : r1[d];
  }
  static_assert(K == 4, "quad broadcasts assume four lanes per cell");
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  if (k == 0 && valid) ld4r<SOA>(res, cell, sq, acc);
  float v[4][4];
  int hv[4];
  for (int d = 0; d < 4; ++d) {
    v[0][d] = quad_bcast<0>(r[d]);
    v[1][d] = quad_bcast<1>(r[d]);
    v[2][d] = quad_bcast<2>(r[d]);
    v[3][d] = quad_bcast<3>(r[d]);
  }
  hv[0] = quad_bcast<0>(has);
  hv[1] = quad_bcast<1>(has);
  hv[2] = quad_bcast<2>(has);
  hv[3] = quad_bcast<3>(has);
  for (int j = 0; j < 4; ++j)
    if (hv[j])
      for (int d = 0; d < 4; ++d) acc[d] += v[j][d];
  if (k == 0 && valid) st4r<SOA>(res, cell, sq, acc);
}

template <bool SOA>
__device__ __forceinline__ void bres_edge_mixed(const double *__restrict x,
                                                const double *__restrict q,
                                                const float *__restrict adt, int2 bn,
                                                int cell, int bound, int sx, int sq,
                                                float *r) {
  float x1[2], x2[2], q1[4];
  ld2r<SOA>(x, bn.x, sx, x1);
  ld2r<SOA>(x, bn.y, sx, x2);
  ld4r<SOA>(q, cell, sq, q1);
  float a1 = adt[cell];
  for (int d = 0; d < 4; ++d) r[d] = 0.f;
  op2_kf::bres_calc(x1, x2, q1, &a1, r, &bound);
}

template <bool SOA>
__global__ void k_bres_atomic_mixed(const double *__restrict x, const double *__restrict q,
                                    const float *__restrict adt, float *res,
                                    const int2 *__restrict pbedge,
                                    const int *__restrict pbecell,
                                    const int *__restrict bound, int n, int sx, int sq) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  int cell = pbecell[e];
  float r[4];
  bres_edge_mixed<SOA>(x, q, adt, pbedge[e], cell, bound[e], sx, sq, r);
  atomic_add4s<SOA>(res, cell, sq, r);
}

template <bool SOA>
__global__ void k_bres_gather_mixed(const double *__restrict x, const double *__restrict q,
                                    const float *__restrict adt, float *res,
                                    const int2 *__restrict pbedge,
                                    const int *__restrict bound,
                                    const int *__restrict offsets,
                                    const int *__restrict entries,
                                    const int *__restrict targets, int ntargets, int sx,
                                    int sq) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntargets) return;
  int cell = targets[t];
  float acc[4];
  ld4r<SOA>(res, cell, sq, acc);
  for (int k = offsets[t]; k < offsets[t + 1]; ++k) {
    int e = entries[k];
    float r[4];
    bres_edge_mixed<SOA>(x, q, adt, pbedge[e], cell, bound[e], sx, sq, r);
    for (int d = 0; d < 4; ++d) acc[d] += r[d];
  }
  st4r<SOA>(res, cell, sq, acc);
}

}  // namespace

// ===========================================================================
// loop stubs
// ===========================================================================
namespace {

bool loop_soa(const op_arg *args, int nargs, int *stride) {
  int soa = -1;
  *stride = 0;
  for (int m = 0; m < nargs; ++m) {
    const op_arg &a = args[m];
    if (a.argtype != OP_ARG_DAT || !a.opt || a.dat->dim <= 1) continue;
    int s = op2h_dat_soa_stride(a.dat);
    int this_soa = s > 0;
    if (soa >= 0 && this_soa != soa) {
      printf("op2hip: loop mixes AoS and SoA dats; declare all dats of a loop "
             "with the same layout\n");
      exit(-1);
    }
    soa = this_soa;
  }
  return soa == 1;
}

bool is_float(const op_arg &a) { return a.dat && !strncmp(a.dat->type, "float", 5); }

int set_stride(const op_arg &a) {
  int s = op2h_dat_soa_stride(a.dat);
  return s;
}

void account(int kernel_idx, op_set set, int nargs, const op_arg *args) {
  OP_kernels[kernel_idx].transfer += (float)op2h_algorithmic_bytes(set, nargs, args);
}

}  // namespace

// ---------------------------------------------------------------------------
// Loop-chain fusion inside a captured step.  The stubs leave launches pending
// (op2h_defer) and the next stub folds them into its own:
//   - the direct loops of one cell set run per cell in one kernel: an update
//     (and/or a save_soln) is held until the adt_calc that follows and then
//     launched as [update] [save_soln] adt_calc per cell (adt depends on its
//     own cell's q only);
//   - an owner-plan res_calc is held until the bres_calc that follows and
//     both run as one owner launch, each owned cell adding its boundary
//     fluxes after its interior ones;
//   - whole time steps (save_soln, then twice adt_calc, res_calc, bres_calc,
//     update) run as two launches, one per half step (k_half_step), where the
//     owner plan covers every cell and its patches fit their lists.
// Every cell sees the operations of the unfused loops in the same order, and
// the reductions are sums of pairs and extrema that do not depend on how the
// cells are grouped, so every result is the unfused one bit for bit.  Anything
// else launches what is recorded as it was.
// ---------------------------------------------------------------------------
namespace {

// R: the type of res and adt, double, or float in mixed mode (the update in
// FP64 from FP32 res and adt, adt_calc in FP32 from x and q rounded, as
// k_update<float> and k_adt_calc_mixed).
template <class R, bool SOA, bool UPD, bool SAVE>
__global__ void __launch_bounds__(1024)
    k_direct_chain(const double *qold, double *__restrict q, R *__restrict res,
                   R *adt, double *qold_out, const double *__restrict x,
                   const int *__restrict pcell, const uint2 *__restrict prow,
                   const int *__restrict pbase, int n, int s, int sx, UpdateParts parts,
                   const int *__restrict oldidx, int chunk, int res_dead) {
  // qold (read by update, written by save_soln) and adt (read by update,
  // written by adt_calc) are read before they are written, by the same
  // thread for the same cell: not restrict-qualified.  res_dead: the update's
  // zeros in res are not stored (the res_calc that follows in the same step
  // starts its sums from +0.0 instead of reading them)
  constexpr bool MIX = std::is_same<R, float>::value;
  UpdateAcc acc;
  // the update's cells per workgroup (its partials are the update's)
  const CellRange cr = cell_range(n, chunk);
  for (int c = cr.c; c < cr.end; c += cr.step) {
    double qn[4];
    if (UPD) {
      double qo[4], r[4], cs = 0.0;
      const double a = (double)adt[c];
      R rr[4];
      ld4<SOA>(qold, c, s, qo);
      ld4r<SOA>(res, c, s, rr);
      for (int d = 0; d < 4; ++d) r[d] = (double)rr[d];
      const int ci = oldidx ? oldidx[c] : c;
      double mx = -INFINITY;
      int at;
      op2_k::update(qo, qn, r, &a, &cs, &mx, &ci, &at);
      op2h_red::add_cell(acc, cs, mx, ci);
      st4<SOA>(q, c, s, qn);
      if (!res_dead) {
        const R z[4] = {0, 0, 0, 0};
        st4r<SOA>(res, c, s, z);
      }
    } else {
      ld4<SOA>(q, c, s, qn);
    }
    if (SAVE) st4<SOA>(qold_out, c, s, qn);
    int4 cn;
    if (prow) {  // compact rows: four 16-bit offsets from the cell group's base
      const uint2 u = prow[c];
      const int b = pbase[c >> 6];
      cn = make_int4(b + (int)(u.x & 0xFFFFu), b + (int)(u.x >> 16), b + (int)(u.y & 0xFFFFu),
                     b + (int)(u.y >> 16));
    } else {
      cn = reinterpret_cast<const int4 *>(pcell)[c];
    }
    R x1[2], x2[2], x3[2], x4[2], qr[4] = {(R)qn[0], (R)qn[1], (R)qn[2], (R)qn[3]}, a2;
    ld2r<SOA>(x, cn.x, sx, x1);
    ld2r<SOA>(x, cn.y, sx, x2);
    ld2r<SOA>(x, cn.z, sx, x3);
    ld2r<SOA>(x, cn.w, sx, x4);
    if constexpr (MIX)
      op2_kf::adt_calc(x1, x2, x3, x4, qr, &a2);
    else
      op2_k::adt_calc(x1, x2, x3, x4, qr, &a2);
    adt[c] = a2;
  }
  if (UPD) op2h_red::write_partial(acc, parts, cr.L);
}

template <class R, bool SOA>
__global__ void __launch_bounds__(1024)
    k_res_bres_owner(const double *__restrict x, const double *__restrict q,
                     const R *__restrict adt, R *__restrict res, OwnerArgs P, BoundaryArgs B,
                     int sx, int sq, int zero_acc) {
  extern __shared__ double lf[];
  owner_res_bres_block<R, SOA>(xcd_block(kXcds), x, q, adt, res, P, B, sx, sq, (R *)lf,
                               zero_acc != 0);
}

// One half step (op2_dev::half_step_patch) over all patches of the owner
// plan: a grid of workgroups that walk them, with one reduction partial per
// workgroup.
template <class R, bool SOA>
__global__ void __launch_bounds__(1024)
    k_half_step(HalfArgs<R> H, PatchArgs P, BoundaryArgs B, int npatch, int nc, int nn,
                UpdateParts parts) {
  extern __shared__ double lf[];
  UpdateAcc acc;
  for (int b = xcd_block(kXcds); b < npatch; b += gridDim.x) {
    half_step_patch<R, SOA, false>(b, H, P, B, 0, lf, nc, nn, acc);
    __syncthreads();  // the next patch restages the LDS
  }
  op2h_red::write_partial(acc, parts, blockIdx.x);
}

// The boundary edges of each owned cell (at position pos[cell] of the owned
// list, -1: not owned), up to four, in any order.  *bad: an edge of an unowned
// cell, or a fifth of one cell.
__global__ void k_bnd_edges(const int *__restrict becell, int n, const int *__restrict pos,
                            int *__restrict cnt, int4 *slots, int *bad) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int i = pos[becell[e]];
  const int k = i >= 0 ? atomicAdd(&cnt[i], 1) : 4;
  if (k < 4) reinterpret_cast<int *>(slots)[4 * (size_t)i + k] = e;
  else *bad = 1;
}

// Boundary edges of each block's owned cells.
__global__ void __launch_bounds__(256)
    k_bnd_totals(const int *__restrict owned_offs, const int *__restrict cnt,
                 int *__restrict total) {
  __shared__ int s;
  const int b = blockIdx.x;
  if (threadIdx.x == 0) s = 0;
  __syncthreads();
  int n = 0;
  for (int i = owned_offs[b] + threadIdx.x; i < owned_offs[b + 1]; i += 256) n += cnt[i];
  if (n) atomicAdd(&s, n);
  __syncthreads();
  if (threadIdx.x == 0) total[b] = s;
}

// Each owned cell's record: its interior increments (csr4), then its boundary
// edges in order (of `key` when given: the application's) as 0x8000 | j, j
// counting the block's boundary edges in owned order; edges[offs[b] + j] names
// them.  *bad: more than four entries of a cell, or too many j.
__global__ void __launch_bounds__(256)
    k_bnd_records(const int *__restrict owned_offs, const ushort4 *__restrict csr4,
                  const int *__restrict cnt, const int4 *__restrict slots,
                  const int *__restrict key, const int *__restrict offs,
                  ushort4 *__restrict rec, int *__restrict edges, int *bad) {
  __shared__ int part[256];
  const int b = blockIdx.x, t = threadIdx.x;
  const int o0 = owned_offs[b], no = owned_offs[b + 1] - o0;
  const int per = (no + 255) / 256, lo = min(no, t * per), hi = min(no, lo + per);
  int n = 0;
  for (int i = lo; i < hi; ++i) n += cnt[o0 + i];
  part[t] = n;
  __syncthreads();
  int j = 0;
  for (int i = 0; i < t; ++i) j += part[i];
  for (int i = lo; i < hi; ++i) {
    const ushort4 c = csr4[o0 + i];
    unsigned short ent[4] = {c.x, c.y, c.z, c.w};
    const int m = min(cnt[o0 + i], 4);
    if (m) {
      const int4 s4 = slots[o0 + i];
      int e[4] = {s4.x, s4.y, s4.z, s4.w}, k = 0;
      while (k < 4 && ent[k] != 0xFFFF) ++k;
      auto before = [&](int x, int y) { return key ? key[x] < key[y] : x < y; };
      for (int p = 1; p < m; ++p) {
        const int v = e[p];
        int q = p;
        for (; q > 0 && before(v, e[q - 1]); --q) e[q] = e[q - 1];
        e[q] = v;
      }
      for (int p = 0; p < m; ++p, ++j, ++k) {
        if (k >= 4 || j >= 0x7FFF) {
          *bad = 1;
          break;
        }
        ent[k] = (unsigned short)(0x8000 | j);
        edges[offs[b] + j] = e[p];
      }
    }
    rec[o0 + i] = make_ushort4(ent[0], ent[1], ent[2], ent[3]);
  }
}

// Rows of a four-node map as 16-bit offsets from the lowest node of their
// 64-cell group, one wave per group; *wide is set where a group's nodes span
// more than 65535.
__global__ void __launch_bounds__(256)
    k_pack_rows(const int4 *__restrict pcell, int n, uint2 *__restrict rec,
                int *__restrict base, int *wide) {
  const int g = blockIdx.x * 4 + (threadIdx.x >> 6), c = 64 * g + (threadIdx.x & 63);
  if (64 * g >= n) return;  // the whole wave
  const bool in = c < n;
  const int4 r = in ? pcell[c] : make_int4(INT_MAX, INT_MAX, INT_MAX, INT_MAX);
  int lo = min(min(r.x, r.y), min(r.z, r.w));
  int hi = in ? max(max(r.x, r.y), max(r.z, r.w)) : -1;
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o));
    hi = max(hi, __shfl_xor(hi, o));
  }
  if (hi - lo > 0xFFFF) {
    *wide = 1;
    return;
  }
  if ((threadIdx.x & 63) == 0) base[g] = lo;
  if (in)
    rec[c] = make_uint2((unsigned)(r.x - lo) | ((unsigned)(r.y - lo) << 16),
                        (unsigned)(r.z - lo) | ((unsigned)(r.w - lo) << 16));
}

// A pending run of direct loops over one cell set: [update] [save_soln].
// The update's launch shape: g workgroups, one reduction partial each
// (at most 2048, the finish kernels' and the no-allocation scratch's limit).
// Cache-resident data (op2h_streaming false for its 136 bytes per cell): g
// contiguous chunks on XCD-ordered workgroups, of one cell per thread while
// the chip has room for them all (update and finish of 59,000 cells 6.95 us
// against 8.08 with three, 120,000 8.15 against 8.74) and of about three
// beyond, for fewer partials (250,000 cells 10.85 against 10.93, 500,000
// 15.5 against 18.8); streaming data: one cell per thread up to 2048
// workgroups, a grid-stride sweep beyond.  chunk 0 = grid-stride.
struct UpdateShape {
  int g, chunk;
};
constexpr int kUpdateOneEach = 512 * 256;
UpdateShape update_shape(int n, int bs) {
  if (n > 0 && !op2h_streaming((size_t)n * 136)) {
    const int one = grid_for(n, bs);
    const int g = n <= kUpdateOneEach && one <= 4 * op2h_red::kRedThreads
                      ? one
                      : std::max(1, std::min(grid_for(n, 3 * bs), 2048));
    return {g, (n + g - 1) / g};
  }
  return {std::max(1, std::min(grid_for(n, bs), 2048)), 0};
}

// One {hi, lo, max, loc} partial per workgroup in `mem` (g of them).
constexpr size_t kPartBytes = 3 * sizeof(double) + sizeof(int);
UpdateParts update_parts(void *mem, int g) {
  double *d = (double *)mem;
  return UpdateParts{d, d + g, d + 2 * (size_t)g, (int *)(d + 3 * (size_t)g)};
}

// Most workgroups of a half step: the partials one reduction takes.
constexpr int kHalfGrid = op2h_red::kRedThreads * op2h_red::kRedMaxLoads;

struct PendingDirect {
  bool upd = false, save = false, soa = false;
  op_set set = nullptr;
  hipStream_t st = nullptr;
  int n = 0, s = 0;
  // update (its partials handed to the graph's history kernel: up to `cap`)
  int g = 0, bs = 0, chunk = 0, cap = 0;
  bool mixed = false;  // res and adt FP32, else FP64
  const double *qold = nullptr;
  double *q = nullptr;
  void *res = nullptr, *adt = nullptr;
  UpdateParts parts{};
  const int *oldidx = nullptr;
  // save_soln: src -> dst, n2 16-byte vectors when run on its own
  const double *save_src = nullptr;
  double *save_dst = nullptr;
  int save_n2 = 0, save_bs = 256;
};

template <class R>
void launch_update(bool ext, void *e0, void *e1, const PendingDirect &P) {
  launch_k(ext, e0, e1, P.soa ? k_update<R, true> : k_update<R, false>, P.g, P.bs, 0, P.st,
           P.qold, P.q, (R *)P.res, (const R *)P.adt, P.n, P.s, P.parts, P.oldidx, P.chunk);
}

void launch_direct(const PendingDirect &P) {
  if (P.upd) {
    op2h_gbl_partials_used(P.parts.hi, P.g);
    op2h_gbl_partials_used(P.parts.mx, P.g);
    if (P.mixed) launch_update<float>(false, nullptr, nullptr, P);
    else launch_update<double>(false, nullptr, nullptr, P);
  }
  if (P.save)
    launch_k(false, nullptr, nullptr, k_save_soln, grid_for(P.save_n2, P.save_bs), P.save_bs, 0,
             P.st, (const double2 *)P.save_src, (double2 *)P.save_dst, P.save_n2);
}

// A pending fused direct chain ([update] [save_soln] adt_calc per cell).
struct PendingChain {
  bool mixed = false;
  PendingDirect P;
  int g = 0, bs = 0, chunk = 0, n = 0, sq = 0, sx = 0;
  double *q = nullptr;
  void *adt = nullptr;
  const double *x = nullptr;
  const int *pcell = nullptr;
  const uint2 *prow = nullptr;  // compact rows of pcell, or null
  const int *pbase = nullptr;
  hipStream_t st = nullptr;
};

template <class R>
void launch_chain_as(const PendingChain &C, bool res_dead) {
  const PendingDirect &P = C.P;
  auto kern = P.upd ? (P.save ? (P.soa ? k_direct_chain<R, true, true, true> : k_direct_chain<R, false, true, true>)
                              : (P.soa ? k_direct_chain<R, true, true, false> : k_direct_chain<R, false, true, false>))
                    : (P.soa ? k_direct_chain<R, true, false, true> : k_direct_chain<R, false, false, true>);
  launch_k(false, nullptr, nullptr, kern, C.g, C.bs, 0, C.st, P.qold, C.q, (R *)P.res,
           (R *)C.adt, P.save_dst, C.x, C.pcell, C.prow, C.pbase, C.n, C.sq, C.sx, P.parts,
           P.oldidx, C.chunk, (int)(res_dead && P.upd));
}

// res_dead: the update's zeros in res are not stored (the owner res_calc
// launched right after it sums from +0.0 over every cell of the set)
void launch_chain(const PendingChain &C, bool res_dead) {
  if (C.P.upd) {
    op2h_gbl_partials_used(C.P.parts.hi, C.P.g);
    op2h_gbl_partials_used(C.P.parts.mx, C.P.g);
  }
  if (C.mixed) launch_chain_as<float>(C, res_dead);
  else launch_chain_as<double>(C, res_dead);
}

// An owner-plan res_calc.
struct PendingRes {
  bool soa = false, mixed = false;
  hipStream_t st = nullptr;
  const op2h_owner_plan *plan = nullptr;
  unsigned epoch = 0;  // op2h_plan_epoch(): the plan pointer's validity
  OwnerArgs A{};
  const double *x = nullptr, *q = nullptr;
  const void *adt = nullptr;
  void *res = nullptr;
  int sx = 0, sq = 0, bs = 0;
  size_t lds = 0;
  op_map pecell = nullptr;
  op_set cells = nullptr;
  bool zero = false;  // res holds the update's zeros: sums start from +0.0
};

template <class R>
void launch_res_as(bool ext, void *e0, void *e1, const PendingRes &P) {
  if (P.plan->nblocks)
    launch_k(ext, e0, e1,
             P.A.csr4 ? (P.soa ? k_res_owner<R, true, true> : k_res_owner<R, false, true>)
                      : (P.soa ? k_res_owner<R, true, false> : k_res_owner<R, false, false>),
             P.plan->nblocks, P.bs, P.lds, P.st, P.x, P.q, (const R *)P.adt, (R *)P.res, P.A,
             P.sx, P.sq, (int)P.zero);
}

void launch_res(bool ext, void *e0, void *e1, const PendingRes &P) {
  if (P.mixed) launch_res_as<float>(ext, e0, e1, P);
  else launch_res_as<double>(ext, e0, e1, P);
}

template <class R>
void launch_res_bres_as(const PendingRes &P, const BoundaryArgs &B) {
  if (P.plan->nblocks)
    launch_k(false, nullptr, nullptr, P.soa ? k_res_bres_owner<R, true> : k_res_bres_owner<R, false>,
             P.plan->nblocks, P.bs, P.lds, P.st, P.x, P.q, (const R *)P.adt, (R *)P.res, P.A, B,
             P.sx, P.sq, (int)P.zero);
}

// The captured loops not launched yet.  Nothing runs while a graph is being
// captured, so the stubs only record what they would launch and the whole run
// of loops is launched when something else comes (or the capture ends), with
// every following loop known: g_halves, the complete [chain] res_calc
// bres_calc groups; then at most one of g_direct ([update] [save_soln]),
// g_chain (the same with the adt_calc that follows) or g_chain with g_res.
struct Half {
  bool chained = false;  // C precedes R
  PendingChain C;
  PendingRes R;
  BoundaryArgs B{};
};
std::vector<Half> g_halves;
PendingDirect g_direct;
PendingChain g_chain;
bool g_res_chained = false;  // g_chain precedes g_res
PendingRes g_res;
PendingRes g_last_res;  // the latest owner-plan res_calc, pending or not

// Device memory of the fused half steps for one owner plan and its dats: the
// other copies of q and adt and the patches' lists (allocated before
// a capture starts, for the latest owner-plan res_calc).
struct HalfMem {
  unsigned epoch = 0;
  const op2h_owner_plan *plan = nullptr;
  const double *q = nullptr;
  bool mixed = false;
  const int *pcell = nullptr;
  const ushort4 *rec = nullptr;  // the boundary records the lists hold
  double *q2 = nullptr;
  void *adt2 = nullptr;
  PatchArgs patches{};
  int nc = 0, nn = 0;
};
HalfMem g_half_mem;
unsigned long long g_half_steps = 0;  // k_half_step launches

// Whether halves h and k (with the direct loops D that follow k, and its
// adt_calc C if that follows too) are one time step of the form
//   save_soln adt_calc res_calc bres_calc update
//             adt_calc res_calc bres_calc update [save_soln] [adt_calc]
// on the same dats, which two k_half_step launches run.
bool is_step(const Half &h, const Half &k, const PendingDirect *D, const PendingChain *C) {
  const HalfMem &M = g_half_mem;
  const PendingRes &R = h.R;
  if (!h.chained || !k.chained || !D || !D->upd || M.epoch != op2h_plan_epoch() ||
      R.epoch != M.epoch || M.plan != R.plan || M.q != R.q || M.mixed != R.mixed ||
      M.pcell != h.C.pcell || M.rec != h.B.rec)
    return false;
  const op2h_owner_plan *p = R.plan;
  if (!p->nblocks || p->n_owned != R.cells->size || p->max_owned > R.bs) return false;
  const PendingRes &S = k.R;
  if (S.plan != p || S.x != R.x || S.q != R.q || S.adt != R.adt || S.res != R.res ||
      S.mixed != R.mixed || S.soa != R.soa || S.sx != R.sx || S.sq != R.sq || S.bs != R.bs ||
      S.st != R.st || k.B.rec != h.B.rec || k.B.pbedge != h.B.pbedge || k.B.bound != h.B.bound)
    return false;
  auto chain_fits = [&](const PendingChain &c) {
    return c.q == R.q && c.adt == R.adt && c.x == R.x && c.mixed == R.mixed &&
           c.P.soa == R.soa && c.n == R.cells->size && c.pcell == h.C.pcell && c.st == R.st;
  };
  const PendingDirect &A = h.C.P, &U = k.C.P;
  auto update_fits = [&](const PendingDirect &d) {
    return d.upd && d.q == R.q && d.qold == A.save_dst && d.res == R.res && d.adt == R.adt &&
           d.mixed == R.mixed && d.soa == R.soa && d.set == R.cells && d.st == R.st &&
           d.cap >= 1 && d.oldidx == U.oldidx;
  };
  return A.save && A.save_src == R.q && A.save_dst != R.q && chain_fits(h.C) &&
         chain_fits(k.C) && (!C || chain_fits(*C)) && update_fits(U) && !U.save &&
         update_fits(*D) && (!D->save || (D->save_src == R.q && D->save_dst == A.save_dst));
}

template <class R>
void launch_half_as(const Half &h, const HalfArgs<R> &H, const PendingDirect &D) {
  const PendingRes &P = h.R;
  const HalfMem &M = g_half_mem;
  auto kern = P.soa ? k_half_step<R, true> : k_half_step<R, false>;
  const size_t lds = patch_lds_bytes<R>(M.nc, M.nn);
  // as many workgroups as the GPU holds at once, each walking the same number
  // of patches: 126 us at 2.88 million cells with the 4 per CU that fit,
  // 159 with 5 and 140 with 6 per CU (a second, nearly empty round), 125 with a
  // quarter of the patches each; nothing in it at 720,000 (34 to 35 us)
  int resident = 0, cus = 0, dev = 0;
  KCHECK(hipGetDevice(&dev));
  KCHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  KCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&resident, (const void *)kern, P.bs, lds));
  const int npatch = P.plan->nblocks;
  const int rounds = (npatch + std::max(1, resident * cus) - 1) / std::max(1, resident * cus);
  const int grid = std::min((npatch + rounds - 1) / rounds, D.cap);
  op2h_gbl_partials_used(D.parts.hi, grid);
  op2h_gbl_partials_used(D.parts.mx, grid);
  launch_k(false, nullptr, nullptr, kern, grid, P.bs, lds, P.st, H, M.patches, h.B, npatch, M.nc,
           M.nn, D.parts);
  ++g_half_steps;
}

// The time step of halves h and k as two launches (is_step holds).  D: the
// second update; adt: an adt_calc follows it; dead_save: the next time step is
// run the same way, so nothing reads the copy of q that D's save_soln would
// make, nor was this step's own copy made when saved is false.  res holds zeros
// in memory where h.R.zero says so (the update before zeroed this very res).
template <class R>
void launch_step_as(const Half &h, const Half &k, const PendingDirect &D, bool adt,
                    bool dead_save, bool saved) {
  const HalfMem &M = g_half_mem;
  double *q = const_cast<double *>(h.R.q), *qold = h.C.P.save_dst;
  R *a = (R *)const_cast<void *>(h.R.adt), *a2 = (R *)M.adt2;
  HalfArgs<R> H;
  H.x = h.R.x;
  H.q = q;
  H.adt = a;
  H.res = (R *)h.R.res;
  H.qold = nullptr;  // the step's first q, which save_soln copies: q itself
  H.q_out = M.q2;
  H.adt_out = a2;
  H.qold_out = qold;
  H.oldidx = k.C.P.oldidx;
  H.sx = h.R.sx;
  H.sq = h.R.sq;
  H.flags = kHalfAdt | (h.R.zero ? 0 : kHalfReadRes | kHalfZeroRes);
  launch_half_as<R>(h, H, k.C.P);
  H.q = M.q2;
  H.adt = a2;
  H.qold = q;
  H.q_out = q;
  H.adt_out = a;
  H.flags = (adt ? kHalfAdt : kHalfCopyAdt) |
            (D.save ? (dead_save ? 0 : kHalfSaveNew) : (saved ? 0 : kHalfSaveOld));
  launch_half_as<R>(k, H, D);
}

// Launches everything recorded, in order: time steps as pairs of half steps,
// other loops as direct chains and res_calc + bres_calc.
void launch_recorded(bool direct, bool chain, bool res) {
  const std::vector<Half> hs = std::move(g_halves);
  g_halves.clear();
  const PendingDirect D = g_direct;
  const PendingChain C = g_chain;
  const int n = (int)hs.size();
  const bool tail_chain = chain || (res && g_res_chained);
  // what follows half i: its update's record, and the chain's when adt_calc does too
  auto follows = [&](int i, const PendingDirect **d, const PendingChain **c) {
    *c = i + 1 < n ? (hs[i + 1].chained ? &hs[i + 1].C : nullptr) : tail_chain ? &C : nullptr;
    *d = *c ? &(*c)->P : (i + 1 == n && direct) ? &D : nullptr;
  };
  auto step_at = [&](int i) {
    if (i + 1 >= n) return false;
    const PendingDirect *d;
    const PendingChain *c;
    follows(i + 1, &d, &c);
    return is_step(hs[i], hs[i + 1], d, c);
  };
  bool folded = false;   // the chain or update after the last launch is part of it
  bool saved = true;     // qold holds the copy of q that half i's chain makes
  for (int i = 0; i < n;) {
    if (step_at(i)) {
      if (!folded) launch_chain(hs[i].C, false);
      const PendingDirect *d;
      const PendingChain *c;
      follows(i + 1, &d, &c);
      const bool dead = c && d->save && step_at(i + 2);
      if (hs[i].R.mixed) launch_step_as<float>(hs[i], hs[i + 1], *d, c, dead, saved);
      else launch_step_as<double>(hs[i], hs[i + 1], *d, c, dead, saved);
      folded = true;
      saved = !dead;
      i += 2;
    } else {
      if (hs[i].chained && !folded) launch_chain(hs[i].C, hs[i].R.zero);
      if (hs[i].R.mixed) launch_res_bres_as<float>(hs[i].R, hs[i].B);
      else launch_res_bres_as<double>(hs[i].R, hs[i].B);
      folded = false;
      saved = true;
      ++i;
    }
  }
  if (direct && !folded) launch_direct(D);
  if (tail_chain && !folded) launch_chain(C, res && g_res.zero);
  if (res) launch_res(false, nullptr, nullptr, g_res);
  g_direct = PendingDirect();
  g_chain = PendingChain();
  g_res_chained = false;
  g_res = PendingRes();
  KCHECK(hipGetLastError());
}

void flush_direct(void *) { launch_recorded(true, false, false); }
void flush_chain(void *) { launch_recorded(false, true, false); }
void flush_res(void *) { launch_recorded(false, false, true); }
void flush_halves(void *) { launch_recorded(false, false, false); }

// The fused res_calc + bres_calc records for an owner plan and the boundary
// map (bedge -> cell), built on the device once per plan: each owned cell's
// interior increments, then its boundary edges (ascending; under transparent
// renumbering in the application's order).  Null when a cell has more than
// four increments in all, the local ids do not fit 15 bits, or the device has
// no room to build them.
struct BoundaryRec {
  unsigned epoch = 0;  // op2h_plan_epoch() when built
  bool ok = false;
  BoundaryArgs B{};
};

// `build` false: only a record built before (inside a capture nothing may
// be allocated or uploaded).
const BoundaryArgs *boundary_args(const op2h_owner_plan *p, op_map pbecell, op_map pbedge,
                                  op_dat bound, hipStream_t st, bool build) {
  static std::map<std::pair<const void *, int>, BoundaryRec> cache;
  auto key = std::make_pair((const void *)p, pbecell->index);
  auto it = cache.find(key);
  if (it != cache.end() && it->second.epoch == op2h_plan_epoch()) {
    if (!it->second.ok) return nullptr;
    it->second.B.bound = (const int *)bound->data_d;
    it->second.B.pbedge = (const int2 *)pbedge->map_d;
    return &it->second.B;
  }
  if (!build) return nullptr;
  BoundaryRec &slot = cache[key];
  slot = BoundaryRec();
  slot.epoch = op2h_plan_epoch();
  if (!p->csr4 || pbecell->dim != 1 || (long long)p->max_elems * p->ninc >= 0x8000) return nullptr;
  const int nb = p->nblocks, no = p->n_owned, ncell = p->to_size;
  const int nbe = pbecell->from->size;
  if (!nb) return nullptr;
  char name[96];
  snprintf(name, sizeof name, "res_bres.fused.%p.%d", (const void *)p, pbecell->index);
  const size_t b_rec = ((size_t)8 * std::max(no, 1) + 255) / 256 * 256;
  const size_t b_offs = ((size_t)4 * (nb + 1) + 255) / 256 * 256;
  int fresh = 0;
  char *buf = (char *)op2h_plan_user(name, b_rec + b_offs + 4 * (size_t)std::max(nbe, 1), &fresh);
  // scratch: each owned cell's boundary edges and their number, each cell's
  // position, each block's number, the flag
  const size_t b_slots = (size_t)16 * no, b_cnt = (size_t)4 * no, b_pos = (size_t)4 * ncell;
  char *tmp = (char *)op2h_extra_alloc(b_slots + b_cnt + b_pos + 4 * (size_t)nb + 4);
  if (!tmp) return nullptr;
  int4 *slots = (int4 *)tmp;
  int *cnt = (int *)(tmp + b_slots), *pos = (int *)(tmp + b_slots + b_cnt);
  int *total = (int *)(tmp + b_slots + b_cnt + b_pos), *bad = total + nb;
  KCHECK(hipMemsetAsync(cnt, 0, b_cnt, st));
  KCHECK(hipMemsetAsync(pos, 0xFF, b_pos, st));
  KCHECK(hipMemsetAsync(bad, 0, 4, st));
  k_patch_pos<<<grid_for(no, 256), 256, 0, st>>>(p->owned, no, pos);
  if (nbe)
    k_bnd_edges<<<grid_for(nbe, 256), 256, 0, st>>>(pbecell->map_d, nbe, pos, cnt, slots, bad);
  k_bnd_totals<<<nb, 256, 0, st>>>(p->owned_offs, cnt, total);
  std::vector<int> offs((size_t)nb + 1, 0);
  KCHECK(hipMemcpyAsync(offs.data() + 1, total, 4 * (size_t)nb, hipMemcpyDeviceToHost, st));
  KCHECK(hipStreamSynchronize(st));
  for (int b = 0; b < nb; ++b) offs[b + 1] += offs[b];
  KCHECK(hipMemcpyAsync(buf + b_rec, offs.data(), 4 * ((size_t)nb + 1), hipMemcpyHostToDevice, st));
  k_bnd_records<<<nb, 256, 0, st>>>(p->owned_offs, (const ushort4 *)p->csr4, cnt, slots,
                                    op2h_set_old_index(pbecell->from), (const int *)(buf + b_rec),
                                    (ushort4 *)buf, (int *)(buf + b_rec + b_offs), bad);
  KCHECK(hipGetLastError());
  int failed = 0;
  KCHECK(hipMemcpyAsync(&failed, bad, 4, hipMemcpyDeviceToHost, st));
  KCHECK(hipStreamSynchronize(st));
  KCHECK(hipFree(tmp));
  if (failed) return nullptr;
  BoundaryArgs &B = slot.B;
  B.rec = (const ushort4 *)buf;
  B.offs = (const int *)(buf + b_rec);
  B.edges = (const int *)(buf + b_rec + b_offs);
  B.pbedge = (const int2 *)pbedge->map_d;
  B.bound = (const int *)bound->data_d;
  slot.ok = true;
  return &B;
}

// Compact rows of a four-node map (cells -> nodes) for the fused direct
// chain: per cell its nodes as 16-bit offsets from the lowest node of its
// 64-cell group, 8 bytes instead of 16, where every group's nodes lie within
// 65535 of that base (a locally numbered mesh; else null).  Packed on the
// device when a capture starts: only captured chains read them, and nothing
// may be allocated once it has started.
struct CompactRows {
  unsigned epoch = 0;
  const int *map = nullptr;
  const uint2 *rec = nullptr;  // null: the rows do not fit
  const int *base = nullptr;
};
CompactRows g_rows;
struct {
  unsigned epoch = 0;
  op_map map = nullptr;
  hipStream_t st = nullptr;
} g_last_pcell;  // the latest adt_calc's
struct {
  unsigned epoch = 0;
  const op2h_owner_plan *plan = nullptr;
  const ushort4 *rec = nullptr;
} g_last_bres;  // the latest fused res_calc + bres_calc records built

const CompactRows *compact_rows(op_map m) {
  return g_rows.epoch == op2h_plan_epoch() && g_rows.map == m->map_d && g_rows.rec ? &g_rows
                                                                                    : nullptr;
}

void pack_compact_rows(op_map m, hipStream_t st) {
  if (g_rows.epoch == op2h_plan_epoch() && g_rows.map == m->map_d) return;
  g_rows = CompactRows();
  g_rows.epoch = op2h_plan_epoch();
  g_rows.map = m->map_d;
  const int n = m->from->size, ng = (n + 63) / 64;
  if (m->dim != 4 || n < 1) return;
  char name[64];
  snprintf(name, sizeof name, "compact_rows.%d", m->index);
  const size_t b_rec = (8 * (size_t)n + 255) / 256 * 256;
  const size_t b_base = (4 * (size_t)ng + 255) / 256 * 256;
  int fresh = 0;
  char *buf = (char *)op2h_plan_user(name, b_rec + b_base + 4, &fresh);
  int *wide = (int *)(buf + b_rec + b_base);
  const int zero = 0;
  int any = 0;
  KCHECK(hipMemcpyAsync(wide, &zero, sizeof zero, hipMemcpyHostToDevice, st));
  k_pack_rows<<<grid_for(ng, 4), 256, 0, st>>>((const int4 *)m->map_d, n, (uint2 *)buf,
                                               (int *)(buf + b_rec), wide);
  KCHECK(hipMemcpyAsync(&any, wide, sizeof any, hipMemcpyDeviceToHost, st));
  KCHECK(hipStreamSynchronize(st));
  if (any) return;
  g_rows.rec = (const uint2 *)buf;
  g_rows.base = (const int *)(buf + b_rec);
}

// The memory of the fused half steps, for the latest owner-plan res_calc and
// the latest adt_calc's map when they are over the same cells, and the device
// has room (about 66 bytes a cell).
void make_half_mem() {
  const PendingRes &R = g_last_res;
  const op_map pcell = g_last_pcell.map;
  const unsigned now = op2h_plan_epoch();
  g_half_mem = HalfMem();
  if (!R.plan || R.epoch != now || g_last_pcell.epoch != now || !pcell ||
      pcell->from != R.cells || pcell->dim != 4 || !R.plan->csr4 || !R.plan->nblocks ||
      R.plan->n_owned != R.cells->size || R.plan->max_owned > R.bs)
    return;
  const op2h_owner_plan *p = R.plan;
  if (g_last_bres.epoch != now || g_last_bres.plan != p) return;
  char name[96];
  int fresh = 0, part = 0;
  HalfMem M;
  if (!build_patches(
          R.A, p->nblocks, g_last_bres.rec, (const int4 *)pcell->map_d, R.cells->size, R.st,
          [&](size_t bytes) {
            snprintf(name, sizeof name, "half_step.lists%d.%p", part++, (const void *)p);
            return op2h_extra_plan_user(name, bytes, &fresh);
          },
          &M.patches, &M.nc, &M.nn) ||
      (R.mixed ? patch_lds_bytes<float>(M.nc, M.nn) : patch_lds_bytes<double>(M.nc, M.nn)) >
          kPatchLds)
    return;
  const size_t rows = (size_t)(R.soa ? R.cells->stride : R.cells->size);
  const size_t b_q = 4 * sizeof(double) * rows;
  snprintf(name, sizeof name, "half_step.q.%p", (const void *)p);
  M.q2 = (double *)op2h_extra_plan_user(
      name, b_q + (R.mixed ? sizeof(float) : sizeof(double)) * rows, &fresh);
  if (!M.q2) return;
  M.adt2 = (char *)M.q2 + b_q;
  M.epoch = now;
  M.plan = p;
  M.q = R.q;
  M.mixed = R.mixed;
  M.pcell = pcell->map_d;
  M.rec = g_last_bres.rec;
  g_half_mem = M;
}

void before_capture() {
  if (g_last_pcell.map && g_last_pcell.epoch == op2h_plan_epoch())
    pack_compact_rows(g_last_pcell.map, g_last_pcell.st);
  make_half_mem();
}

const struct CaptureHook {
  CaptureHook() { op2h_register_capture_hook(before_capture); }
} g_capture_hook;

}  // namespace

extern "C" unsigned long long op2h_half_step_count(void) { return g_half_steps; }

extern "C" void op_par_loop_airfoil_1_save_soln(char const *name, op_set set,
                                                op_arg arg0, op_arg arg1) {
  op_arg args[2] = {arg0, arg1};
  op2h_loop_ctx ctx;
  op2h_accept_deferred("direct_chain");
  op2h_loop_begin(&ctx, 0, name, set, 2, args, OP2H_PLAN_ATOMIC, 256);
  hipStream_t st = (hipStream_t)ctx.stream;
  const bool fuse = op2h_fusion_enabled() != 0;
  bool held = op2h_take_deferred("direct_chain", nullptr) != 0;
  if (held && !fuse) {  // launched first, in its place in the order
    flush_direct(nullptr);
    held = false;
  }
  if (set->size > 0) {
    int stride = 0;
    bool soa = loop_soa(args, 2, &stride);
    // identical layouts: the copy covers the whole device allocation
    long long ndouble = soa ? 4LL * set->stride : 4LL * set->size;
    int n2 = (int)(ndouble / 2);
    PendingDirect &P = g_direct;
    if (held && !(P.upd && !P.save && P.set == set && P.soa == soa &&
                  P.q == (double *)args[0].data_d)) {
      flush_direct(nullptr);  // not the update this copy follows
      held = false;
    }
    if (fuse) {  // held for the adt_calc that follows
      if (!held) {
        P = PendingDirect();
        P.set = set;
        P.soa = soa;
        P.st = st;
        P.n = set->size;
        P.s = soa ? set->stride : 0;
      }
      P.save = true;
      P.save_src = (const double *)args[0].data_d;
      P.save_dst = (double *)args[1].data_d;
      P.save_n2 = n2;
      P.save_bs = ctx.block_size;
      op2h_defer("direct_chain", flush_direct, nullptr);
      account(0, set, 2, args);
      op2h_loop_end(&ctx);
      return;
    }
    LoopTimer tm(&ctx);
    launch_k(tm.ext, tm.e0, tm.e1, k_save_soln, grid_for(n2, ctx.block_size), ctx.block_size,
             0, st, (const double2 *)args[0].data_d, (double2 *)args[1].data_d, n2);
    tm.done();
    KCHECK(hipGetLastError());
  } else if (held) {
    flush_direct(nullptr);
  }
  account(0, set, 2, args);
  op2h_loop_end(&ctx);
}

extern "C" void op_par_loop_airfoil_2_adt_calc(char const *name, op_set set,
                                               op_arg arg0, op_arg arg1,
                                               op_arg arg2, op_arg arg3,
                                               op_arg arg4, op_arg arg5) {
  op_arg args[6] = {arg0, arg1, arg2, arg3, arg4, arg5};
  op2h_loop_ctx ctx;
  op2h_accept_deferred("direct_chain");
  op2h_loop_begin(&ctx, 1, name, set, 6, args, OP2H_PLAN_ATOMIC, 256);
  hipStream_t st = (hipStream_t)ctx.stream;
  bool held = op2h_take_deferred("direct_chain", nullptr) != 0;
  if (held && !op2h_fusion_enabled()) {
    flush_direct(nullptr);
    held = false;
  }
  if (set->size > 0) {
    int dummy;
    bool soa = loop_soa(args, 6, &dummy);
    int sx = set_stride(args[0]), sq = set_stride(args[4]);
    const double *x = (const double *)args[0].data_d;
    const double *q = (const double *)args[4].data_d;
    double *adt = (double *)args[5].data_d;
    const int *pcell = args[0].map->map_d;
    int g = grid_for(set->size, ctx.block_size);
    if (held) {
      PendingDirect P = g_direct;
      const double *qsrc = P.upd ? P.q : P.save_src;
      const bool mixed = is_float(args[5]);
      if (P.set == set && P.soa == soa && (soa ? sq == P.s : true) && qsrc == q &&
          (!P.upd || (P.mixed == mixed && P.adt == args[5].data_d))) {
        g_direct = PendingDirect();
        // [update] [save_soln] adt_calc per cell: the update's launch shape
        // (its partials), else adt_calc's
        const int gg = P.upd ? P.g : g, bb = P.upd ? P.bs : ctx.block_size;
        const int chunk = P.upd ? P.chunk : 0;
        PendingChain &C = g_chain;
        C = PendingChain();
        C.P = P;
        C.g = gg;
        C.bs = bb;
        C.chunk = chunk;
        C.q = P.q ? P.q : (double *)q;
        C.mixed = mixed;
        C.adt = args[5].data_d;
        C.x = x;
        C.pcell = pcell;
        if (const CompactRows *cr = compact_rows(args[0].map)) {
          C.prow = cr->rec;
          C.pbase = cr->base;
        }
        C.n = set->size;
        C.sq = sq;
        C.sx = sx;
        C.st = st;
        // held for the res_calc that follows, which may take the update's
        // zeros in res as known (launched as it is by anything else)
        op2h_defer("chain", flush_chain, nullptr);
        account(1, set, 6, args);
        op2h_loop_end(&ctx);
        return;
      }
      flush_direct(nullptr);
    }
    g_last_pcell.epoch = op2h_plan_epoch();
    g_last_pcell.map = args[0].map;
    g_last_pcell.st = st;
    LoopTimer tm(&ctx);
    if (is_float(args[5])) {
      float *adtf = (float *)args[5].data_d;
      launch_k(tm.ext, tm.e0, tm.e1, soa ? k_adt_calc_mixed<true> : k_adt_calc_mixed<false>, g,
               ctx.block_size, 0, st, x, q, adtf, pcell, set->size, sx, sq);
    } else {
      // streams: pcell rows, q and adt
      const bool nt = op2h_streaming((size_t)set->size * 56) != 0;
      launch_k(tm.ext, tm.e0, tm.e1,
               nt ? (soa ? k_adt_calc<true, true> : k_adt_calc<false, true>)
                  : (soa ? k_adt_calc<true, false> : k_adt_calc<false, false>),
               g, ctx.block_size, 0, st, x, q, adt, pcell, set->size, sx, sq);
    }
    tm.done();
    KCHECK(hipGetLastError());
  } else if (held) {
    flush_direct(nullptr);
  }
  account(1, set, 6, args);
  op2h_loop_end(&ctx);
}

extern "C" void op_par_loop_airfoil_3_res_calc(char const *name, op_set set,
                                               op_arg arg0, op_arg arg1,
                                               op_arg arg2, op_arg arg3,
                                               op_arg arg4, op_arg arg5,
                                               op_arg arg6, op_arg arg7) {
  op_arg args[8] = {arg0, arg1, arg2, arg3, arg4, arg5, arg6, arg7};
  op2h_loop_ctx ctx;
  op2h_accept_deferred("chain");
  op2h_loop_begin(&ctx, 2, name, set, 8, args, OP2H_PLAN_STAGED, 256);
  hipStream_t st = (hipStream_t)ctx.stream;
  // a fused direct chain held for this loop: launched with it, with or
  // without the update's zeros in res (only an owner plan covering every
  // cell can take them as known)
  bool chain = op2h_take_deferred("chain", nullptr) != 0;
  if (chain && (!op2h_fusion_enabled() || set->size == 0 || ctx.plan != OP2H_PLAN_OWNER)) {
    flush_chain(nullptr);
    chain = false;
  }
  if (set->size > 0) {
    int dummy;
    bool soa = loop_soa(args, 8, &dummy);
    int sx = set_stride(args[0]), sq = set_stride(args[2]);
    const double *x = (const double *)args[0].data_d;
    const double *q = (const double *)args[2].data_d;
    const double *adt = (const double *)args[4].data_d;
    double *res = (double *)args[6].data_d;
    const int2 *pedge = (const int2 *)args[0].map->map_d;
    const int2 *pecell = (const int2 *)args[2].map->map_d;
    const int bs = ctx.block_size;
    const bool mixed = is_float(args[6]);
    if (mixed != is_float(args[4])) {
      printf("op2hip: res_calc needs adt and res both FP32 (mixed mode) or both FP64\n");
      exit(-1);
    }
    if (ctx.plan == OP2H_PLAN_OWNER) {
      ctx.part_size = bs;
      const op2h_owner_plan *p = op2h_plan_owner_local(&ctx);
      PendingRes R;
      R.A = owner_args_res(p, args, st);
      R.lds = (mixed ? sizeof(float) : sizeof(double)) * 4 * (size_t)R.A.max_e;
      if (R.lds > 160 * 1024) {
        printf("op2hip: res_calc owner plan needs %zu bytes of LDS; use a smaller block\n",
               R.lds);
        exit(-1);
      }
      R.soa = soa;
      R.mixed = mixed;
      R.st = st;
      R.plan = p;
      R.epoch = op2h_plan_epoch();
      R.x = x;
      R.q = q;
      R.adt = args[4].data_d;
      R.res = args[6].data_d;
      R.sx = sx;
      R.sq = sq;
      R.bs = bs;
      R.pecell = args[6].map;
      R.cells = args[6].dat->set;
      // res is dead between the chain's update (which sets every cell's res
      // to +0.0) and this loop when the plan owns every cell: the zeros are
      // neither stored nor read
      R.zero = chain && g_chain.P.upd && g_chain.P.mixed == mixed && g_chain.P.res == R.res &&
               p->n_owned == R.cells->size;
      g_last_res = R;
      if (op2h_fusion_enabled()) {  // held for the bres_calc that follows
        g_res = R;
        g_res_chained = chain;
        op2h_defer("res_owner", flush_res, nullptr);
      } else {
        LoopTimer tm(&ctx);
        launch_res(tm.ext, tm.e0, tm.e1, R);
        tm.done();
      }
      KCHECK(hipGetLastError());
      account(2, set, 8, args);
      op2h_loop_end(&ctx);
      return;
    }
    if (mixed) {
      // mixed precision: atomic plan, else the gather plan
      const float *adtf = (const float *)args[4].data_d;
      float *resf = (float *)args[6].data_d;
      op2h_kernel_timer_start(&ctx);
      if (ctx.plan == OP2H_PLAN_ATOMIC) {
        int g = grid_for(set->size, bs);
        if (soa) k_res_atomic_mixed<true><<<g, bs, 0, st>>>(x, q, adtf, resf, pedge, pecell, set->size, sx, sq);
        else k_res_atomic_mixed<false><<<g, bs, 0, st>>>(x, q, adtf, resf, pedge, pecell, set->size, sx, sq);
      } else {
        const op2h_gather_plan *p = op2h_plan_gather(args[6].map);
        if (p->max_count > 4) {
          printf("op2hip: mixed-precision res_calc supports at most 4 edges per cell\n");
          exit(-1);
        }
        char key[96];
        snprintf(key, sizeof key, "res_calc.gather4.%d.%d", args[0].map->index,
                 args[2].map->index);
        int fresh = 0;
        int4 *rec = (int4 *)op2h_plan_user(key, sizeof(int4) * 4 * (size_t)p->ntargets, &fresh);
        if (fresh)
          k_pack_res_gather<4><<<grid_for(4 * (long long)p->ntargets, 256), 256, 0, st>>>(
              pedge, pecell, p->offsets, p->entries, p->ntargets, rec);
        int g = grid_for(4 * (long long)p->ntargets, bs);
        if (soa) k_res_gather_packed_mixed<true, 4><<<g, bs, 0, st>>>(x, q, adtf, resf, rec, p->targets, p->ntargets, sx, sq);
        else k_res_gather_packed_mixed<false, 4><<<g, bs, 0, st>>>(x, q, adtf, resf, rec, p->targets, p->ntargets, sx, sq);
      }
      op2h_kernel_timer_stop(&ctx);
      KCHECK(hipGetLastError());
      account(2, set, 8, args);
      op2h_loop_end(&ctx);
      return;
    }
    switch (ctx.plan) {
      case OP2H_PLAN_ATOMIC: {
        op2h_kernel_timer_start(&ctx);
        int g = grid_for(set->size, bs);
        if (soa) k_res_atomic<true><<<g, bs, 0, st>>>(x, q, adt, res, pedge, pecell, set->size, sx, sq);
        else k_res_atomic<false><<<g, bs, 0, st>>>(x, q, adt, res, pedge, pecell, set->size, sx, sq);
        op2h_kernel_timer_stop(&ctx);
        break;
      }
      case OP2H_PLAN_COLOR: {
        const op2h_color_plan *p = op2h_plan_color(&ctx);
        op2h_kernel_timer_start(&ctx);
        for (int c = 0; c < p->ncolors; ++c) {
          int s0 = p->col_offsets_h[c], s1 = p->col_offsets_h[c + 1];
          int g = grid_for(s1 - s0, bs);
          if (!g) continue;
          if (soa) k_res_color<true><<<g, bs, 0, st>>>(x, q, adt, res, pedge, pecell, p->col_reord, s0, s1, sx, sq);
          else k_res_color<false><<<g, bs, 0, st>>>(x, q, adt, res, pedge, pecell, p->col_reord, s0, s1, sx, sq);
        }
        op2h_kernel_timer_stop(&ctx);
        break;
      }
      case OP2H_PLAN_GATHER: {
        const op2h_gather_plan *p = op2h_plan_gather(args[6].map);
        LoopTimer tm(&ctx);
        if (p->max_count <= 4) {
          // packed per-(cell, edge) records, built once per plan
          char key[96];
          snprintf(key, sizeof key, "res_calc.gather4.%d.%d", args[0].map->index,
                   args[2].map->index);
          int fresh = 0;
          int4 *rec = (int4 *)op2h_plan_user(key, sizeof(int4) * 4 * (size_t)p->ntargets, &fresh);
          if (fresh)
            k_pack_res_gather<4><<<grid_for(4 * (long long)p->ntargets, 256), 256, 0, st>>>(
                pedge, pecell, p->offsets, p->entries, p->ntargets, rec);
          int g = grid_for(4 * (long long)p->ntargets, bs);
          launch_k(tm.ext, tm.e0, tm.e1,
                   soa ? k_res_gather_packed<true, 4> : k_res_gather_packed<false, 4>, g, bs, 0,
                   st, x, q, adt, res, rec, p->targets, p->ntargets, sx, sq);
        } else if (p->max_count <= 8) {
          if (tm.ext) KCHECK(hipEventRecord((hipEvent_t)tm.e0, st));
          int g = grid_for(8 * (long long)p->ntargets, bs);
          if (soa) k_res_gather_lanes<true, 8><<<g, bs, 0, st>>>(x, q, adt, res, pedge, pecell, p->offsets, p->entries, p->targets, p->ntargets, sx, sq);
          else k_res_gather_lanes<false, 8><<<g, bs, 0, st>>>(x, q, adt, res, pedge, pecell, p->offsets, p->entries, p->targets, p->ntargets, sx, sq);
        } else {
          if (tm.ext) KCHECK(hipEventRecord((hipEvent_t)tm.e0, st));
          int g = grid_for(p->ntargets, bs);
          if (soa) k_res_gather<true><<<g, bs, 0, st>>>(x, q, adt, res, pedge, pecell, p->offsets, p->entries, p->targets, p->ntargets, sx, sq);
          else k_res_gather<false><<<g, bs, 0, st>>>(x, q, adt, res, pedge, pecell, p->offsets, p->entries, p->targets, p->ntargets, sx, sq);
        }
        if (tm.ext && p->max_count > 4) KCHECK(hipEventRecord((hipEvent_t)tm.e1, st));
        tm.done();
        break;
      }
      default: {  // STAGED
        ctx.part_size = bs;
        const op2h_staged_plan *p = op2h_plan_staged(&ctx);
        int sn = p->map_of_arg[0], sc = p->map_of_arg[2];
        StagedArgs A;
        A.blkmap = p->blkmap;
        A.offset = p->offset;
        A.nelems = p->nelems;
        A.nthrcol = p->nthrcol;
        A.thrcol = p->thrcol;
        A.ind_offs_n = p->ind_offs[sn];
        A.ind_sizes_n = p->ind_sizes[sn];
        A.ind_map_n = p->ind_map[sn];
        A.ind_offs_c = p->ind_offs[sc];
        A.ind_sizes_c = p->ind_sizes[sc];
        A.ind_map_c = p->ind_map[sc];
        A.loc_n0 = p->loc_map[p->loc_of_arg[0]];
        A.loc_n1 = p->loc_map[p->loc_of_arg[1]];
        A.loc_c0 = p->loc_map[p->loc_of_arg[2]];
        A.loc_c1 = p->loc_map[p->loc_of_arg[3]];
        A.max_n = p->max_ind_h[sn];
        A.max_c = p->max_ind_h[sc];
        size_t lds = sizeof(double) * (2 * (size_t)A.max_n + 9 * (size_t)A.max_c);
        if (lds > 160 * 1024) {
          printf("op2hip: res_calc staged plan needs %zu bytes of LDS\n", lds);
          exit(-1);
        }
        op2h_kernel_timer_start(&ctx);
        for (int c = 0; c < p->ncolors; ++c) {
          int nb = p->ncolblk_h[c];
          if (!nb) continue;
          if (soa) k_res_staged<true><<<nb, bs, lds, st>>>(x, q, adt, res, A, p->colstart_h[c], sx, sq);
          else k_res_staged<false><<<nb, bs, lds, st>>>(x, q, adt, res, A, p->colstart_h[c], sx, sq);
        }
        op2h_kernel_timer_stop(&ctx);
        break;
      }
    }
    KCHECK(hipGetLastError());
  }
  account(2, set, 8, args);
  op2h_loop_end(&ctx);
}

extern "C" void op_par_loop_airfoil_4_bres_calc(char const *name, op_set set,
                                                op_arg arg0, op_arg arg1,
                                                op_arg arg2, op_arg arg3,
                                                op_arg arg4, op_arg arg5) {
  op_arg args[6] = {arg0, arg1, arg2, arg3, arg4, arg5};
  op2h_loop_ctx ctx;
  op2h_accept_deferred("res_owner");
  op2h_loop_begin(&ctx, 3, name, set, 6, args, OP2H_PLAN_STAGED, 256);
  hipStream_t st = (hipStream_t)ctx.stream;
  bool held = op2h_take_deferred("res_owner", nullptr) != 0;
  if (held && !op2h_fusion_enabled()) {
    flush_res(nullptr);
    held = false;
  }
  if (set->size > 0) {
    int dummy;
    bool soa = loop_soa(args, 6, &dummy);
    int sx = set_stride(args[0]), sq = set_stride(args[2]);
    const double *x = (const double *)args[0].data_d;
    const double *q = (const double *)args[2].data_d;
    const double *adt = (const double *)args[3].data_d;
    double *res = (double *)args[4].data_d;
    const int *bound = (const int *)args[5].data_d;
    const int2 *pbedge = (const int2 *)args[0].map->map_d;
    const int *pbecell = args[2].map->map_d;
    const int bs = ctx.block_size;
    // the res_calc this loop follows, on the same dats: the two as one owner
    // launch (inside a capture), its boundary records built beforehand
    const PendingRes &L = held ? g_res : g_last_res;
    const bool same = L.plan && L.epoch == op2h_plan_epoch() && L.x == x && L.q == q &&
                      L.adt == args[3].data_d && L.res == args[4].data_d && L.soa == soa &&
                      L.sx == sx && L.sq == sq && L.mixed == is_float(args[4]) &&
                      args[2].map->to == L.pecell->to && args[4].map == args[2].map;
    const BoundaryArgs *B = same ? boundary_args(L.plan, args[2].map, args[0].map, args[5].dat,
                                                 st, !ctx.capturing)
                                 : nullptr;
    if (B && !ctx.capturing) {
      g_last_bres.epoch = op2h_plan_epoch();
      g_last_bres.plan = L.plan;
      g_last_bres.rec = B->rec;
    }
    if (held) {
      if (B) {
        Half h;
        h.chained = g_res_chained;
        if (h.chained) h.C = g_chain;
        h.R = g_res;
        h.B = *B;
        g_halves.push_back(h);
        g_chain = PendingChain();
        g_res = PendingRes();
        g_res_chained = false;
        op2h_defer("halves", flush_halves, nullptr);  // held for the update
        account(3, set, 6, args);
        op2h_loop_end(&ctx);
        return;
      }
      flush_res(nullptr);
    }
    if (is_float(args[4])) {
      const float *adtf = (const float *)args[3].data_d;
      float *resf = (float *)args[4].data_d;
      op2h_kernel_timer_start(&ctx);
      if (ctx.plan == OP2H_PLAN_ATOMIC) {
        int g = grid_for(set->size, bs);
        if (soa) k_bres_atomic_mixed<true><<<g, bs, 0, st>>>(x, q, adtf, resf, pbedge, pbecell, bound, set->size, sx, sq);
        else k_bres_atomic_mixed<false><<<g, bs, 0, st>>>(x, q, adtf, resf, pbedge, pbecell, bound, set->size, sx, sq);
      } else {
        const op2h_gather_plan *p = op2h_plan_gather(args[4].map);
        int g = grid_for(p->ntargets, bs);
        if (soa) k_bres_gather_mixed<true><<<g, bs, 0, st>>>(x, q, adtf, resf, pbedge, bound, p->offsets, p->entries, p->targets, p->ntargets, sx, sq);
        else k_bres_gather_mixed<false><<<g, bs, 0, st>>>(x, q, adtf, resf, pbedge, bound, p->offsets, p->entries, p->targets, p->ntargets, sx, sq);
      }
      op2h_kernel_timer_stop(&ctx);
      KCHECK(hipGetLastError());
      account(3, set, 6, args);
      op2h_loop_end(&ctx);
      return;
    }
    switch (ctx.plan) {
      case OP2H_PLAN_ATOMIC: {
        LoopTimer tm(&ctx);
        int g = grid_for(set->size, bs);
        launch_k(tm.ext, tm.e0, tm.e1, soa ? k_bres_atomic<true> : k_bres_atomic<false>, g, bs,
                 0, st, x, q, adt, res, pbedge, pbecell, bound, set->size, sx, sq);
        tm.done();
        break;
      }
      case OP2H_PLAN_COLOR: {
        const op2h_color_plan *p = op2h_plan_color(&ctx);
        op2h_kernel_timer_start(&ctx);
        for (int c = 0; c < p->ncolors; ++c) {
          int s0 = p->col_offsets_h[c], s1 = p->col_offsets_h[c + 1];
          int g = grid_for(s1 - s0, bs);
          if (!g) continue;
          if (soa) k_bres_color<true><<<g, bs, 0, st>>>(x, q, adt, res, pbedge, pbecell, bound, p->col_reord, s0, s1, sx, sq);
          else k_bres_color<false><<<g, bs, 0, st>>>(x, q, adt, res, pbedge, pbecell, bound, p->col_reord, s0, s1, sx, sq);
        }
        op2h_kernel_timer_stop(&ctx);
        break;
      }
      // One increment per boundary edge: an owner partition would evaluate
      // each edge once in its cell's block, which is what the gather plan does.
      case OP2H_PLAN_OWNER:
      case OP2H_PLAN_GATHER: {
        const op2h_gather_plan *p = op2h_plan_gather(args[4].map);
        op2h_kernel_timer_start(&ctx);
        int g = grid_for(p->ntargets, bs);
        if (soa) k_bres_gather<true><<<g, bs, 0, st>>>(x, q, adt, res, pbedge, bound, p->offsets, p->entries, p->targets, p->ntargets, sx, sq);
        else k_bres_gather<false><<<g, bs, 0, st>>>(x, q, adt, res, pbedge, bound, p->offsets, p->entries, p->targets, p->ntargets, sx, sq);
        op2h_kernel_timer_stop(&ctx);
        break;
      }
      default: {  // STAGED
        ctx.part_size = bs;
        const op2h_staged_plan *p = op2h_plan_staged(&ctx);
        int sn = p->map_of_arg[0], sc = p->map_of_arg[2];
        BStagedArgs A;
        A.blkmap = p->blkmap;
        A.offset = p->offset;
        A.nelems = p->nelems;
        A.nthrcol = p->nthrcol;
        A.thrcol = p->thrcol;
        A.ind_offs_n = p->ind_offs[sn];
        A.ind_sizes_n = p->ind_sizes[sn];
        A.ind_map_n = p->ind_map[sn];
        A.ind_offs_c = p->ind_offs[sc];
        A.ind_sizes_c = p->ind_sizes[sc];
        A.ind_map_c = p->ind_map[sc];
        A.loc_n0 = p->loc_map[p->loc_of_arg[0]];
        A.loc_n1 = p->loc_map[p->loc_of_arg[1]];
        A.loc_c0 = p->loc_map[p->loc_of_arg[2]];
        A.max_n = p->max_ind_h[sn];
        A.max_c = p->max_ind_h[sc];
        size_t lds = sizeof(double) * (2 * (size_t)A.max_n + 9 * (size_t)A.max_c);
        if (lds > 160 * 1024) {
          printf("op2hip: bres_calc staged plan needs %zu bytes of LDS\n", lds);
          exit(-1);
        }
        op2h_kernel_timer_start(&ctx);
        for (int c = 0; c < p->ncolors; ++c) {
          int nb = p->ncolblk_h[c];
          if (!nb) continue;
          if (soa) k_bres_staged<true><<<nb, bs, lds, st>>>(x, q, adt, res, bound, A, p->colstart_h[c], sx, sq);
          else k_bres_staged<false><<<nb, bs, lds, st>>>(x, q, adt, res, bound, A, p->colstart_h[c], sx, sq);
        }
        op2h_kernel_timer_stop(&ctx);
        break;
      }
    }
    KCHECK(hipGetLastError());
  } else if (held) {
    flush_res(nullptr);
  }
  account(3, set, 6, args);
  op2h_loop_end(&ctx);
}

extern "C" void op_par_loop_airfoil_5_update(char const *name, op_set set,
                                             op_arg arg0, op_arg arg1,
                                             op_arg arg2, op_arg arg3,
                                             op_arg arg4, op_arg arg5,
                                             op_arg arg6, op_arg arg7) {
  op_arg args[8] = {arg0, arg1, arg2, arg3, arg4, arg5, arg6, arg7};
  op2h_loop_ctx ctx;
  op2h_accept_deferred("halves");
  op2h_loop_begin(&ctx, 4, name, set, 8, args, OP2H_PLAN_ATOMIC, 256);
  hipStream_t st = (hipStream_t)ctx.stream;
  int dummy;
  bool soa = loop_soa(args, 8, &dummy);
  int s = set_stride(args[0]);
  const int bs = ctx.block_size;
  const UpdateShape shape = update_shape(set->size, bs);
  const int g = shape.g;
  // res_calc + bres_calc recorded before this update, if any
  const bool held = op2h_take_deferred("halves", nullptr) != 0;
  if (held && (!op2h_fusion_enabled() || set->size == 0)) flush_halves(nullptr);
  // inside a captured graph the partials go to the runtime, whose history
  // kernel finishes both reductions of every update of the step in one pass
  // (same tree as k_update_finish); otherwise finish them here.  Where the
  // update may run inside a half step there is room for its blocks' partials.
  const int cap = g_halves.empty()
                      ? g
                      : std::max(g, std::min(g_halves.back().R.plan->nblocks, kHalfGrid));
  double *slot_rms = nullptr, *slot_max = nullptr;
  UpdateParts parts{};
  const bool deferred = op2h_gbl_partials2(&ctx, 4, cap, &parts.hi, &parts.lo) != 0;
  if (deferred && !op2h_gbl_partials(&ctx, 5, 7, cap, &parts.mx, &parts.loc)) {
    printf("op2hip: update: maxerr/errloc cannot be deferred with rms\n");
    exit(-1);
  }
  if (!deferred) {
    if (!g_halves.empty()) flush_halves(nullptr);
    slot_rms = (double *)op2h_gbl_result(&ctx, 4, -1);
    slot_max = (double *)op2h_gbl_result(&ctx, 5, 7);
    parts = update_parts(op2h_reduct_scratch((size_t)g * kPartBytes), g);
  }
  if (is_float(args[2]) != is_float(args[3])) {
    printf("op2hip: update needs res and adt both FP32 (mixed mode) or both FP64\n");
    exit(-1);
  }
  if (deferred && op2h_fusion_enabled() && set->size > 0) {
    // held for the save_soln / adt_calc that follow (its partials are
    // finished by the graph's history kernel either way)
    PendingDirect &P = g_direct;
    P = PendingDirect();
    P.upd = true;
    P.mixed = is_float(args[2]);
    P.set = set;
    P.soa = soa;
    P.st = st;
    P.n = set->size;
    P.s = s;
    P.g = g;
    P.bs = bs;
    P.chunk = shape.chunk;
    P.qold = (const double *)args[0].data_d;
    P.q = (double *)args[1].data_d;
    P.res = args[2].data_d;
    P.adt = args[3].data_d;
    P.cap = cap;
    P.parts = parts;
    P.oldidx = op2h_set_old_index(set);
    op2h_defer("direct_chain", flush_direct, nullptr);
    account(4, set, 8, args);
    op2h_loop_end(&ctx);
    return;
  }
  if (deferred) {  // on its own inside a capture
    if (!g_halves.empty()) flush_halves(nullptr);
    op2h_gbl_partials_used(parts.hi, g);
    op2h_gbl_partials_used(parts.mx, g);
  }
  LoopTimer tm(&ctx);
  PendingDirect U;
  U.soa = soa;
  U.st = st;
  U.n = set->size;
  U.s = s;
  U.g = g;
  U.bs = bs;
  U.chunk = shape.chunk;
  U.qold = (const double *)args[0].data_d;
  U.q = (double *)args[1].data_d;
  U.res = args[2].data_d;
  U.adt = args[3].data_d;
  U.parts = parts;
  U.oldidx = op2h_set_old_index(set);
  if (is_float(args[2])) launch_update<float>(tm.ext, tm.e0, nullptr, U);
  else launch_update<double>(tm.ext, tm.e0, nullptr, U);
  if (!deferred)
    launch_k(tm.ext, nullptr, tm.e1, k_update_finish, 1, kFinishThreads, 0, st, parts, g,
             slot_rms, slot_max);
  tm.done();
  KCHECK(hipGetLastError());
  account(4, set, 8, args);
  op2h_loop_end(&ctx);
}

// ---------------------------------------------------------------------------
// The update loop on caller-owned device arrays without allocating: the same
// kernels as op_par_loop_airfoil_5_update (same workgroup count for a block
// size, so the same reduction tree and the same bits), with the per-workgroup
// partials in a file-scope device array instead of runtime-allocated memory.
// For callers that cannot allocate device memory (code under HIP graph
// capture, serving loops, harnesses that forbid it).  Every call on one device
// shares that device's array: calls that overlap on one device race.
// ---------------------------------------------------------------------------
namespace {
constexpr int kNoAllocMaxParts = 2048;  // the stub's workgroup cap
constexpr size_t kNoAllocScratchBytes = (size_t)kNoAllocMaxParts * kPartBytes;  // 56 KiB
constexpr int kNoAllocMaxDevices = 64;
void *g_scratch_addr[kNoAllocMaxDevices];  // device address of `scratch`, per device
}  // namespace

static __device__ __align__(256) char scratch[kNoAllocScratchBytes];

extern "C" int op2h_update_noalloc(int ncell, int soa_stride, int block, const double *qold,
                                   double *q, double *res, const double *adt,
                                   op2h_update_result *result, void *stream) {
  if (ncell < 0 || block < 64 || block > 1024 || block % 64 != 0 || !result ||
      (ncell > 0 && (!qold || !q || !res || !adt)) ||
      (soa_stride != 0 && soa_stride < ncell)) {
    printf("op2h_update_noalloc: bad arguments (ncell %d, soa_stride %d, block %d)\n", ncell,
           soa_stride, block);
    return -1;
  }
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kNoAllocMaxDevices) {
    printf("op2h_update_noalloc: no usable current device\n");
    return -2;
  }
  if (!g_scratch_addr[dev]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      printf("op2h_update_noalloc: hipGetSymbolAddress failed: %s\n", hipGetErrorString(e));
      return -2;
    }
    g_scratch_addr[dev] = ptr;
  }
  const UpdateShape shape = update_shape(ncell, block);  // the stub's
  const int g = shape.g;
  if ((size_t)g * kPartBytes > kNoAllocScratchBytes) {
    printf("op2h_update_noalloc: %d partials exceed the %zu-byte scratch\n", g,
           kNoAllocScratchBytes);
    return -3;
  }
  const UpdateParts parts = update_parts(g_scratch_addr[dev], g);
  hipStream_t st = (hipStream_t)stream;
  // every partial the finish kernel reads is written by this call's k_update
  if (soa_stride)
    k_update<double, true><<<g, block, 0, st>>>(qold, q, res, adt, ncell, soa_stride, parts,
                                                nullptr, shape.chunk);
  else
    k_update<double, false><<<g, block, 0, st>>>(qold, q, res, adt, ncell, 0, parts, nullptr,
                                                 shape.chunk);
  k_update_finish<<<1, kFinishThreads, 0, st>>>(parts, g, &result->rms, &result->maxerr);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    printf("op2h_update_noalloc: launch failed: %s\n", hipGetErrorString(e));
    return -4;
  }
  return 0;
}
