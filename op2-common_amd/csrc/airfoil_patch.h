// Half time steps of the airfoil application in one launch: res_calc,
// bres_calc, update and the adt_calc that follows (with the save_soln in
// between), per owner-compute patch of cells, shared by the single-mesh
// captured steps (airfoil_kernels.hip) and the ensemble (ensemble.hip).
//
// What a half step writes (q and adt) goes to other arrays than the ones its
// neighbours still read: the first half of a step reads q, adt and writes
// q_out, adt_out; the second half the other way round, its update reading the
// step's first q (qold) from the array it overwrites, each cell its own.  res
// stays in registers, and the step's copy of q (save_soln) is that array
// itself.  Per cell it moves 128 bytes in a step's first half and 162 in the
// second at 720,000 cells (counted), where a direct chain and a res_calc +
// bres_calc launch move 280-315.
// Measured, one half step against the mean of those launches it replaces:
// 30.4 against 44.0 us at 720,000 cells (FP64, 256-cell patches), 110 against
// 173 at 2.88 million, 99 against 144 in mixed mode there, and 6.4 against 11.7
// at 7,200 cells; 108 MB a launch at 720,000 cells, 3.65 TB/s, 2,156 MB at 11.5
// million, 4.6 TB/s.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>
#include <cstdio>
#include <cstdlib>

#include "airfoil_device.h"

namespace op2_dev {

// The patches' lists.  A patch stages its owned cells (in owned order, so
// owned cell i is local cell i and thread i's) and then the other cells their
// edges touch, and the corner nodes of its owned cells.
struct PatchArgs {
  const int4 *head;            // per patch: lowest cell, lowest node, cells, nodes staged
  const unsigned short *cells; // [patch][cstride] offsets from the lowest cell
  const unsigned short *nodes; // [patch][nstride] offsets from the lowest node
  // per owned cell, in owned order: up to four increments in the sequential
  // order (entry below), and its corners' local nodes, 16 bits each
  const uint2 *edges, *corners;
  const int *owned_offs;
  int cstride, nstride;
};

// An increment: the other cell's local number (12 bits), the edge's first
// corner k of the cell (its nodes are corners k and k + 1 mod 4: 2 bits),
// whether the edge lists them the other way round, whether the cell is the
// edge's second; boundary edges and absent increments have numbers no local
// cell has.
constexpr int kEntryBits = 12;
constexpr unsigned kEntryMask = (1u << kEntryBits) - 1;
constexpr unsigned kEntryBoundary = 0xE00;  // + index among the patch's boundary edges
constexpr unsigned kEntryNone = 0xFFF;
constexpr int kPatchMaxNodes = 2048, kPatchMaxHalo = 1024;  // list building, per patch

enum HalfFlags {
  kHalfReadRes = 1,   // sums start from res (else from +0.0)
  kHalfZeroRes = 2,   // the update's zeros are stored to res
  kHalfAdt = 4,       // adt_calc of the new q to adt_out
  kHalfCopyAdt = 8,   // no adt_calc follows: adt_out = adt
  kHalfSaveOld = 16,  // qold_out = the update's qold (no save_soln follows)
  kHalfSaveNew = 32,  // qold_out = the new q (a save_soln follows)
};

template <class R>
struct HalfArgs {
  const double *x, *q;
  const R *adt;
  R *res;
  const double *qold;  // null: q itself; may be q_out (each thread reads its cell first)
  double *q_out, *qold_out;
  R *adt_out;
  const int *oldidx;  // op_arg_idx: the application's index of a cell, or null
  int sx, sq, flags;
};

// LDS of a patch with nc staged cells and nn nodes, as arrays of pairs: per
// cell {q0, q1}, {q2, q3}, {ri, p} and adt, per node x.  Neighbouring lanes
// mostly read neighbouring cells, so one 16-byte read per lane from consecutive
// pairs meets no bank twice; rows of four doubles would at every other lane.
template <class R>
struct PatchLds {
  using P2 = typename std::conditional<std::is_same<R, float>::value, float2, double2>::type;
  P2 *qa, *qb, *rp, *x;
  R *adt;
  __device__ PatchLds(void *mem, int nc, int nn)
      : qa((P2 *)mem), qb(qa + nc), rp(qb + nc), x(rp + nc), adt((R *)(x + nn)) {}
};
template <class R>
constexpr size_t patch_lds_bytes(int nc, int nn) {
  return sizeof(R) * (7 * (size_t)nc + 2 * (size_t)nn);
}

// Patches up to the LDS of a CU run as half steps: also where only one of them
// fits there at once they are faster than the loops they stand for.  1024-cell
// patches (83 KiB in FP64, 42 in mixed mode), a step: 75 us against 92 at
// 720,000 cells, 257 against 358 at 2.88 million, 207 against 294 mixed there;
// 111 against 152 for an ensemble of 16 members, 1.1 million cells.
constexpr size_t kPatchLds = 160 * 1024;

template <class R>
__device__ __forceinline__ R airfoil_eps() {
  if constexpr (std::is_same<R, float>::value) return eps_f;
  else return eps_d;
}
__device__ __forceinline__ void cell_terms(const double *q, double *ri, double *p) {
  op2_k::cell_terms(q, ri, p);
}
__device__ __forceinline__ void cell_terms(const float *q, float *ri, float *p) {
  op2_kf::cell_terms(q, ri, p);
}

// Stages local cell j of the patch: q and what res_calc computes of the cell
// alone.
template <class R>
__device__ __forceinline__ void stage_cell(const PatchLds<R> &L, int j, const double *qd, R a) {
  using P2 = typename PatchLds<R>::P2;
  const R q[4] = {(R)qd[0], (R)qd[1], (R)qd[2], (R)qd[3]};
  R ri, p;
  cell_terms(q, &ri, &p);
  L.qa[j] = P2{q[0], q[1]};
  L.qb[j] = P2{q[2], q[3]};
  L.rp[j] = P2{ri, p};
  L.adt[j] = a;
}

// Patch b's half step; blockDim.x >= its owned cells.  Bound by memory
// latency and then FP64 issue: the lists and then the rows they name are the
// only dependent global loads, each issued for all of a thread's cells and
// nodes before the first is waited for; everything else a cell needs comes
// from LDS.  Each cell adds its own edges' fluxes (an edge inside the patch is
// evaluated by both its cells: the two divisions a flux holds belong to the
// cells and are done once per staged cell, which leaves 54 operations a side,
// less than passing the flux through LDS and another barrier), in edge order
// and from both sides with res_flux's bits, so the results are the sequential
// executor's.  105 VGPRs, 4 waves per SIMD; capped to 5 or 6 waves it was
// slower (30.4, 30.4, 32.5 us at 720k cells), reading the next patch's lists
// ahead of the arithmetic changed nothing.  idx0: subtracted from the cell for the reductions' element
// index (an ensemble member's first cell).  QI: boundary edges with their
// member's free stream.
template <class R, bool SOA, bool QI>
__device__ __forceinline__ void half_step_patch(int b, const HalfArgs<R> &H, const PatchArgs &P,
                                                const BoundaryArgs &B, int idx0, void *mem,
                                                int nc_lds, int nn_lds,
                                                op2h_red::UpdateAcc &acc) {
  using P2 = typename PatchLds<R>::P2;
  const PatchLds<R> L(mem, nc_lds, nn_lds);
  const int4 head = P.head[b];
  const int o0 = P.owned_offs[b], no = P.owned_offs[b + 1] - o0;
  const int t = threadIdx.x, bs = blockDim.x;
  const bool mine = t < no;
  const unsigned short *cl = P.cells + (size_t)b * P.cstride;
  const unsigned short *nl = P.nodes + (size_t)b * P.nstride;
  // the lists: this thread's first two cells (the first its own when mine)
  // and nodes; lanes past the end take the patch's first
  const bool c_in[2] = {t < head.z, t + bs < head.z}, n_in[2] = {t < head.w, t + bs < head.w};
  int cell[2], node[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    cell[k] = cl[c_in[k] ? t + k * bs : 0];
    node[k] = nl[n_in[k] ? t + k * bs : 0];
  }
  uint2 ent = make_uint2(0u, 0u), cor = make_uint2(0u, 0u);
  if (mine) {
    ent = P.edges[o0 + t];
    cor = P.corners[o0 + t];
  }
  // their rows
  double qd[2][4], qo[4] = {0.0, 0.0, 0.0, 0.0};
  R ad[2], xd[2][2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    cell[k] += head.x;
    ld4<SOA>(H.q, cell[k], H.sq, qd[k]);
    ad[k] = H.adt[cell[k]];
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) ld2r<SOA>(H.x, head.y + node[k], H.sx, xd[k]);
  if (H.qold && mine) ld4<SOA>(H.qold, cell[0], H.sq, qo);
  if (!H.qold)
    for (int d = 0; d < 4; ++d) qo[d] = qd[0][d];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (c_in[k]) stage_cell<R>(L, t + k * bs, qd[k], ad[k]);
    if (n_in[k]) L.x[t + k * bs] = P2{xd[k][0], xd[k][1]};
  }
  for (int j = t + 2 * bs; j < head.z; j += bs) {
    const int c = head.x + cl[j];
    double qj[4];
    ld4<SOA>(H.q, c, H.sq, qj);
    stage_cell<R>(L, j, qj, H.adt[c]);
  }
  for (int j = t + 2 * bs; j < head.w; j += bs) {
    R xj[2];
    ld2r<SOA>(H.x, head.y + nl[j], H.sx, xj);
    L.x[j] = P2{xj[0], xj[1]};
  }
  __syncthreads();
  if (!mine) return;
  const int c = cell[0];
  R r[4] = {0, 0, 0, 0};
  if (H.flags & kHalfReadRes) ld4r<SOA>(H.res, c, H.sq, r);
  const unsigned long long corners = ((unsigned long long)cor.y << 32) | cor.x;
  unsigned long long es = ((unsigned long long)ent.y << 32) | ent.x;
#pragma unroll
  for (int k = 0; k < 4; ++k, es >>= 16) {
    const unsigned e = (unsigned)es & 0xFFFFu, id = e & kEntryMask;
    if (id < kEntryBoundary) {
      const unsigned c0 = (e >> kEntryBits) & 3u, swap = (e >> (kEntryBits + 2)) & 1u;
      const unsigned na = (unsigned)(corners >> (16 * ((c0 + swap) & 3u))) & 0xFFFFu;
      const unsigned nb = (unsigned)(corners >> (16 * ((c0 + 1u - swap) & 3u))) & 0xFFFFu;
      // the edge's two cells in its own order
      const bool second = (e >> 15) != 0;
      const unsigned i1 = second ? id : (unsigned)t, i2 = second ? (unsigned)t : id;
      const P2 xa = L.x[na], xb = L.x[nb], a1 = L.qa[i1], b1 = L.qb[i1], t1 = L.rp[i1],
               a2 = L.qa[i2], b2 = L.qb[i2], t2 = L.rp[i2];
      const R q1[4] = {a1.x, a1.y, b1.x, b1.y}, q2[4] = {a2.x, a2.y, b2.x, b2.y};
      op2_k::add_flux<R>(xa.x - xb.x, xa.y - xb.y, q1, t1.x, t1.y, q2, t2.x, t2.y,
                         L.adt[i1] + L.adt[i2], second, airfoil_eps<R>(), r);
    } else if (id != kEntryNone) {
      const int be = B.edges[B.offs[b] + (int)(id - kEntryBoundary)];
      const int2 bn = B.pbedge[be];
      const P2 qa = L.qa[t], qb = L.qb[t];
      const R q1[4] = {qa.x, qa.y, qb.x, qb.y}, a = L.adt[t];
      R xa[2], xb[2];
      ld2r<SOA>(H.x, bn.x, H.sx, xa);
      ld2r<SOA>(H.x, bn.y, H.sx, xb);
      const int bnd = B.bound[be];
      if constexpr (std::is_same<R, float>::value)
        op2_kf::bres_calc(xa, xb, q1, &a, r, &bnd);
      else if constexpr (QI)
        op2_k::bres_calc_q(xa, xb, q1, &a, r, &bnd, B.qinf + 4 * (size_t)B.bmesh[be]);
      else
        op2_k::bres_calc(xa, xb, q1, &a, r, &bnd);
    }
  }
  double qn[4], rd[4] = {(double)r[0], (double)r[1], (double)r[2], (double)r[3]};
  const R a = L.adt[t];
  const double da = (double)a;
  double cs = 0.0;
  const int idx = H.oldidx ? H.oldidx[c] : c - idx0;
  double mx = -INFINITY;
  int at;
  op2_k::update(qo, qn, rd, &da, &cs, &mx, &idx, &at);
  op2h_red::add_cell(acc, cs, mx, idx);
  st4<SOA>(H.q_out, c, H.sq, qn);
  if (H.flags & (kHalfZeroRes | kHalfCopyAdt | kHalfSaveOld | kHalfSaveNew)) {
    const R z[4] = {0, 0, 0, 0};
    if (H.flags & kHalfZeroRes) st4r<SOA>(H.res, c, H.sq, z);
    if (H.flags & kHalfCopyAdt) H.adt_out[c] = a;
    if (H.flags & kHalfSaveOld) st4<SOA>(H.qold_out, c, H.sq, qo);
    if (H.flags & kHalfSaveNew) st4<SOA>(H.qold_out, c, H.sq, qn);
  }
  if (H.flags & kHalfAdt) {
    const R qr[4] = {(R)qn[0], (R)qn[1], (R)qn[2], (R)qn[3]};
    const P2 v0 = L.x[cor.x & 0xFFFFu], v1 = L.x[cor.x >> 16], v2 = L.x[cor.y & 0xFFFFu],
             v3 = L.x[cor.y >> 16];
    const R x1[2] = {v0.x, v0.y}, x2[2] = {v1.x, v1.y}, x3[2] = {v2.x, v2.y}, x4[2] = {v3.x, v3.y};
    R an;
    if constexpr (std::is_same<R, float>::value)
      op2_kf::adt_calc(x1, x2, x3, x4, qr, &an);
    else
      op2_k::adt_calc(x1, x2, x3, x4, qr, &an);
    H.adt_out[c] = an;
  }
}

// ---- building the lists, one workgroup per patch ----

// An open-addressed set of ints in LDS with an insertion list.
struct LdsSet {
  int *tab, *list, *n;
  int size, cap;  // table size (a power of two), list capacity
  // False: full (the caller reports the patch as unfit).
  __device__ bool insert(int key) {
    unsigned h = ((unsigned)key * 2654435761u) & (size - 1);
    for (int probe = 0; probe < size; ++probe, h = (h + 1) & (size - 1)) {
      const int old = atomicCAS(&tab[h], -1, key);
      if (old == key) return true;
      if (old == -1) {
        const int at = atomicAdd(n, 1);
        if (at < cap) list[at] = key;
        return at < cap;
      }
    }
    return false;
  }
  __device__ int find(int key) const {
    unsigned h = ((unsigned)key * 2654435761u) & (size - 1);
    for (int probe = 0; probe < size; ++probe, h = (h + 1) & (size - 1))
      if (tab[h] == key) return (int)h;
    return -1;
  }
};

// position of each owned cell in the owned list
static __global__ void k_patch_pos(const int *__restrict owned, int n, int *__restrict pos) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) pos[owned[i]] = i;
}

// info: [0] most cells of a patch, [1] most nodes, [2] 1 when some patch does
// not fit (an edge whose nodes are not consecutive corners of its cell, spans
// over 65535, too many cells or boundary edges).  FILL false: counts only.
template <bool FILL>
static __global__ void __launch_bounds__(256)
    k_patch_lists(const int4 *__restrict inst, const int *__restrict elem_offs,
                  const int *__restrict owned_offs, const int *__restrict owned,
                  const int *__restrict pos, const ushort4 *__restrict rec,
                  const int4 *__restrict pcell, int *info, int4 *__restrict head,
                  unsigned short *__restrict cells, unsigned short *__restrict nodes,
                  uint2 *__restrict edges, uint2 *__restrict corners, int cstride,
                  int nstride) {
  __shared__ int tab_c[2 * kPatchMaxHalo], list_c[kPatchMaxHalo];
  __shared__ int tab_n[2 * kPatchMaxNodes], list_n[kPatchMaxNodes];
  __shared__ unsigned short id_c[2 * kPatchMaxHalo], id_n[2 * kPatchMaxNodes];
  __shared__ int cnt[2], lo[2], hi[2], bad;
  const int b = blockIdx.x, t = threadIdx.x;
  const int e0 = elem_offs[b], e1 = elem_offs[b + 1], o0 = owned_offs[b], o1 = owned_offs[b + 1];
  const int no = o1 - o0;
  for (int i = t; i < 2 * kPatchMaxHalo; i += 256) tab_c[i] = -1;
  for (int i = t; i < 2 * kPatchMaxNodes; i += 256) tab_n[i] = -1;
  if (t < 2) {
    cnt[t] = 0;
    lo[t] = INT_MAX;
    hi[t] = -1;
  }
  if (t == 0) bad = 0;
  __syncthreads();
  LdsSet C{tab_c, list_c, &cnt[0], 2 * kPatchMaxHalo, kPatchMaxHalo};
  LdsSet N{tab_n, list_n, &cnt[1], 2 * kPatchMaxNodes, kPatchMaxNodes};
  bool ok = true;
  int cmin = INT_MAX, cmax = -1, nmin = INT_MAX, nmax = -1;
  for (int j = e0 + t; j < e1; j += 256) {
    const int c[2] = {inst[j].z, inst[j].w};
    for (int k = 0; k < 2; ++k) {
      const int p = pos[c[k]];
      if (p < o0 || p >= o1) {
        ok &= C.insert(c[k]);
        cmin = min(cmin, c[k]);
        cmax = max(cmax, c[k]);
      }
    }
  }
  for (int i = o0 + t; i < o1; i += 256) {
    const int c = owned[i];
    const int4 r = pcell[c];
    cmin = min(cmin, c);
    cmax = max(cmax, c);
    const int n[4] = {r.x, r.y, r.z, r.w};
    for (int k = 0; k < 4; ++k) {
      ok &= N.insert(n[k]);
      nmin = min(nmin, n[k]);
      nmax = max(nmax, n[k]);
    }
  }
  atomicMin(&lo[0], cmin);
  atomicMin(&lo[1], nmin);
  atomicMax(&hi[0], cmax);
  atomicMax(&hi[1], nmax);
  if (!ok) bad = 1;
  __syncthreads();
  const int nh = min(cnt[0], kPatchMaxHalo), nn = min(cnt[1], kPatchMaxNodes);
  const int c0 = lo[0], n0 = lo[1];
  if (t == 0) {
    if (hi[0] - c0 > 0xFFFF || hi[1] - n0 > 0xFFFF || no + nh > (int)kEntryBoundary) bad = 1;
    if (bad) info[2] = 1;
    if (!FILL) {
      atomicMax(&info[0], no + nh);
      atomicMax(&info[1], nn);
    }
  }
  __syncthreads();
  if (!FILL || bad) return;
  // the sets in ascending order: each item's rank
  for (int i = t; i < nh; i += 256) {
    const int v = list_c[i];
    int rank = 0;
    for (int k = 0; k < nh; ++k) rank += list_c[k] < v;
    id_c[C.find(v)] = (unsigned short)(no + rank);
    cells[(size_t)b * cstride + no + rank] = (unsigned short)(v - c0);
  }
  for (int i = t; i < nn; i += 256) {
    const int v = list_n[i];
    int rank = 0;
    for (int k = 0; k < nn; ++k) rank += list_n[k] < v;
    id_n[N.find(v)] = (unsigned short)rank;
    nodes[(size_t)b * nstride + rank] = (unsigned short)(v - n0);
  }
  if (t == 0) head[b] = make_int4(c0, n0, no + nh, nn);
  __syncthreads();
  for (int i = t; i < no; i += 256) {
    const int c = owned[o0 + i];
    const int4 r = pcell[c];
    const int n[4] = {r.x, r.y, r.z, r.w};
    unsigned l[4], ent[4];
    for (int k = 0; k < 4; ++k) l[k] = id_n[N.find(n[k])];
    cells[(size_t)b * cstride + i] = (unsigned short)(c - c0);
    corners[o0 + i] = make_uint2(l[0] | (l[1] << 16), l[2] | (l[3] << 16));
    const ushort4 e = rec[o0 + i];
    const unsigned short in[4] = {e.x, e.y, e.z, e.w};
    for (int k = 0; k < 4; ++k) {
      if (in[k] == 0xFFFF) {
        ent[k] = kEntryNone;
      } else if (in[k] & 0x8000) {
        const unsigned j = in[k] & 0x7FFFu;
        if (kEntryBoundary + j >= kEntryNone) info[2] = 1;
        ent[k] = kEntryBoundary + j;
      } else {
        const int4 g = inst[e0 + (in[k] >> 1)];
        const int second = in[k] & 1, other = second ? g.z : g.w;
        const int p = pos[other];
        const unsigned id = p >= o0 && p < o1 ? (unsigned)(p - o0) : id_c[C.find(other)];
        int at = -1, swap = 0;
        for (int m = 0; m < 4; ++m) {
          const int u = n[m], v = n[(m + 1) & 3];
          if (at < 0 && u == g.x && v == g.y) at = m;
          if (at < 0 && u == g.y && v == g.x) {
            at = m;
            swap = 1;
          }
        }
        if (at < 0) info[2] = 1;
        ent[k] = id | ((unsigned)(at & 3) << kEntryBits) | ((unsigned)swap << (kEntryBits + 2)) |
                 ((unsigned)second << 15);
      }
    }
    edges[o0 + i] = make_uint2(ent[0] | (ent[1] << 16), ent[2] | (ent[3] << 16));
  }
}

// Builds the lists for an owner partition whose every cell (ncell of them) is
// owned; `alloc(bytes)` gives device memory that outlives them, or null.
// Returns false when a patch does not fit or there is no memory (any asked for
// then is unused).  Blocks until the device has built them.
template <class Alloc>
bool build_patches(const OwnerArgs &O, int nblocks, const ushort4 *rec, const int4 *pcell,
                   int ncell, hipStream_t st, Alloc alloc, PatchArgs *out, int *nc_max,
                   int *nn_max) {
  auto ck = [](hipError_t e) {
    if (e != hipSuccess) {
      printf("op2hip: building the patch lists failed: %s\n", hipGetErrorString(e));
      exit(-1);
    }
  };
  const size_t b_info = 256, b_pos = ((size_t)4 * ncell + 255) / 256 * 256;
  char *mem = (char *)alloc(b_info + b_pos);
  if (!mem) return false;
  int *info = (int *)mem, *pos = (int *)(mem + b_info);
  const int zeros[3] = {0, 0, 0};
  int got[3];
  ck(hipMemcpyAsync(info, zeros, sizeof zeros, hipMemcpyHostToDevice, st));
  k_patch_pos<<<(ncell + 255) / 256, 256, 0, st>>>(O.owned, ncell, pos);
  k_patch_lists<false><<<nblocks, 256, 0, st>>>(O.inst, O.elem_offs, O.owned_offs, O.owned, pos,
                                                rec, pcell, info, nullptr, nullptr, nullptr,
                                                nullptr, nullptr, 0, 0);
  ck(hipMemcpyAsync(got, info, sizeof got, hipMemcpyDeviceToHost, st));
  ck(hipStreamSynchronize(st));
  if (got[2]) return false;
  const int cs = (got[0] + 63) / 64 * 64, ns = (got[1] + 63) / 64 * 64;
  const size_t b_head = ((size_t)16 * nblocks + 255) / 256 * 256;
  const size_t b_ent = ((size_t)8 * ncell + 255) / 256 * 256;
  const size_t b_cells = ((size_t)2 * cs * nblocks + 255) / 256 * 256;
  char *m = (char *)alloc(b_head + 2 * b_ent + b_cells + (size_t)2 * ns * nblocks);
  if (!m) return false;
  int4 *head = (int4 *)m;
  uint2 *edges = (uint2 *)(m + b_head), *corners = (uint2 *)(m + b_head + b_ent);
  unsigned short *cells = (unsigned short *)(m + b_head + 2 * b_ent);
  unsigned short *nodes = (unsigned short *)(m + b_head + 2 * b_ent + b_cells);
  k_patch_lists<true><<<nblocks, 256, 0, st>>>(O.inst, O.elem_offs, O.owned_offs, O.owned, pos,
                                               rec, pcell, info, head, cells, nodes, edges,
                                               corners, cs, ns);
  ck(hipGetLastError());
  ck(hipMemcpyAsync(got, info, sizeof got, hipMemcpyDeviceToHost, st));
  ck(hipStreamSynchronize(st));
  if (got[2]) return false;
  *out = PatchArgs{head, cells, nodes, edges, corners, O.owned_offs, cs, ns};
  *nc_max = got[0];
  *nn_max = got[1];
  return true;
}

}  // namespace op2_dev
