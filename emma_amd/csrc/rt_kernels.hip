// rt_kernels.hip -- gfx950 kernels of the resident-level radiation step.
//
// One level step (the work of advancerad + RadSolver's final update for one
// level, rad_utils.c:1775-2006): a thread per cell reads its own state and its
// neighbours' through the oct index tables of the level's SoA arrays (no
// stencil copy; neighbours in the same tile through LDS), forms the
// Lax-Friedrichs M1 fluxes, updates, runs the chemistry sub-stepper in FP64 and
// writes the next state; split cells write the mean of their children instead.
// One kernel (level_step_kernel, level_step_tiled, level_step_split, with the
// straggler pass behind the tiled ones), or two where several groups' chemistry
// would hold the transport's registers (transport_kernel, chemistry_kernel);
// cell_step, with neighbours straight from memory, is the persistent kernel's
// per-cell form.  State is
// double-buffered (read A, write B), so the reference's rfieldnew copy
// (clean_new_rad) disappears; coarse-fine refluxes go to small per-level
// accumulators that the coarser level folds in on its next step.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "rt_fill.h"
#include "rt_kernels.h"
#include "rt_physics_fast.h"

namespace emma {

// ------------------------------------------------------------------ helpers
__device__ __forceinline__ int xcd_block(int nb) {
  // blocks are dealt round-robin to the 8 XCDs; give each XCD a contiguous
  // range of cells so that neighbour octs share its L2
  const int b = blockIdx.x;
  const int per = nb >> 3;
  return (b & 7) * per + (b >> 3);
}

// The tile of a block: of all tiles of the level, or of the launch's list (-1:
// no tile; the whole block)
template <typename R>
__device__ __forceinline__ int block_tile(const LevelArgs<R>& a) {
  const int i = xcd_block(a.nblocks);
  if (a.tiles == nullptr) return i;
  return i < a.ntiles ? a.tiles[i] : -1;
}

// The tile a block takes on a complete Morton-ordered cube of n = 2^m octs a
// side.  A tile is 32 Morton-consecutive octs, a 4 x 4 x 2 brick, so the
// tile index interleaves the tile coordinates (z, x, y from the lowest bit:
// tz0 tx0 ty0 tz1 ...; tz has one bit more).  Blocks are dealt round-robin
// to the 8 XCDs; XCD k takes octant k (the top bit of tx, ty, tz) and walks
// it z fastest, then y, then x: the neighbours across the largest faces
// (4 x 4 octs, +-z) are the next and previous tiles, the +-y ones n/4
// tiles away, within the ~128 tiles an XCD holds at once, so their halo
// cells are still in its L2.  In Morton order most of them were not.
__device__ __forceinline__ int raster_tile(int m) {
  const int b = blockIdx.x;
  const int k = b & 7, p = b >> 3;
  const int nz = 1 << (m - 2), ny = 1 << (m - 3);  // octant extent in tiles along z, y
  const int tz = (p & (nz - 1)) | ((k >> 2) << (m - 2));
  const int ty = ((p >> (m - 2)) & (ny - 1)) | (((k >> 1) & 1) << (m - 3));
  const int tx = (p >> (2 * m - 5)) | ((k & 1) << (m - 3));
  int t = 0;
#pragma unroll
  for (int i = 0; i < 14; i++) {
    if (i < m - 2) {
      t |= ((tz >> i) & 1) << (3 * i);
      t |= ((tx >> i) & 1) << (3 * i + 1);
      t |= ((ty >> i) & 1) << (3 * i + 2);
    }
  }
  t |= ((tz >> (m - 2)) & 1) << (3 * (m - 2));
  return t;
}

__device__ __forceinline__ void raise_status(int* status, int code, int level, int cell) {
  if (atomicCAS(status, 0, code) == 0) {
    status[1] = level;
    status[2] = cell;
  }
}

// lanes of mask m below this lane
__device__ __forceinline__ int lanes_below_mask(unsigned long long m) {
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

template <typename R>
__device__ __forceinline__ void load4(const LevelArgs<R>& a, const R* e, const R* fx, const R* fy, const R* fz,
                                      int n, int j, int g, R& oe, R& ofx, R& ofy, R& ofz) {
  oe = e[g * n + j];
  ofx = fx[g * n + j];
  ofy = fy[g * n + j];
  ofz = fz[g * n + j];
}

// Element i of an array whose base is the same in every lane of the wave.
// The base goes through readfirstlane (free for a value already in SGPRs) so
// that the optimiser cannot fold a per-lane index into it, and the byte
// offset is a 32-bit unsigned value: the access then takes the scalar-base
// form of the global load/store (64-bit base in SGPRs + 32-bit offset in one
// VGPR) rather than a 64-bit address per lane, and arrays indexed by the same
// cell share one offset register.  The level size limit (max_level_cells)
// keeps every offset below 4 GiB.
#define EMMA_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ EMMA_GLOBAL char* uniform_base(T* base) {
  const unsigned long long p = (unsigned long long)base;
  const unsigned long long lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)p);
  const unsigned long long hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(p >> 32));
  return (EMMA_GLOBAL char*)((hi << 32) | lo);
}
// the 32-bit byte offset, kept opaque so that a select or mask that formed
// the index is not pushed through the zero extension (which would hide the
// 32-bit offset from the instruction selector)
template <typename T>
__device__ __forceinline__ size_t byte_offset(int i) {
  unsigned off = (unsigned)i * (unsigned)sizeof(T);
  asm("" : "+v"(off));
  return (size_t)off;
}
template <typename T>
__device__ __forceinline__ T gld(const T* base, int i) {
  return *(const EMMA_GLOBAL T*)(uniform_base(base) + byte_offset<T>(i));
}
template <typename T>
__device__ __forceinline__ void gst(T* base, int i, T v) {
  *(EMMA_GLOBAL T*)(uniform_base(base) + byte_offset<T>(i)) = v;
}

// the same with the non-temporal hint (streamed: the line is not kept in L2
// for reuse).  For a large level's next state and its once-read chemistry
// inputs, which would otherwise push out of L2 the neighbouring tiles' cells
// that halo reads are about to fetch; small levels, whose next step finds
// their state in L2, keep the plain form.
template <typename T>
__device__ __forceinline__ void gst_nt(T* base, int i, T v) {
  __builtin_nontemporal_store(v, (EMMA_GLOBAL T*)(uniform_base(base) + byte_offset<T>(i)));
}
template <typename T>
__device__ __forceinline__ T gld_nt(const T* base, int i) {
  return __builtin_nontemporal_load((const EMMA_GLOBAL T*)(uniform_base(base) + byte_offset<T>(i)));
}
template <bool NT, typename T>
__device__ __forceinline__ void gst_out(T* base, int i, T v) {
  if constexpr (NT)
    gst_nt(base, i, v);
  else
    gst(base, i, v);
}
template <bool NT, typename T>
__device__ __forceinline__ T gld_in(const T* base, int i) {
  if constexpr (NT)
    return gld_nt(base, i);
  else
    return gld(base, i);
}

template <typename R, bool Fast>
__device__ __forceinline__ Closure<R> closure_of(R fx, R fy, R fz, R ee, R c) {
  if constexpr (Fast)
    return closure_fast(fx, fy, fz, ee, c);
  else
    return closure<R>(fx, fy, fz, ee, c);
}

// The level-step kernels take (LevelArgs, ChemConst) by value but read them
// through the kernarg segment pointer where they are used.  By-value kernel
// arguments are all loaded into SGPRs at kernel entry; a level step has more
// of them than there are SGPRs, and the overflow is spilled to VGPR lanes and
// read back with a v_readlane per use.  Loads at the point of use keep only
// the live ones in SGPRs.  The explicit arguments sit at offset 0 and right
// after the LevelArgs block (both 8-byte aligned).
template <typename R>
struct KernArgs {
  const LevelArgs<R>& a;
  const ChemConst& K;
};
template <typename R>
__device__ __forceinline__ KernArgs<R> kernargs() {
  static_assert(sizeof(LevelArgs<R>) % alignof(ChemConst) == 0, "ChemConst follows LevelArgs unpadded");
  const char* kp = (const char*)__builtin_amdgcn_kernarg_segment_ptr();  // constant address space -> generic
  return {*reinterpret_cast<const LevelArgs<R>*>(kp), *reinterpret_cast<const ChemConst*>(kp + sizeof(LevelArgs<R>))};
}

// ------------------------------------------------------------------ pieces
// reionisation-time bookkeeping of RadSolver (rad_utils.c:1901-1913)
template <typename R>
__device__ __forceinline__ void xion_times(const LevelArgs<R>& a, int cell) {
  const double xion = a.nhplus[cell] / a.nh[cell];
  if (xion < 0.5) a.t_last[cell] = a.tphy;
  if ((xion >= 0.5) && (a.t_first[cell] == -1)) a.t_first[cell] = a.tphy;
}

// split cell: its next state is the mean of its 8 children (rad_utils.c:1955-2006);
// group g's fields, and the cell fields
template <typename R>
__device__ __forceinline__ void restrict_group(const LevelArgs<R>& a, int cell, int ch, int g) {
  const int n = a.ncell, nf = a.nfine, j0 = ch * 8;
  R se = R(0), sx = R(0), sy = R(0), sz = R(0), ss = R(0);
#pragma unroll
  for (int k = 0; k < 8; k++) {
    // plain indexing: the eight children's values merge into wide loads
    const int j = g * nf + j0 + k;
    se += a.fe[j] * R(0.125);
    sx += a.ffx[j] * R(0.125);
    sy += a.ffy[j] * R(0.125);
    sz += a.ffz[j] * R(0.125);
    ss += a.fsrc[j] * R(0.125);
  }
  gst(a.eo + g * n, cell, se);
  gst(a.fxo + g * n, cell, sx);
  gst(a.fyo + g * n, cell, sy);
  gst(a.fzo + g * n, cell, sz);
  gst(a.src + g * n, cell, ss);
}

template <typename R>
__device__ __forceinline__ void restrict_scalars(const LevelArgs<R>& a, int cell, int ch) {
  const int j0 = ch * 8;
  // (no branch inside the loop: the 32 loads go out together)
  double snp = 0., sei = 0., stp = 0., snh = 0.;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int j = j0 + k;
    snp += a.fnhplus[j] * 0.125;
    sei += a.feint[j] * 0.125;
    stp += a.ftemp[j] * 0.125;
    snh += a.fnh[j] * 0.125;
  }
  gst(a.nhpluso, cell, snp);
  gst(a.einto, cell, sei);
  gst(a.tempo, cell, stp);
  gst(a.nh, cell, snh);
  if (a.t_first != nullptr) {
    double stf = 0., stl = 0.;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      stf += a.ft_first[j0 + k] * 0.125;
      stl += a.ft_last[j0 + k] * 0.125;
    }
    a.t_first[cell] = stf;
    a.t_last[cell] = stl;
  }
}

template <typename R>
__device__ __forceinline__ void restrict_cell(const LevelArgs<R>& a, int cell, int ch, int ng) {
  for (int g = 0; g < ng; g++) restrict_group(a, cell, ch, g);
  restrict_scalars(a, cell, ch);
}

// Reflux accumulators: [pair][group][component][sub-slot].  The sub-slots (one
// per cell of the oct face, Sub = 4, or the face's sum, Sub = 1) are innermost:
// the four lanes of an oct face add a component to adjacent words, one request
// of the L2's atomic units in place of four, and a (pair, group) is one 128 B
// line in FP64, read back with wide loads.  With the sub-slot outside
// ([pair][sub-slot][component][group]) the three-group FP64 tree of 64^3 cells
// and 9,000 and 2,500 octs took 213.5 us a coarse step, 41 of them the adds and
// 9 the reads; now 171.5.
template <int GA, int Sub>
__device__ __forceinline__ size_t acc_at(int pair, int g) {
  return ((size_t)pair * GA + g) * (4 * Sub);
}

// reflux of one face flux into the coarse leaf behind it (scatterstencilrad,
// rad_utils.c:1738-1762): the coarse cell gains -/+ F dt/dx / 8.  The cell's
// own accumulator of the reflux pair p (sub-slot q: its place in the oct
// face).  No other lane adds to it in this launch, so the sum is the same every
// run; the add is an atomic only so that the lane need not wait for the old
// value.
template <typename R, int GA>
__device__ __forceinline__ void reflux(const LevelArgs<R>& a, int p, int q, int f, int g, const R F[4], R dts) {
  R* acc = a.cracc + acc_at<GA, kRefluxCell>(p, g) + q;
  const R w = (f & 1) ? R(1) : R(-1);  // pow(-1, face+1)
#pragma unroll
  for (int v = 0; v < 4; v++) atomicAdd(acc + v * kRefluxCell, F[v] * dts * w * R(0.125));
}

// the refluxes of the finer octs behind a leaf's faces, added to its base
// state in pair order; their accumulators are cleared.  Sub: accumulators per
// pair, GA: groups an accumulator holds, groups [g0, g0 + NG) are taken.
template <typename R, int GA, int NG, int Sub>
__device__ __forceinline__ void fold_reflux(const LevelArgs<R>& a, int ch, int g0, int ng, R* Ue, R* Ux, R* Uy, R* Uz) {
  const int code = -2 - ch;
  const int p0 = code >> 3, m = code & 7;
  // all loads before the clearing stores.  A leaf has at most six pairs:
  // the tiled kernel's loop unrolls, and its loads (an accumulator's 4G
  // values are contiguous), clamped to the leaf's last accumulator, go out
  // together instead of one pair after another; the per-cell kernels take a
  // pair's 16 values of a group at a time
  constexpr int kPairs = 6;
  R s[NG][4];
#pragma unroll
  for (int g = 0; g < NG; g++) s[g][0] = s[g][1] = s[g][2] = s[g][3] = R(0);
#pragma unroll(Sub == 1 ? kPairs : 1)
  for (int i = 0; i < (Sub == 1 ? kPairs : m); i++) {
#pragma unroll
    for (int g = 0; g < NG; g++) {
      if (g < ng) {
        const R* p = a.racc + acc_at<GA, Sub>(p0 + min(i, m - 1), g0 + g);
        R x[4 * Sub];
#pragma unroll
        for (int k = 0; k < 4 * Sub; k++) x[k] = p[k];
#pragma unroll
        for (int q = 0; q < Sub; q++)
#pragma unroll
          for (int v = 0; v < 4; v++) s[g][v] += i < m ? x[v * Sub + q] : R(0);
      }
    }
  }
#pragma unroll(Sub == 1 ? kPairs : 1)
  for (int i = 0; i < (Sub == 1 ? kPairs : m); i++) {
    if (i < m) {
#pragma unroll
      for (int g = 0; g < NG; g++) {
        if (g < ng) {
          R* p = a.racc + acc_at<GA, Sub>(p0 + i, g0 + g);
#pragma unroll
          for (int k = 0; k < 4 * Sub; k++) p[k] = R(0);
        }
      }
    }
  }
#pragma unroll
  for (int g = 0; g < NG; g++) {
    if (g < ng) {
      Ue[g] += s[g][0];
      Ux[g] += s[g][1];
      Uy[g] += s[g][2];
      Uz[g] += s[g][3];
    }
  }
}

// A leaf whose chemistry budget is spent (st == 1): the transported N, F are
// stored unscaled (fscale = 1) and the cell goes on the straggler list, one
// atomic per wave.  Returns whether it was put off.
template <typename R>
__device__ __forceinline__ bool defer_leaf(const LevelArgs<R>& a, int cell, int& st, int& nit) {
  const bool deferred = st == 1;
  const unsigned long long dm = __ballot(deferred);
  if (dm != 0ull) {
    const int leader = __ffsll((long long)dm) - 1;
    int base = 0;
    if ((int)__lane_id() == leader) base = atomicAdd(a.defer_ctl, __popcll(dm));
    base = __shfl(base, leader);
    if (deferred) {
      const int slot = base + lanes_below_mask(dm);
      if (slot < a.defer_cap)
        a.defer_list[slot] = cell;
      else
        raise_status(a.status, -1, a.level, cell);  // list smaller than the level (host sizes it)
      st = 0;
      nit = 0;
    }
  }
  return deferred;
}

// leaf cell after its transport (T: the updated state): N<0/NaN guard,
// chemistry, write of the next state.  Returns the accepted chemistry
// sub-steps.
// The chemistry inputs (src, x n_H, eint, n_H) come from memory, or from
// `pre` when the caller loaded them early (pre_src[GA], pre[3]).
template <typename R, int G, bool Fast, int Sub, bool NT = false>
__device__ __forceinline__ int finish_leaf(const LevelArgs<R>& a, const ChemConst& K, int cell, int ng, const R* Te,
                                           const R* Tx, const R* Ty, const R* Tz, const R* pre_src = nullptr,
                                           const double* pre = nullptr) {
  constexpr int GA = G > 0 ? G : kMaxGrp;
  const int n = a.ncell;
  double e[GA], src[GA];
  R fx[GA], fy[GA], fz[GA];  // fluxes after transport, in the storage type
#pragma unroll
  for (int g = 0; g < GA; g++) {
    if (g < ng) {
      e[g] = (double)Te[g];
      fx[g] = Tx[g];
      fy[g] = Ty[g];
      fz[g] = Tz[g];
      src[g] = (double)(pre_src != nullptr ? pre_src[g] : gld(a.src + g * n, cell));
    }
  }
  // rad_utils.c:1611-1650 (the second test reads e[1], i.e. fx[0] when G=1)
  if (e[0] < 0 || isnan(e[0]) || isnan(ng > 1 ? e[1 < GA ? 1 : 0] : (double)fx[0]))
    raise_status(a.status, -3, a.level, cell);
  double nhplus = pre != nullptr ? pre[0] : gld(a.nhplus, cell);
  double eint = pre != nullptr ? pre[1] : gld(a.eint, cell);
  const double nh = pre != nullptr ? pre[2] : gld(a.nh, cell);
  double temp = 0.;
  int nit = 0;
  int st;
  bool deferred = false;  // chemistry left to the straggler pass
  if constexpr (Fast) {
    double fscale[GA];
    st = chem_cell_fast<G>(K, ng, e, fscale, src, nhplus, eint, nh, temp, a.chemonly, nit,
                           Sub == kRefluxTiled && a.chem_budget > 0 ? a.chem_budget : -1, (double)a.chem_keep);
    if constexpr (Sub == kRefluxTiled) {
      deferred = defer_leaf(a, cell, st, nit);
    }
#pragma unroll
    for (int g = 0; g < GA; g++) {
      if (g < ng) {
        const R fs = (R)fscale[g];
        fx[g] *= fs;
        fy[g] *= fs;
        fz[g] *= fs;
      }
    }
  } else {
    double dfx[GA], dfy[GA], dfz[GA];
#pragma unroll
    for (int g = 0; g < GA; g++) {
      if (g < ng) {
        dfx[g] = (double)fx[g];
        dfy[g] = (double)fy[g];
        dfz[g] = (double)fz[g];
      }
    }
    st = chem_cell<G>(K, ng, e, dfx, dfy, dfz, src, nhplus, eint, nh, temp, a.chemonly, nit);
#pragma unroll
    for (int g = 0; g < GA; g++) {
      if (g < ng) {
        fx[g] = (R)dfx[g];
        fy[g] = (R)dfy[g];
        fz[g] = (R)dfz[g];
      }
    }
  }
  if (st != 0) raise_status(a.status, st, a.level, cell);
#pragma unroll
  for (int g = 0; g < GA; g++) {
    if (g < ng) {
      R ev = (R)e[g];
      // FP32 storage: a density the chemistry left at (or just above) its
      // floor must not round below it, or the next step would stop at the
      // floor test (chem_utils.c:382); only the rounding is corrected
      if constexpr (sizeof(R) == 4)
        if (!deferred && e[g] >= K.emin_grp[g] && ev < K.emin_grp_up[g]) ev = K.emin_grp_up[g];
      gst_out<NT>(a.eo + g * n, cell, ev);
      gst_out<NT>(a.fxo + g * n, cell, fx[g]);
      gst_out<NT>(a.fyo + g * n, cell, fy[g]);
      gst_out<NT>(a.fzo + g * n, cell, fz[g]);
    }
  }
  gst_out<NT>(a.nhpluso, cell, nhplus);
  gst_out<NT>(a.einto, cell, eint);
  gst_out<NT>(a.tempo, cell, temp);
  return nit;
}

// COARSERAD coarse level: a split cell takes the transport update of its own
// state (updatefieldrad without the split test, rad_utils.c:1548-1552) and
// keeps x, eint, T (chemrad skips it)
template <typename R, int GA>
__device__ __forceinline__ void transport_split_cell(const LevelArgs<R>& a, int cell, int ng, const R* Te, const R* Tx,
                                                     const R* Ty, const R* Tz) {
  const int n = a.ncell;
#pragma unroll
  for (int g = 0; g < GA; g++) {
    if (g < ng) {
      gst(a.eo + g * n, cell, Te[g]);
      gst(a.fxo + g * n, cell, Tx[g]);
      gst(a.fyo + g * n, cell, Ty[g]);
      gst(a.fzo + g * n, cell, Tz[g]);
    }
  }
  const double e0 = (double)Te[0];
  const double e1 = ng > 1 ? (double)Te[1 < GA ? 1 : 0] : (double)Tx[0];
  if (e0 < 0 || isnan(e0) || isnan(e1)) raise_status(a.status, -3, a.level, cell);
  gst(a.nhpluso, cell, gld(a.nhplus, cell));
  gst(a.einto, cell, gld(a.eint, cell));
  gst(a.tempo, cell, gld(a.temp, cell));
}

// per-block counters: accepted chemistry sub-steps and leaf cell-updates,
// one atomic pair per block into a spread slot.  The wave sums come from
// ballots (scalar popcounts): the leaf flags directly, the sub-step counts
// bit plane by bit plane over their low 4 bits; a lane with 16 or more
// sub-steps adds the rest with its own atomic.
template <int NW>
__device__ __forceinline__ void block_counters(unsigned long long* counters, unsigned int nit, unsigned int leaf) {
  __shared__ unsigned int red[2][NW];
  unsigned long long* slot = counters + (size_t)(blockIdx.x % kCounterSlots) * kCounterStride;
  unsigned int s0 = 0;
#pragma unroll
  for (int b = 0; b < 4; b++) s0 += (unsigned int)__popcll(__ballot((nit >> b) & 1u)) << b;
  const unsigned int s1 = (unsigned int)__popcll(__ballot(leaf != 0u));
  if (nit >= 16u) atomicAdd(slot, (unsigned long long)(nit & ~15u));
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[0][w] = s0;
    red[1][w] = s1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t0 = 0, t1 = 0;
    for (int i = 0; i < NW; i++) {
      t0 += red[0][i];
      t1 += red[1][i];
    }
    atomicAdd(slot + 0, t0);
    atomicAdd(slot + 1, t1);
  }
}

// ------------------------------------------------------------------ level step
// One thread per cell; neighbours straight from global memory.  Fast selects
// the mixed-precision physics (rt_physics_fast.h); FP64 (Fast = false) keeps
// the reference's operation order.  The persistent kernel's per-cell items;
// the per-level launches run the kernels below through LDS.
// The cells of block `block` (256 consecutive cells, 32 octs).
template <typename R, int G, bool Fast>
__device__ __forceinline__ void cell_step(const LevelArgs<R>& a, const ChemConst& K, int block, int lc) {
  constexpr int GA = G > 0 ? G : kMaxGrp;
  const int ng = G > 0 ? G : a.ng;
  const int cell = block * 256 + lc;
  unsigned int nit_acc = 0;
  unsigned int leaf = 0;
  if (cell < a.ncell) {
    const int n = a.ncell;
    const int oct = cell >> 3, ic = cell & 7;
    const int ch = a.child[cell];
    if (a.t_first != nullptr) xion_times(a, cell);
    if (ch >= 0 && !a.update_split) {
      restrict_cell(a, cell, ch, ng);
    } else {
      const R c = a.c, hc = a.hc, dts = a.dtsurdx;
      R Ue[GA], Ux[GA], Uy[GA], Uz[GA];
      R De[GA], Dx[GA], Dy[GA], Dz[GA];
      Closure<R> Q[GA];
#pragma unroll
      for (int g = 0; g < GA; g++) {
        if (g < ng) {
          Ue[g] = a.e[g * n + cell];
          Ux[g] = a.fx[g * n + cell];
          Uy[g] = a.fy[g * n + cell];
          Uz[g] = a.fz[g * n + cell];
          if constexpr (Fast)
            Q[g] = closure_fast(Ux[g], Uy[g], Uz[g], Ue[g], c);
          else
            Q[g] = closure<R>(Ux[g], Uy[g], Uz[g], Ue[g], c);
          De[g] = Dx[g] = Dy[g] = Dz[g] = R(0);
        }
      }
      // six faces in the reference order (rad_utils.c:1566-1574): f = 2d+s
#pragma unroll
      for (int f = 0; f < (a.transport ? 6 : 0); f++) {
        const int d = f >> 1, s = f & 1;
        const int nc = ic ^ (1 << d);
        const R* Ne = a.e;
        const R* Nx = a.fx;
        const R* Ny = a.fy;
        const R* Nz = a.fz;
        int nn = n, j, split;
        int coarse_face = 0, pr = -1, reflect = 0;
        if (((ic >> d) & 1) != s) {  // neighbour inside the oct
          j = oct * 8 + nc;
          split = a.child[j] >= 0;
        } else {
          const int no = a.nei[oct * 6 + f];
          if (no >= 0) {
            j = no * 8 + nc;
            split = a.child[j] >= 0;
          } else if (no <= kNeiReflective) {  // domain face (rad_utils.c:1106-1213, 1376-1407)
            j = oct * 8 + trans_source(f, ic);
            split = a.child[j] >= 0;
            reflect = no == kNeiReflective;
          } else {  // coarse leaf injected into the stencil
            j = -1 - no;
            split = 0;
            Ne = a.ce;
            Nx = a.cfx;
            Ny = a.cfy;
            Nz = a.cfz;
            nn = a.ncoarse;
            coarse_face = 1;
            pr = a.rpair[oct * 6 + f];
          }
        }
        const R ffact = (split && !a.keep_split_flux) ? R(0) : R(1);
        const R one = (f & 1) ? R(-1) : R(1);
#pragma unroll
        for (int g = 0; g < GA; g++) {
          if (g < ng) {
            R ve, vx, vy, vz;
            load4(a, Ne, Nx, Ny, Nz, nn, j, g, ve, vx, vy, vz);
            if (reflect) {
              if (d == 0) vx = -vx;
              if (d == 1) vy = -vy;
              if (d == 2) vz = -vz;
            }
            Closure<R> qn;
            if constexpr (Fast)
              qn = closure_fast(vx, vy, vz, ve, c);
            else
              qn = closure<R>(vx, vy, vz, ve, c);
            R F[4];
            lf_flux<R>(d, s, Ue[g], Ux[g], Uy[g], Uz[g], Q[g], ve, vx, vy, vz, qn, hc, F);
#pragma unroll
            for (int v = 0; v < 4; v++) F[v] *= ffact;
            De[g] += F[0] * dts * one;
            Dx[g] += F[1] * dts * one;
            Dy[g] += F[2] * dts * one;
            Dz[g] += F[3] * dts * one;
            if (coarse_face) {
              // the cell's place in the oct face: its two coordinates across d
              const int q = ((ic >> ((d + 1) % 3)) & 1) | (((ic >> ((d + 2) % 3)) & 1) << 1);
              reflux<R, GA>(a, pr, q, f, g, F, dts);
            }
          }
        }
      }
      if (ch <= -2) fold_reflux<R, GA, GA, kRefluxCell>(a, ch, 0, ng, Ue, Ux, Uy, Uz);
#pragma unroll
      for (int g = 0; g < GA; g++) {
        if (g < ng) {
          Ue[g] += De[g];
          Ux[g] += Dx[g];
          Uy[g] += Dy[g];
          Uz[g] += Dz[g];
        }
      }
      if (ch >= 0) {
        transport_split_cell<R, GA>(a, cell, ng, Ue, Ux, Uy, Uz);
      } else {
        leaf = 1;
        nit_acc = (unsigned)finish_leaf<R, G, Fast, kRefluxCell>(a, K, cell, ng, Ue, Ux, Uy, Uz);
      }
    }
  }
  if (a.counters != nullptr) block_counters<4>(a.counters, nit_acc, leaf);
}

// The same step with every closure computed once.  FP64 with any group count
// and mixed precision with other than 1 or 3 groups; the operations and their
// order are those of cell_step, so the results are the same bit for bit.
//
// cell_step is bound by its FP64 instructions: seven closures per cell and
// group (its own and six neighbours', five divisions and two square roots
// each) where two are enough.  Here a 256-thread work-group owns 32
// consecutive octs, one cell per thread, and takes one photon group at a time:
// each cell's state and closure go to LDS once, neighbours in the tile are read
// from there, and only the halo (a third to a half of the leaving faces on a
// complete level) is evaluated again: on complete levels (variant kListed) one
// listed halo face per lane in one round, on sparse ones each lane its own
// leaving face in each direction pass.
template <typename R>
__device__ __forceinline__ CellLds<R>* cell_lds() {
  __shared__ CellLds<R> lds;
  return &lds;
}

// what a thread's cell needs for the transport of any group
struct CellFaces {
  int cell, ch;
  int noD[3];    // nei_oct entry of the face that leaves the oct, per direction
  int pairD[3];  // its reflux pair where a coarse leaf lies behind it, -1 elsewhere
  bool valid, restricted, moves, listed;
  unsigned long long hball[3];  // listed: lanes whose face in direction d is a halo face,
  int hbase[3];                 // and the first halo slot of direction d
};

// where the neighbour across a halo face lies
struct HaloCell {
  int j, d;
  bool on, coarse, refl;
};

// the halo face in direction d of cell hcell, nei_oct entry no
__device__ __forceinline__ HaloCell halo_cell(bool on, int hcell, int d, int no) {
  HaloCell h;
  const int hic = hcell & 7, side = (hic >> d) & 1;
  const bool bound = on && no <= kNeiReflective;  // domain face (rad_utils.c:1106-1213, 1376-1407)
  h.on = on;
  h.d = d;
  h.coarse = on && no < 0 && !bound;
  h.refl = bound && no == kNeiReflective;
  h.j = !on ? 0 : bound ? (hcell & ~7) + trans_source(2 * d + side, hic) : h.coarse ? -1 - no : no * 8 + (hic ^ (1 << d));
  return h;
}

// the flux from a split neighbour is dropped (RADSTEP)
template <typename R>
__device__ __forceinline__ bool halo_cancel(const LevelArgs<R>& a, const HaloCell& h) {
  return h.on && !h.coarse && !a.keep_split_flux && gld(a.child, h.j) >= 0;
}

// group g of its state
template <typename R>
__device__ __forceinline__ void halo_load(const LevelArgs<R>& a, const HaloCell& h, int g, R v[4]) {
  if (!h.on) return;
  // the lane's array is this level's plus a per-lane distance (0, or the
  // coarse array's address minus this level's), both bases scalar: no 64-bit
  // address per lane and array
  const size_t o = byte_offset<R>(h.j);
  auto load = [&](const R* own, const R* coarser) {
    const R* const ob = own + (size_t)g * a.ncell;
    const R* const cb = coarser + (size_t)g * a.ncoarse;
    const unsigned long long dist = (unsigned long long)cb - (unsigned long long)ob;
    return *(const EMMA_GLOBAL R*)(uniform_base(ob) + (h.coarse ? dist : 0ull) + o);
  };
  v[0] = load(a.e, a.ce);
  v[1] = load(a.fx, a.cfx);
  v[2] = load(a.fy, a.cfy);
  v[3] = load(a.fz, a.cfz);
}

// into LDS slot i, with its closure
template <typename R, bool Fast>
__device__ __forceinline__ void halo_put(const LevelArgs<R>& a, CellLds<R>& lds, const HaloCell& h, const R v[4], int i) {
  if (!h.on) return;
  const R ve = v[0];
  R vx = v[1], vy = v[2], vz = v[3];
  if (h.refl) {
    if (h.d == 0) vx = -vx;
    if (h.d == 1) vy = -vy;
    if (h.d == 2) vz = -vz;
  }
  lds.put(i, ve, vx, vy, vz, closure_of<R, Fast>(vx, vy, vz, ve, a.c));
}

__device__ __forceinline__ bool in_tile32(int no, int tile) {
  return no >= tile * kTileOcts && no < (tile + 1) * kTileOcts;
}

// sparse levels: the cell's own halo face of direction d
__device__ __forceinline__ HaloCell own_face(const CellFaces& c, int tile, int d) {
  return halo_cell(c.moves && !in_tile32(c.noD[d], tile), c.cell, d, c.noD[d]);
}

// group g of the cell's state
template <typename R>
__device__ __forceinline__ void own_load(const LevelArgs<R>& a, int cell, int g, R T[4]) {
  if (cell >= a.ncell) return;
  T[0] = gld(a.e + (size_t)g * a.ncell, cell);
  T[1] = gld(a.fx + (size_t)g * a.ncell, cell);
  T[2] = gld(a.fy + (size_t)g * a.ncell, cell);
  T[3] = gld(a.fz + (size_t)g * a.ncell, cell);
}

// the tile's cancel flags and, on complete levels, each wave's halo list (this
// lane's entry in hl); before the first group's transport.  The loads that group
// g needs first go out here, with the ones they'd otherwise wait behind: the
// cell's state T with the topology, the halo state H with the cancel flags
template <typename R>
__device__ __forceinline__ CellFaces cell_faces(const LevelArgs<R>& a, int tile, int lc, CellLds<R>& lds, HaloCell& hl,
                                                int g, R T[4], R H[4]) {
  CellFaces c;
  const int wv = lc >> 6, lane = lc & 63;
  c.cell = tile * kTileCells + lc;
  const int oct = c.cell >> 3, ic = c.cell & 7;
  c.valid = c.cell < a.ncell;
  c.listed = a.variant == kListed;
  c.ch = -1;
  const bool transport = a.transport != 0;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    c.noD[d] = 0;
    c.pairD[d] = -1;
    c.hball[d] = 0ull;
    c.hbase[d] = 0;
  }
  if (c.valid) {
    c.ch = gld(a.child, c.cell);
    if (transport) {
#pragma unroll
      for (int d = 0; d < 3; d++) c.noD[d] = gld(a.nei, oct * 6 + 2 * d + ((ic >> d) & 1));
    }
  }
  own_load(a, c.cell, g, T);
  c.restricted = c.ch >= 0 && !a.update_split;  // takes its children's mean, no transport
  c.moves = c.valid && transport && !c.restricted;
  hl.on = false;
  if (!transport) return c;
  lds.cancel[lc] = (unsigned char)(c.ch >= 0 && !a.keep_split_flux);
  if (a.ncoarse > 0) {
#pragma unroll
    for (int d = 0; d < 3; d++)
      if (c.moves && c.noD[d] < 0 && c.noD[d] > kNeiReflective)
        c.pairD[d] = gld(a.rpair, oct * 6 + 2 * d + ((ic >> d) & 1));
  }
  if (c.listed) {
    int nhalo = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const bool out = c.moves && !in_tile32(c.noD[d], tile);
      c.hball[d] = __ballot(out);
      c.hbase[d] = nhalo;
      nhalo += __popcll(c.hball[d]);
      if (out) {
        const int slot = c.hbase[d] + lanes_below_mask(c.hball[d]);  // < kHaloCap (variant chosen from the topology)
        lds.item[wv][slot] = (unsigned char)(lane * 4 + d);
        lds.item_nei[wv][slot] = c.noD[d];
      }
    }
    // the list is written and read by lanes of the same wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int it = lds.item[wv][lane];
    hl = halo_cell(lane < nhalo, (c.cell & ~63) + (it >> 2), it & 3, lds.item_nei[wv][lane]);
    halo_load(a, hl, g, H);
    lds.cancel[kTileCells + lc] = (unsigned char)halo_cancel(a, hl);
  } else {
    // each lane's own slot serves one direction after the other: their flags
    // as bits of one byte (the three loads at once, lanes without a face read
    // cell 0)
    unsigned flags = 0;
    int hch[3];
    bool on[3];
    halo_load(a, own_face(c, tile, 0), g, H);
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const HaloCell h = own_face(c, tile, d);
      on[d] = h.on && !h.coarse && !a.keep_split_flux;
      hch[d] = gld(a.child, on[d] ? h.j : 0);
    }
#pragma unroll
    for (int d = 0; d < 3; d++) flags |= on[d] && hch[d] >= 0 ? 1u << d : 0u;
    lds.cancel[kTileCells + lc] = (unsigned char)flags;
  }
  return c;
}

// Transport of group g of the thread's cell: its updated state in T, the
// refluxes of the finer octs folded in.  T and H come with the cell's and the
// halo's state (from cell_faces; H is used up).  GA: groups of a reflux
// accumulator.  All threads of the work-group.
template <typename R, int GA, bool Fast>
__device__ __forceinline__ void transport_group(const LevelArgs<R>& a, const CellFaces& cf, const HaloCell& hl, int tile,
                                                int lc, CellLds<R>& lds, int g, R T[4], R H[4]) {
  const int ic = cf.cell & 7, hslot0 = kTileCells + (lc & ~63), lane = lc & 63;
  const R c = a.c, hc = a.hc, dts = a.dtsurdx;
  const bool fold = cf.valid && !cf.restricted && cf.ch <= -2;
  if (!a.transport) {
    if (fold) fold_reflux<R, GA, 1, kRefluxCell>(a, cf.ch, g, 1, &T[0], &T[1], &T[2], &T[3]);
    return;
  }
  const R ue = T[0], ux = T[1], uy = T[2], uz = T[3];
  Closure<R> Q;
  if (cf.valid) {
    Q = closure_of<R, Fast>(ux, uy, uz, ue, c);
    lds.put(lc, ue, ux, uy, uz, Q);
  }
  if (cf.listed) halo_put<R, Fast>(a, lds, hl, H, hslot0 + lane);
  __syncthreads();
  if (!cf.moves) return;
  R D[4] = {R(0), R(0), R(0), R(0)};
#pragma unroll
  for (int d = 0; d < 3; d++) {
    // one face in d lies inside the oct and one leaves it; bit says which is
    // which (bit 1: the minus face is the inside one)
    const int bit = (ic >> d) & 1, jin = lc ^ (1 << d);
    const bool inT = in_tile32(cf.noD[d], tile);
    const int jl = (int)(((unsigned)cf.noD[d] - (unsigned)(tile * kTileOcts)) * 8u + (unsigned)(ic ^ (1 << d)));
    const int slot = cf.listed ? cf.hbase[d] + lanes_below_mask(cf.hball[d]) : lane;
    const int jout = inT ? jl : hslot0 + slot;
    // (own slot: written and read by this lane alone)
    if (!cf.listed) {
      halo_put<R, Fast>(a, lds, own_face(cf, tile, d), H, hslot0 + lane);
      if (d < 2) halo_load(a, own_face(cf, tile, d + 1), g, H);
    }
    const bool cin = lds.cancel[jin] != 0;
    const bool cout = (cf.listed || inT) ? lds.cancel[jout] != 0 : ((lds.cancel[jout] >> d) & 1) != 0;
    // the flux from a neighbour is multiplied by 0 or 1 (rad_utils.c:518-526)
    const R keepm = (bit ? cin : cout) ? R(0) : R(1), keepp = (bit ? cout : cin) ? R(0) : R(1);
    const int jm = bit ? jin : jout, jp = bit ? jout : jin;
    R Fm[4], Fp[4], ve, vx, vy, vz;
    Closure<R> qv;
    lds.get(jm, ve, vx, vy, vz, qv);
    lf_flux<R>(d, 0, ue, ux, uy, uz, Q, ve, vx, vy, vz, qv, hc, Fm);
    lds.get(jp, ve, vx, vy, vz, qv);
    lf_flux<R>(d, 1, ue, ux, uy, uz, Q, ve, vx, vy, vz, qv, hc, Fp);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      Fm[v] *= keepm;
      Fp[v] *= keepp;
      // the minus face first, as the six faces are numbered
      D[v] += Fm[v] * dts;
      D[v] -= Fp[v] * dts;
    }
    if (cf.pairD[d] >= 0) {
      // the cell's place in the oct face: its two coordinates across d
      const int q = ((ic >> ((d + 1) % 3)) & 1) | (((ic >> ((d + 2) % 3)) & 1) << 1);
      R F[4];
#pragma unroll
      for (int v = 0; v < 4; v++) F[v] = bit ? Fp[v] : Fm[v];
      reflux<R, GA>(a, cf.pairD[d], q, 2 * d + bit, g, F, dts);
    }
  }
  if (fold) fold_reflux<R, GA, 1, kRefluxCell>(a, cf.ch, g, 1, &T[0], &T[1], &T[2], &T[3]);
#pragma unroll
  for (int v = 0; v < 4; v++) T[v] += D[v];
}

// One group, FP64: transport and chemistry in one kernel, four waves per SIMD
// (64^3 cells 22.2 us with the allocation left free, 20.1 so).
__global__ __launch_bounds__(kTileCells) __attribute__((amdgpu_waves_per_eu(4))) void level_step_kernel(
    LevelArgs<double> a_by_value, ChemConst K_by_value) {
  const KernArgs<double> args = kernargs<double>();
  const LevelArgs<double>& a = args.a;
  CellLds<double>& lds = *cell_lds<double>();
  const int tile = block_tile(a), lc = (int)threadIdx.x;
  if (tile < 0) return;
  HaloCell hl;
  double T[4], H[4];
  const CellFaces cf = cell_faces(a, tile, lc, lds, hl, 0, T, H);
  transport_group<double, 1, false>(a, cf, hl, tile, lc, lds, 0, T, H);
  unsigned int nit_acc = 0, leaf = 0;
  if (cf.valid) {
    if (a.t_first != nullptr) xion_times(a, cf.cell);
    if (cf.restricted) {
      restrict_cell(a, cf.cell, cf.ch, 1);
    } else if (cf.ch >= 0) {
      transport_split_cell<double, 1>(a, cf.cell, 1, &T[0], &T[1], &T[2], &T[3]);
    } else {
      leaf = 1;
      nit_acc = (unsigned)finish_leaf<double, 1, false, kRefluxCell>(a, args.K, cf.cell, 1, &T[0], &T[1], &T[2], &T[3]);
    }
  }
  if (a.counters != nullptr) block_counters<kTileWaves>(a.counters, nit_acc, leaf);
}

// More groups: the transport as a kernel of its own, one group a work-group
// (gridDim.y = ng), which leaves the transported state in the next state's
// arrays, and the chemistry after it.  In one kernel the chemistry's registers
// (168 to 256) held the transport to one to three waves per SIMD, and a small
// level waited for all groups' transport in one wave's chain; apart, the
// transport takes 106 (FP32 58).  A level step of 32^3 cells, nine FP64 groups:
// 41 -> 26.2 us, though the transported state is written and read once more;
// 64^3 cells, nine FP32 groups 55.4 -> 49.6 us.  A work-group that took several
// groups in turn to reuse the topology kept more alive across them (125 and 76
// registers) and was slower at both sizes, 27.0 and 51.3 us.
template <typename R, int GA, bool Fast>
__global__ __launch_bounds__(kTileCells) void transport_kernel(LevelArgs<R> a_by_value, ChemConst K_by_value) {
  const LevelArgs<R>& a = kernargs<R>().a;
  CellLds<R>& lds = *cell_lds<R>();
  const int tile = block_tile(a), lc = (int)threadIdx.x, g = (int)blockIdx.y;
  if (tile < 0) return;
  HaloCell hl;
  R T[4], H[4];
  const CellFaces cf = cell_faces(a, tile, lc, lds, hl, g, T, H);
  transport_group<R, GA, Fast>(a, cf, hl, tile, lc, lds, g, T, H);
  if (!cf.valid || cf.restricted) return;
  const size_t o = (size_t)g * a.ncell;
  gst(a.eo + o, cf.cell, T[0]);
  gst(a.fxo + o, cf.cell, T[1]);
  gst(a.fyo + o, cf.cell, T[2]);
  gst(a.fzo + o, cf.cell, T[3]);
  // COARSERAD: a split cell's check (a leaf's is the chemistry's)
  if (cf.ch >= 0 && ((g == 0 && (T[0] < R(0) || isnan(T[0]))) || (g == 1 && isnan(T[0]))))
    raise_status(a.status, -3, a.level, cf.cell);
}

// (191 VGPRs for three FP64 groups, 208 for nine FP32 ones: held to 128 or 168
// the spills cost more than the waves bring, 62 -> 71 and 52 -> 70 us a step)
template <typename R, int G, bool Fast>
__global__ __launch_bounds__(kTileCells) void chemistry_kernel(LevelArgs<R> a_by_value, ChemConst K_by_value) {
  const KernArgs<R> args = kernargs<R>();
  const LevelArgs<R>& a = args.a;
  const int tile = block_tile(a);
  if (tile < 0) return;
  const int cell = tile * kTileCells + (int)threadIdx.x;
  unsigned int nit_acc = 0, leaf = 0;
  if (cell < a.ncell) {
    const int ch = gld(a.child, cell);
    if (a.t_first != nullptr) xion_times(a, cell);
    if (ch >= 0 && !a.update_split) {
      restrict_cell(a, cell, ch, G);
    } else if (ch >= 0) {
      gst(a.nhpluso, cell, gld(a.nhplus, cell));
      gst(a.einto, cell, gld(a.eint, cell));
      gst(a.tempo, cell, gld(a.temp, cell));
    } else {
      R Te[G], Tx[G], Ty[G], Tz[G];
#pragma unroll
      for (int g = 0; g < G; g++) {
        const size_t o = (size_t)g * a.ncell;
        Te[g] = gld(a.eo + o, cell);
        Tx[g] = gld(a.fxo + o, cell);
        Ty[g] = gld(a.fyo + o, cell);
        Tz[g] = gld(a.fzo + o, cell);
      }
      leaf = 1;
      nit_acc = (unsigned)finish_leaf<R, G, Fast, kRefluxCell>(a, args.K, cell, G, Te, Tx, Ty, Tz);
    }
  }
  if (a.counters != nullptr) block_counters<kTileWaves>(a.counters, nit_acc, leaf);
}

// ------------------------------------------------------------------ tiled level step
// Mixed precision, G fixed.  A 256-thread block owns 32 consecutive octs
// (Morton order: a 4x4x2 brick of octs on a complete level), one cell per
// thread.  With about 38 KB of LDS at G=3, four blocks share a CU, so the
// barrier phases of one block overlap the memory phases of the others.
//
// The Lax-Friedrichs flux through a face normal to d splits into one share
// per side: 2F = A(M) + B(P) with A = P + c U on the minus side and
// B = P - c U on the plus side, P the physical flux (lf_share).  So each
// cell computes its own A_d and B_d once per direction and a face costs one
// LDS read of the neighbour's share plus an add.  The block runs the three
// directions as three passes over one LDS share buffer.
//
// Neighbours outside the tile (same-level octs of other tiles, injected
// coarse leaves) are the halo.  The neighbour's share and whether the face
// flux is cancelled (split neighbour, RADSTEP) go to LDS slots of the wave,
// 64 per wave, so an in-tile and a halo face differ only in the LDS address
// read.  A complete level has 64 halo faces per wave (16 in x and y, 32 in
// z): each wave lists them (lane, direction) and evaluates them
// lane-parallel, one per lane, in one round before the direction passes
// (PerDir = false).  Sparse AMR levels have up to 192 (every cell's three
// leaving faces): there each lane evaluates its own halo face of direction d
// at the start of pass d into its own slot (PerDir = true), which needs no
// more LDS than the complete-level kernel.  The host picks the variant from
// the level's topology (the most halo faces in any wave).

// the value of lane (lane ^ m), m = 1, 2 or 4 (wave-uniform), through DPP
// lane moves within rows of 16 (VALU, no LDS): quad permutations for 1 and
// 2, a half-row mirror (lane ^ 7) followed by a quad reversal (lane ^ 3) for
// 4.  Every lane of the wave must be active.
__device__ __forceinline__ float lane_xor(float x, int m) {
  const int v = __float_as_int(x);
  if (m == 1) return __int_as_float(__builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true));  // quad_perm 1,0,3,2
  if (m == 2) return __int_as_float(__builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true));  // quad_perm 2,3,0,1
  const int t = __builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, true);                       // row_half_mirror
  return __int_as_float(__builtin_amdgcn_mov_dpp(t, 0x1B, 0xF, 0xF, true));              // quad_perm 3,2,1,0
}

// The halo variants kListed and kPerDir (rt_kernels.h) share the body below.
// one halo face: the neighbour's state, its split flag, the face direction
// and the side the neighbour lies on
template <int G>
struct HaloFace {
  float v[G][4];
  int child, d, side;
  bool lane, coarse, refl;
};

template <int G, int V>
__device__ __forceinline__ void tiled_step(const LevelArgs<float>& a, const ChemConst& K, int tile, TileLds<G>& lds,
                                           int lc) {
  constexpr bool Listed = V == kListed || V == kListedTop;
  constexpr bool PerDir = !Listed;
  constexpr bool Late = V == kPerDir;  // chemistry inputs loaded in the last direction pass
  constexpr bool NT = Listed;          // non-temporal next state and chemistry inputs (large levels)
  constexpr bool Top = V == kListedTop;  // no coarse faces on the level
  constexpr int kHaloCap = TileLds<G>::kHaloCap;  // halo slots per wave
  // shares: [g][A or B][cell] of the current direction, then the halo slots
  // [wave][slot][g]
  constexpr int kShares = G * 2 * kTileCells;
  float4* sShare = lds.share;
  // 1: the flux through the face is cancelled; [cell], then [wave][slot]
  unsigned char* sCancel = lds.cancel;
  auto& sItem = lds.item;         // halo slot -> lane*4 + direction
  auto& sItemNei = lds.item_nei;  // halo slot -> nei_oct entry of the face
  const int wv = lc >> 6, lane = lc & 63;
  const int cell = tile * kTileCells + lc;
  const int oct0 = tile * kTileOcts;
  const bool valid = cell < a.ncell;
  const int n = a.ncell;
  const float c = a.c, dts = a.dtsurdx;
  // all loads of the cell are issued first: state, child, the oct's face
  // neighbours and the chemistry inputs (their latency hides behind the
  // transport)
  const int oct = cell >> 3, ic = cell & 7;
  float Ue[G], Ux[G], Uy[G], Uz[G], Src[G];
  double pre[3] = {0., 0., 1.};  // x n_H, eint, n_H
  int noD[3] = {0, 0, 0};        // nei_oct entry of the face that leaves the oct, per direction
  int ch = -1;
  if (valid) {
    // in the order of use: topology (halo list), state, chemistry inputs
    ch = gld(a.child, cell);
#pragma unroll
    for (int d = 0; d < 3; d++) noD[d] = gld(a.nei, oct * 6 + 2 * d + ((ic >> d) & 1));
#pragma unroll
    for (int g = 0; g < G; g++) {
      Ue[g] = gld(a.e + g * n, cell);
      Ux[g] = gld(a.fx + g * n, cell);
      Uy[g] = gld(a.fy + g * n, cell);
      Uz[g] = gld(a.fz + g * n, cell);
    }
    // the chemistry inputs: early on complete levels (their latency hides
    // behind the transport); on sparse levels, whose per-direction halo
    // loads need the registers, at the start of the last direction pass
    // (load_chem below)
    if constexpr (!Late) {
#pragma unroll
      for (int g = 0; g < G; g++) Src[g] = gld_in<NT>(a.src + g * n, cell);
      pre[0] = gld_in<NT>(a.nhplus, cell);
      pre[1] = gld_in<NT>(a.eint, cell);
      pre[2] = gld_in<NT>(a.nh, cell);
    }
  }
  sCancel[lc] = (unsigned char)(ch >= 0 && !a.keep_split_flux);
  // sparse levels: the chemistry inputs of a leaf (the only cells whose step
  // runs the chemistry), issued while the last direction pass computes
  auto load_chem = [&]() {
    if (valid && ch < 0) {
#pragma unroll
      for (int g = 0; g < G; g++) Src[g] = gld(a.src + g * n, cell);
      pre[0] = gld(a.nhplus, cell);
      pre[1] = gld(a.eint, cell);
      pre[2] = gld(a.nh, cell);
    }
  };

  const bool transport = a.transport != 0;
  const bool moves = valid && transport && !(ch >= 0 && !a.update_split);
  auto in_tile = [&](int no) { return no >= oct0 && no < oct0 + kTileOcts; };
  // ---- complete levels: list the halo faces per wave
  unsigned long long hball[3] = {0ull, 0ull, 0ull};  // lanes whose face in direction d is a halo face
  int hbase[3] = {0, 0, 0};                          // first halo slot of direction d
  int nhalo = 0;
  if constexpr (!PerDir) {
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const bool out = moves && !in_tile(noD[d]);
      hball[d] = __ballot(out);
      hbase[d] = nhalo;
      nhalo += __popcll(hball[d]);
      if (out) {
        const int slot = hbase[d] + lanes_below_mask(hball[d]);  // < kHaloCap (variant chosen from the topology)
        sItem[wv][slot] = (unsigned char)(lane * 4 + d);
        sItemNei[wv][slot] = noD[d];
      }
    }
    // the list is written and read by lanes of the same wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // the neighbour across the face in direction h.d that leaves the oct of
  // cell hcell, nei_oct entry hno: a same-level cell, an injected coarse
  // leaf, or on a domain face a copy of a cell of the same oct (its normal
  // flux negated when reflective)
  auto load_neighbour = [&](HaloFace<G>& h, int hno, int hcell) {
    // only loads here: the reflective sign and nothing else that needs the
    // loaded values is applied before store_item, so the loads of several
    // faces can be in flight together
    const int hic = hcell & 7;
    h.side = (hic >> h.d) & 1;
    const bool hbound = h.lane && hno <= kNeiReflective;
    h.coarse = h.lane && hno < 0 && !hbound;
    h.refl = hbound && hno == kNeiReflective;
    const int js = hbound ? (hcell & ~7) + trans_source(2 * h.d + h.side, hic)
                          : ((h.lane && !h.coarse) ? hno * 8 + (hic ^ (1 << h.d)) : 0);
    h.child = gld(a.child, js);
    if (Top || __ballot(h.coarse) == 0) {
#pragma unroll
      for (int g = 0; g < G; g++) {
        h.v[g][0] = gld(a.e + g * n, js);
        h.v[g][1] = gld(a.fx + g * n, js);
        h.v[g][2] = gld(a.fy + g * n, js);
        h.v[g][3] = gld(a.fz + g * n, js);
      }
    } else {  // injected coarse leaves (levels with a coarser level only): per-lane arrays
      const int nc = a.ncoarse;
      const int j = h.coarse ? -1 - hno : js;
      const int st = h.coarse ? nc : n;
      // The lane's array is this level's plus a per-lane distance (0, or the
      // coarse array's address minus this level's), both pointers read
      // unconditionally by scalar loads.  A per-lane choice between the two
      // argument fields instead becomes a per-lane vector load of the pointer
      // (one more memory round trip before the data loads), or scalar loads
      // under a branch each.
      auto lane_base = [&](const float* own, const float* coarse) {
        const unsigned long long dist = (unsigned long long)coarse - (unsigned long long)own;
        return uniform_base(own) + (h.coarse ? dist : 0ull);
      };
      const EMMA_GLOBAL char* pe = lane_base(a.e, a.ce);
      const EMMA_GLOBAL char* px = lane_base(a.fx, a.cfx);
      const EMMA_GLOBAL char* py = lane_base(a.fy, a.cfy);
      const EMMA_GLOBAL char* pz = lane_base(a.fz, a.cfz);
#pragma unroll
      for (int g = 0; g < G; g++) {
        const size_t o = byte_offset<float>(g * st + j);
        h.v[g][0] = *(const EMMA_GLOBAL float*)(pe + o);
        h.v[g][1] = *(const EMMA_GLOBAL float*)(px + o);
        h.v[g][2] = *(const EMMA_GLOBAL float*)(py + o);
        h.v[g][3] = *(const EMMA_GLOBAL float*)(pz + o);
      }
    }
  };
  // complete levels: list entry `slot` (read by every lane, used by halo lanes)
  auto load_item = [&](HaloFace<G>& h, int slot) {
    h.lane = slot < nhalo;
    const int it = sItem[wv][PerDir ? 0 : slot];
    h.d = it & 3;
    load_neighbour(h, sItemNei[wv][PerDir ? 0 : slot], (cell & ~63) + (it >> 2));
  };
  // sparse levels: this lane's own face in direction d
  auto load_face = [&](HaloFace<G>& h, int d) {
    h.lane = moves && !in_tile(noD[d]);
    h.d = d;
    load_neighbour(h, noD[d], cell);
  };
  // ... the neighbour's share (a neighbour on the plus side of the face,
  // side 1, contributes B, on the minus side A) and cancel flag
  auto store_item = [&](const HaloFace<G>& h, int slot) {
    if (h.lane) {
      sCancel[kTileCells + wv * kHaloCap + slot] = (unsigned char)(!h.coarse && !a.keep_split_flux && h.child >= 0);
      // reflective face: the normal component negated (h.d differs between lanes: no indexing by it)
      const float sx = (h.refl && h.d == 0) ? -1.f : 1.f, sy = (h.refl && h.d == 1) ? -1.f : 1.f,
                  sz = (h.refl && h.d == 2) ? -1.f : 1.f;
#pragma unroll
      for (int g = 0; g < G; g++) {
        const float vx = h.v[g][1] * sx, vy = h.v[g][2] * sy, vz = h.v[g][3] * sz;
        const Closure<float> q = closure_fast(vx, vy, vz, h.v[g][0], c);
        float X[4];
        lf_share_lane(h.d, h.side ? -1.f : 1.f, h.v[g][0], vx, vy, vz, q, c, X);
        sShare[kShares + (wv * kHaloCap + slot) * G + g] = make_float4(X[0], X[1], X[2], X[3]);
      }
    }
  };
  // ---- one halo face per lane: issue the neighbour's loads ...
  // Straight-line code (every lane loads, lanes without a halo face from
  // cell 0): a load under a divergent branch makes the wait before the
  // closures below cover it as well.
  HaloFace<G> hf[1];
  if constexpr (!PerDir) load_item(hf[0], lane);
  // the reflux pairs of the cell's leaving faces that have a coarse leaf
  // behind them, loaded now for the refluxing in the direction passes
  int pairD[3] = {-1, -1, -1};
  if (valid && a.ncoarse > 0) {
#pragma unroll
    for (int d = 0; d < 3; d++)
      if (noD[d] < 0) pairD[d] = gld(a.rpair, oct * 6 + 2 * d + ((ic >> d) & 1));
  }
  // ---- ... compute this cell's closures meanwhile ...
  Closure<float> Q[G];
  if (valid) {
#pragma unroll
    for (int g = 0; g < G; g++) Q[g] = closure_fast<true>(Ux[g], Uy[g], Uz[g], Ue[g], c);
  }
  if constexpr (!PerDir) store_item(hf[0], lane);

  float De[G], Dx[G], Dy[G], Dz[G];
#pragma unroll
  for (int g = 0; g < G; g++) De[g] = Dx[g] = Dy[g] = Dz[g] = 0.f;
  float ucoef = 0.f;  // coefficient of c U summed over the directions
  if (transport) {
#pragma unroll
    for (int d = 0; d < 3; d++) {
      if constexpr (V == kPerDir) {
        load_face(hf[0], d);  // latency behind this cell's shares
        if (d == 2) load_chem();
      }
      if (valid) {
#pragma unroll
        for (int g = 0; g < G; g++) {
          float X[4];
          lf_share_unrolled(d, 1.f, Ue[g], Ux[g], Uy[g], Uz[g], Q[g], c, X);
          sShare[(g * 2 + 0) * kTileCells + lc] = make_float4(X[0], X[1], X[2], X[3]);
          lf_share_unrolled(d, -1.f, Ue[g], Ux[g], Uy[g], Uz[g], Q[g], c, X);
          sShare[(g * 2 + 1) * kTileCells + lc] = make_float4(X[0], X[1], X[2], X[3]);
        }
      }
      if constexpr (PerDir) store_item(hf[0], lane);  // own slot: written and read by this lane only
      __syncthreads();
      float Rf[G][4];  // flux through a coarse face (refluxing), 0 elsewhere
      int rj = -1;     // the coarse leaf on that face
#pragma unroll
      for (int g = 0; g < G; g++) Rf[g][0] = Rf[g][1] = Rf[g][2] = Rf[g][3] = 0.f;
      const int bit = (ic >> d) & 1;
      if (moves) {
        // Each cell has one face in d inside its oct and one leaving it; bit
        // says which is which (bit 1: the cell sits on the plus side of its
        // oct, so its minus face is the inside one).  The face on the cell's
        // minus side takes the neighbour's A plus the cell's B, the face on
        // its plus side the cell's A plus the neighbour's B.
        const int jin = lc ^ (1 << d);
        const int iin = (1 - bit) * kTileCells + jin;  // neighbour share, inside face
        const bool inT = in_tile(noD[d]);
        // (unsigned: a domain-face entry is near INT_MIN; jl and j are then unused)
        const int jl = (int)(((unsigned)noD[d] - (unsigned)oct0) * 8u + (unsigned)(ic ^ (1 << d)));
        const int slot = PerDir ? lane : hbase[d] + lanes_below_mask(hball[d]);
        const bool coarse_face = !Top && !inT && noD[d] < 0 && noD[d] > kNeiReflective;
        int iout, sout, cout;  // neighbour share, stride over groups, cancel flag: leaving face
        if (inT) {
          iout = bit * kTileCells + jl;
          sout = 2 * kTileCells;
          cout = jl;
        } else {
          iout = kShares + (wv * kHaloCap + slot) * G;
          sout = 1;
          cout = kTileCells + wv * kHaloCap + slot;
        }
        const int j = coarse_face ? -1 - noD[d] : (int)((unsigned)noD[d] * 8u + (unsigned)(ic ^ (1 << d)));
        const bool cancel_out = sCancel[cout] != 0;
        const bool cancel_in = sCancel[jin] != 0;
        const int im = bit ? iin : iout, sm = bit ? 2 * kTileCells : sout;
        const int ip = bit ? iout : iin, sp = bit ? sout : 2 * kTileCells;
        // The shares are doubled: the face fluxes are 2F_m = X_m + B and
        // 2F_p = A + X_p, with X the neighbours' shares and A = P + cU,
        // B = P - cU this cell's.  The update wm 2F_m + wp 2F_p then is
        // wm X_m + wp X_p + (wm + wp) P + (wp - wm) cU.  On complete levels
        // nearly every cell has wm = -wp (both faces carry flux, or
        // neither does): the P term drops and the cU term is summed over the
        // directions and applied once, and only the rare cell with one
        // cancelled face or a coarse face reads its own shares back.  Sparse
        // levels, where coarse faces are common, keep the plain form.
        const float wm = (bit ? cancel_in : cancel_out) ? 0.f : 0.5f * dts;
        const float wp = (bit ? cancel_out : cancel_in) ? 0.f : -0.5f * dts;
        const bool plain = !PerDir && wm == -wp;
        if (plain) ucoef += wp - wm;
#pragma unroll
        for (int g = 0; g < G; g++) {
          const float4 Xm = sShare[im + g * sm];
          const float4 Xp = sShare[ip + g * sp];
          if (!PerDir) {
            De[g] = fmaf(Xp.x, wp, fmaf(Xm.x, wm, De[g]));
            Dx[g] = fmaf(Xp.y, wp, fmaf(Xm.y, wm, Dx[g]));
            Dy[g] = fmaf(Xp.z, wp, fmaf(Xm.z, wm, Dy[g]));
            Dz[g] = fmaf(Xp.w, wp, fmaf(Xm.w, wm, Dz[g]));
          }
          if (!plain || coarse_face) {
            // this cell's shares are read back rather than held across the barrier
            const float4 Ag = sShare[(g * 2 + 0) * kTileCells + lc];
            const float4 Bg = sShare[(g * 2 + 1) * kTileCells + lc];
            const float Fm[4] = {Xm.x + Bg.x, Xm.y + Bg.y, Xm.z + Bg.z, Xm.w + Bg.w};
            const float Fp[4] = {Ag.x + Xp.x, Ag.y + Xp.y, Ag.z + Xp.z, Ag.w + Xp.w};
            if (PerDir) {
              De[g] = fmaf(Fp[0], wp, fmaf(Fm[0], wm, De[g]));
              Dx[g] = fmaf(Fp[1], wp, fmaf(Fm[1], wm, Dx[g]));
              Dy[g] = fmaf(Fp[2], wp, fmaf(Fm[2], wm, Dy[g]));
              Dz[g] = fmaf(Fp[3], wp, fmaf(Fm[3], wm, Dz[g]));
            } else if (!plain) {
              De[g] = fmaf(Ag.x, wp, fmaf(Bg.x, wm, De[g]));
              Dx[g] = fmaf(Ag.y, wp, fmaf(Bg.y, wm, Dx[g]));
              Dy[g] = fmaf(Ag.z, wp, fmaf(Bg.z, wm, Dy[g]));
              Dz[g] = fmaf(Ag.w, wp, fmaf(Bg.w, wm, Dz[g]));
            }
            if (coarse_face) {  // the flux through the coarse face, for refluxing
#pragma unroll
              for (int v = 0; v < 4; v++) Rf[g][v] = bit ? Fp[v] : Fm[v];
            }
          }
        }
        if (coarse_face) rj = j;
      }
      // Refluxing (scatterstencilrad, rad_utils.c:1738-1762): the four cells
      // of an oct face share its coarse neighbour, so their fluxes are summed
      // across lanes first (the same order every run) and each of the four
      // lanes then adds one flux component (E, Fx, Fy, Fz) of every group to
      // the face's reflux pair, whose accumulators no other lane writes (an
      // atomic add without return: the lane does not wait for the old value)
      const unsigned long long rmask = __ballot(rj >= 0);
      if (rmask != 0ull) {
        const int b1 = 1 << ((d + 1) % 3), b2 = 1 << ((d + 2) % 3);
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
          for (int v = 0; v < 4; v++) {
            float x = Rf[g][v];
            x += lane_xor(x, b1);
            x += lane_xor(x, b2);
            Rf[g][v] = x;
          }
        const int l0 = lane & ~(b1 | b2);
        const unsigned long long grp =
            (1ull << l0) | (1ull << (l0 | b1)) | (1ull << (l0 | b2)) | (1ull << (l0 | b1 | b2));
        const unsigned long long mine = rmask & grp;
        const int pr = pairD[d];
        if (rj >= 0 && pr >= 0) {
          float* acc = a.cracc + acc_at<G, kRefluxTiled>(pr, 0);
          const float w = (bit ? 1.f : -1.f) * (0.5f * dts) * 0.125f;  // pow(-1, face+1) dt/dx / 8, shares doubled
          if (mine == grp) {  // the face's four cells all carry flux (always, with 2:1 balance)
            const int k = __popcll(mine & ((1ull << lane) - 1ull));  // component of this lane
#pragma unroll
            for (int g = 0; g < G; g++) {
              const float x = k == 0 ? Rf[g][0] : (k == 1 ? Rf[g][1] : (k == 2 ? Rf[g][2] : Rf[g][3]));
              atomicAdd(acc + g * 4 + k, x * w);
            }
          } else if (lane == __builtin_ctzll(mine)) {
#pragma unroll
            for (int g = 0; g < G; g++)
#pragma unroll
              for (int v = 0; v < 4; v++) atomicAdd(acc + g * 4 + v, Rf[g][v] * w);
          }
        }
      }
      if (d < 2) __syncthreads();  // the next direction overwrites the shares
    }
    const float cu = ucoef * c;
#pragma unroll
    for (int g = 0; g < G; g++) {
      De[g] = fmaf(cu, Ue[g], De[g]);
      Dx[g] = fmaf(cu, Ux[g], Dx[g]);
      Dy[g] = fmaf(cu, Uy[g], Dy[g]);
      Dz[g] = fmaf(cu, Uz[g], Dz[g]);
    }
  }

  if constexpr (Late)
    if (!transport) load_chem();
  unsigned int nit_acc = 0, leaf = 0;
  if (valid) {
    if (a.t_first != nullptr) xion_times(a, cell);
    if (ch >= 0 && !a.update_split) {
      restrict_cell(a, cell, ch, G);
    } else {
      if (ch <= -2) fold_reflux<float, G, G, kRefluxTiled>(a, ch, 0, G, Ue, Ux, Uy, Uz);
#pragma unroll
      for (int g = 0; g < G; g++) {
        Ue[g] += De[g];
        Ux[g] += Dx[g];
        Uy[g] += Dy[g];
        Uz[g] += Dz[g];
      }
      if (ch >= 0) {
        transport_split_cell<float, G>(a, cell, G, Ue, Ux, Uy, Uz);
      } else {
        leaf = 1;
        nit_acc =
            (unsigned)finish_leaf<float, G, true, kRefluxTiled, NT>(a, K, cell, G, Ue, Ux, Uy, Uz, Src, pre);
      }
    }
  }
  if (a.counters != nullptr) block_counters<kTileWaves>(a.counters, nit_acc, leaf);
}

template <int G, bool PerDir>
__global__ __launch_bounds__(kTileCells) __attribute__((amdgpu_waves_per_eu(4))) void level_step_tiled(
    LevelArgs<float> a_by_value, ChemConst K_by_value) {
  const KernArgs<float> args = kernargs<float>();
  __shared__ TileLds<G> lds;
  const int m = args.a.raster_m;
  const int tile = m > 0 ? raster_tile(m) : block_tile(args.a);
  if (tile < 0) return;
  if constexpr (PerDir)
    tiled_step<G, kPerDir>(args.a, args.K, tile, lds, (int)threadIdx.x);
  else if (args.a.ncoarse == 0)  // wave-uniform: the level's arguments
    tiled_step<G, kListedTop>(args.a, args.K, tile, lds, (int)threadIdx.x);
  else
    tiled_step<G, kListed>(args.a, args.K, tile, lds, (int)threadIdx.x);
}

// ------------------------------------------------------------------ small levels
// A level too small to fill the GPU takes as long as one wave's chain of
// instructions: with one cell per lane and three groups, 1,800 vector
// instructions and two memory round trips took 13.9 us, one wave per SIMD.
// Here a work-group owns 64 cells (8 octs) and wave g takes photon group g of
// them, so the transport chain is a third as long and needs no barrier (a
// wave reads only its own shares); then wave 0 runs the chemistry of the 64
// cells while the others wait, and each wave scales and stores its group's
// flux.  All loads go out first: topology, then the state, the leaving faces'
// neighbours and the chemistry inputs.  The arithmetic is tiled_step's per-direction
// form, for a neighbour in the same 32-oct tile with the rounding its own share
// has there (own_share), for others with that of the halo (lf_share_lane), so
// the results are the same bit for bit.
constexpr int kSplitCells = 64;
constexpr int kSplitOcts = kSplitCells / 8;

// the share of a neighbour's state through a face normal to D: own, as
// lf_share of a closure with X2First, otherwise as lf_share_lane
template <int D>
__device__ __forceinline__ void neighbour_share(bool own, float side, const float v[4], float c, float X[4]) {
  // the two kinds of closure differ in which square of |F|^2 rounds by itself
  const float ve = v[0], vx = v[1], vy = v[2], vz = v[3];
  const float p = own ? vy : vx, q = own ? vx : vy;
  const Closure<float> Q = closure_fast_f2(vx, vy, vz, ve, c, fmaf(vz, vz, fmaf(p, p, q * q)));
  const float sc = side * c, w = Q.arg * Q.n[D];
  X[0] = fmaf(sc, ve, v[1 + D]);
#pragma unroll
  for (int i = 0; i < 3; i++) {
    float h = w * Q.n[i];
    if (i == D) {
      const float apart = Q.diag + h, fused = fmaf(w, Q.n[i], Q.diag);
      h = own ? fused : apart;
    }
    X[1 + i] = fmaf(sc, v[1 + i], h);
  }
}

template <int G>
struct SplitLds {
  float4 share[G][3][2][kSplitCells];  // [group][direction][A or B][cell]
  float e[G][kSplitCells];             // transported densities
  float fscale[G][kSplitCells];        // the chemistry's flux factors
};

template <int G>
__global__ __launch_bounds__(64 * G) void level_step_split(LevelArgs<float> a_by_value, ChemConst K_by_value) {
  const KernArgs<float> args = kernargs<float>();
  const LevelArgs<float>& a = args.a;
  const ChemConst& K = args.K;
  __shared__ SplitLds<G> lds;
  // ahead of a large level's waves that step beside it (emma_rt_coarse_step)
  __builtin_amdgcn_s_setprio(3);
  const int g = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
  const int tile = xcd_block(a.nblocks);
  const int n = a.ncell;
  const int cell = tile * kSplitCells + lane;
  const int oct = cell >> 3, ic = cell & 7;
  const int oct0 = tile * kSplitOcts, oct32 = oct0 & ~(kTileOcts - 1);
  const bool valid = cell < n;
  const bool transport = a.transport != 0;
  const float c = a.c, dts = a.dtsurdx;
  int ch = -1;
  int noD[3] = {0, 0, 0};  // nei_oct entry of the face that leaves the oct, per direction
  int pairD[3] = {-1, -1, -1};
  float U[4] = {0.f, 0.f, 0.f, 0.f};
  float Src[G];
  double pre[3] = {0., 0., 1.};  // x n_H, eint, n_H
  if (valid) {
    ch = gld(a.child, cell);
    if (transport) {
#pragma unroll
      for (int d = 0; d < 3; d++) noD[d] = gld(a.nei, oct * 6 + 2 * d + ((ic >> d) & 1));
    }
    U[0] = gld(a.e + g * n, cell);
    U[1] = gld(a.fx + g * n, cell);
    U[2] = gld(a.fy + g * n, cell);
    U[3] = gld(a.fz + g * n, cell);
    if (g == 0) {
#pragma unroll
      for (int q = 0; q < G; q++) Src[q] = gld(a.src + q * n, cell);
      pre[0] = gld(a.nhplus, cell);
      pre[1] = gld(a.eint, cell);
      pre[2] = gld(a.nh, cell);
    }
  }
  const bool restricted = ch >= 0 && !a.update_split;
  if (transport) {
    const bool moves = valid && !restricted;
    const unsigned long long cancels = __ballot(ch >= 0 && !a.keep_split_flux);
    auto in_wave = [&](int no) { return no >= oct0 && no < oct0 + kSplitOcts; };
    // the leaving faces' neighbours outside the 64 cells, every load at once
    // (lanes without one read cell 0)
    float hv[3][4];
    int hchild[3];
    bool hon[3], hcoarse[3], hrefl[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const int side = (ic >> d) & 1, no = noD[d];
      const bool on = moves && !in_wave(no);
      const bool bound = on && no <= kNeiReflective;  // domain face
      const bool coarse = on && no < 0 && !bound;
      hon[d] = on;
      hcoarse[d] = coarse;
      hrefl[d] = bound && no == kNeiReflective;
      const int js = bound ? (cell & ~7) + trans_source(2 * d + side, ic)
                           : (on && !coarse ? no * 8 + (ic ^ (1 << d)) : 0);
      hchild[d] = gld(a.child, js);
      if (__ballot(coarse) == 0ull) {
        hv[d][0] = gld(a.e + g * n, js);
        hv[d][1] = gld(a.fx + g * n, js);
        hv[d][2] = gld(a.fy + g * n, js);
        hv[d][3] = gld(a.fz + g * n, js);
      } else {
        // injected coarse leaves: the lane's array is this level's plus a
        // per-lane distance (0, or the coarse array's address minus this
        // level's), both bases read by scalar loads
        const size_t o = (size_t)(coarse ? -1 - no : js) * sizeof(float);
        auto lane_load = [&](const float* own, const float* coarser) {
          const float* const ob = own + (size_t)g * n;
          const float* const cb = coarser + (size_t)g * a.ncoarse;
          const unsigned long long dist = (unsigned long long)cb - (unsigned long long)ob;
          return *(const EMMA_GLOBAL float*)(uniform_base(ob) + (coarse ? dist : 0ull) + o);
        };
        hv[d][0] = lane_load(a.e, a.ce);
        hv[d][1] = lane_load(a.fx, a.cfx);
        hv[d][2] = lane_load(a.fy, a.cfy);
        hv[d][3] = lane_load(a.fz, a.cfz);
      }
    }
    if (valid && a.ncoarse > 0) {
#pragma unroll
      for (int d = 0; d < 3; d++)
        if (noD[d] < 0) pairD[d] = gld(a.rpair, oct * 6 + 2 * d + ((ic >> d) & 1));
    }
    // this cell's shares of the three directions
    const Closure<float> Q = closure_fast<true>(U[1], U[2], U[3], U[0], c);
#pragma unroll
    for (int d = 0; d < 3; d++) {
      float X[4];
      lf_share_unrolled(d, 1.f, U[0], U[1], U[2], U[3], Q, c, X);
      lds.share[g][d][0][lane] = make_float4(X[0], X[1], X[2], X[3]);
      lf_share_unrolled(d, -1.f, U[0], U[1], U[2], U[3], Q, c, X);
      lds.share[g][d][1][lane] = make_float4(X[0], X[1], X[2], X[3]);
    }
    // written and read by lanes of the same wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float D[4] = {0.f, 0.f, 0.f, 0.f};
    auto direction = [&](auto dd) {
      constexpr int d = decltype(dd)::value;
      const int bit = (ic >> d) & 1, jin = lane ^ (1 << d), no = noD[d];
      const bool inW = in_wave(no);
      const int jl = (int)(((unsigned)no - (unsigned)oct0) * 8u + (unsigned)(ic ^ (1 << d))) & (kSplitCells - 1);
      float Rf[4] = {0.f, 0.f, 0.f, 0.f};
      int rj = -1;
      // the neighbour's share across the leaving face: a neighbour on the
      // plus side contributes B, on the minus side A
      const float4 sin = lds.share[g][d][1 - bit][jin], sout = lds.share[g][d][bit][jl];
      if (hrefl[d]) hv[d][1 + d] = -hv[d][1 + d];
      float X[4];
      neighbour_share<d>(no >= oct32 && no < oct32 + kTileOcts, bit ? -1.f : 1.f, hv[d], c, X);
      if (moves) {
        const float Xin[4] = {sin.x, sin.y, sin.z, sin.w};
        const float Xout[4] = {inW ? sout.x : X[0], inW ? sout.y : X[1], inW ? sout.z : X[2], inW ? sout.w : X[3]};
        const bool cancel_in = (cancels >> jin) & 1ull;
        const bool cancel_out = inW ? (bool)((cancels >> jl) & 1ull)
                                    : (hon[d] && !hcoarse[d] && !a.keep_split_flux && hchild[d] >= 0);
        const float wm = (bit ? cancel_in : cancel_out) ? 0.f : 0.5f * dts;
        const float wp = (bit ? cancel_out : cancel_in) ? 0.f : -0.5f * dts;
        const bool coarse_face = hcoarse[d];
        const float4 Ag = lds.share[g][d][0][lane], Bg = lds.share[g][d][1][lane];
        const float A[4] = {Ag.x, Ag.y, Ag.z, Ag.w}, B[4] = {Bg.x, Bg.y, Bg.z, Bg.w};
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const float Fm = (bit ? Xin[v] : Xout[v]) + B[v];
          const float Fp = A[v] + (bit ? Xout[v] : Xin[v]);
          D[v] = fmaf(Fp, wp, fmaf(Fm, wm, D[v]));
          if (coarse_face) Rf[v] = bit ? Fp : Fm;
        }
        if (coarse_face) rj = -1 - no;
      }
      // refluxing, as in tiled_step
      const unsigned long long rmask = __ballot(rj >= 0);
      if (rmask != 0ull) {
        const int b1 = 1 << ((d + 1) % 3), b2 = 1 << ((d + 2) % 3);
#pragma unroll
        for (int v = 0; v < 4; v++) {
          float x = Rf[v];
          x += lane_xor(x, b1);
          x += lane_xor(x, b2);
          Rf[v] = x;
        }
        const int l0 = lane & ~(b1 | b2);
        const unsigned long long grp =
            (1ull << l0) | (1ull << (l0 | b1)) | (1ull << (l0 | b2)) | (1ull << (l0 | b1 | b2));
        const unsigned long long mine = rmask & grp;
        const int pr = pairD[d];
        if (rj >= 0 && pr >= 0) {
          float* acc = a.cracc + acc_at<G, kRefluxTiled>(pr, g);
          const float w = (bit ? 1.f : -1.f) * (0.5f * dts) * 0.125f;  // pow(-1, face+1) dt/dx / 8, shares doubled
          if (mine == grp) {
            const int k = __popcll(mine & ((1ull << lane) - 1ull));  // component of this lane
            const float x = k == 0 ? Rf[0] : (k == 1 ? Rf[1] : (k == 2 ? Rf[2] : Rf[3]));
            atomicAdd(acc + k, x * w);
          } else if (lane == __builtin_ctzll(mine)) {
#pragma unroll
            for (int v = 0; v < 4; v++) atomicAdd(acc + v, Rf[v] * w);
          }
        }
      }
    };
    direction(std::integral_constant<int, 0>());
    direction(std::integral_constant<int, 1>());
    direction(std::integral_constant<int, 2>());
    if (valid && !restricted) {
      if (ch <= -2) fold_reflux<float, G, 1, kRefluxTiled>(a, ch, g, 1, &U[0], &U[1], &U[2], &U[3]);
#pragma unroll
      for (int v = 0; v < 4; v++) U[v] += D[v];
    }
  } else if (valid && !restricted && ch <= -2) {
    fold_reflux<float, G, 1, kRefluxTiled>(a, ch, g, 1, &U[0], &U[1], &U[2], &U[3]);
  }
  const bool leaf = valid && ch < 0;
  if (G > 1) {
    lds.e[g][lane] = U[0];
    __syncthreads();
  }
  if (g == 0) {
    if (valid && a.t_first != nullptr) xion_times(a, cell);
    int nit = 0;
    if (leaf) {
      double e[G], src[G], fscale[G];
#pragma unroll
      for (int q = 0; q < G; q++) {
        e[q] = (double)(G > 1 ? lds.e[q][lane] : U[0]);
        src[q] = (double)Src[q];
      }
      if (e[0] < 0 || isnan(e[0]) || isnan(G > 1 ? e[G > 1 ? 1 : 0] : (double)U[1]))
        raise_status(a.status, -3, a.level, cell);
      double nhplus = pre[0], eint = pre[1], temp = 0.;
      int st = chem_cell_fast<G>(K, G, e, fscale, src, nhplus, eint, pre[2], temp, a.chemonly, nit,
                                 a.chem_budget > 0 ? a.chem_budget : -1, (double)a.chem_keep);
      const bool deferred = defer_leaf(a, cell, st, nit);
      if (st != 0) raise_status(a.status, st, a.level, cell);
#pragma unroll
      for (int q = 0; q < G; q++) {
        float ev = (float)e[q];
        if (!deferred && e[q] >= K.emin_grp[q] && ev < K.emin_grp_up[q]) ev = K.emin_grp_up[q];
        gst(a.eo + q * n, cell, ev);
        lds.fscale[q][lane] = (float)fscale[q];
      }
      gst(a.nhpluso, cell, nhplus);
      gst(a.einto, cell, eint);
      gst(a.tempo, cell, temp);
    } else if (valid && restricted) {
      restrict_scalars(a, cell, ch);
    } else if (valid) {  // COARSERAD: a split cell with its transported state
      gst(a.nhpluso, cell, gld(a.nhplus, cell));
      gst(a.einto, cell, gld(a.eint, cell));
      gst(a.tempo, cell, gld(a.temp, cell));
    }
    if (a.counters != nullptr) {
      const unsigned long long lb = __ballot(leaf);
      unsigned int s0 = 0;
#pragma unroll
      for (int b = 0; b < 4; b++) s0 += (unsigned int)__popcll(__ballot(((unsigned)nit >> b) & 1u)) << b;
      unsigned long long* slot = a.counters + (size_t)(blockIdx.x % kCounterSlots) * kCounterStride;
      if (nit >= 16) atomicAdd(slot, (unsigned long long)((unsigned)nit & ~15u));
      if (lane == 0) {
        atomicAdd(slot + 0, (unsigned long long)s0);
        atomicAdd(slot + 1, (unsigned long long)__popcll(lb));
      }
    }
  }
  if (valid && restricted) restrict_group(a, cell, ch, g);  // meanwhile: split cells wait for nothing
  if (G > 1) __syncthreads();
  if (leaf) {
    const float fs = lds.fscale[g][lane];
    gst(a.fxo + g * n, cell, U[1] * fs);
    gst(a.fyo + g * n, cell, U[2] * fs);
    gst(a.fzo + g * n, cell, U[3] * fs);
  } else if (valid && !restricted) {
    gst(a.eo + g * n, cell, U[0]);
    gst(a.fxo + g * n, cell, U[1]);
    gst(a.fyo + g * n, cell, U[2]);
    gst(a.fzo + g * n, cell, U[3]);
    if ((g == 0 && (U[0] < 0.f || isnan(U[0]) || (G == 1 && isnan(U[1])))) || (g == 1 && isnan(U[0])))
      raise_status(a.status, -3, a.level, cell);
  }
}

// ------------------------------------------------------------------ chemistry stragglers
// The leaves the tiled kernel put on the straggler list (sub-step loop still
// running after chem_budget tries) take their whole chemistry here, one
// thread each, from the same inputs: the transported N, F the tiled kernel
// stored into the next state, the source and x n_H, eint, n_H of the current
// state.  A wave then holds 64 long loops instead of one long loop among 63
// finished lanes.  Each level-step launch has its own list-length word
// (cleared by the host before the call), so nothing is reset here.
template <int G>
__global__ __launch_bounds__(kStragglerThreads) void chem_straggler_kernel(LevelArgs<float> a_by_value,
                                                                            ChemConst K_by_value) {
  const KernArgs<float> args = kernargs<float>();
  const LevelArgs<float>& a = args.a;
  const ChemConst& K = args.K;
  const int count = min(*(volatile const int*)a.defer_ctl, a.defer_cap);
  const int n = a.ncell;
  unsigned int nit_acc = 0, ncell_acc = 0;
  for (int i = blockIdx.x * kStragglerThreads + (int)threadIdx.x; i < count; i += gridDim.x * kStragglerThreads) {
    ncell_acc++;
    const int cell = gld(a.defer_list, i);
    double e[G], src[G], fscale[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
      e[g] = (double)gld(a.eo + g * n, cell);
      src[g] = (double)gld(a.src + g * n, cell);
    }
    double nhplus = gld(a.nhplus, cell), eint = gld(a.eint, cell), temp = 0.;
    const double nh = gld(a.nh, cell);
    int nit = 0;
    const int st = chem_cell_fast<G>(K, G, e, fscale, src, nhplus, eint, nh, temp, a.chemonly, nit);
    if (st != 0) raise_status(a.status, st, a.level, cell);
    nit_acc += (unsigned)nit;
#pragma unroll
    for (int g = 0; g < G; g++) {
      float ev = (float)e[g];
      if (e[g] >= K.emin_grp[g] && ev < K.emin_grp_up[g]) ev = K.emin_grp_up[g];
      const float fs = (float)fscale[g];
      const float fx = gld(a.fxo + g * n, cell) * fs, fy = gld(a.fyo + g * n, cell) * fs,
                  fz = gld(a.fzo + g * n, cell) * fs;
      gst(a.eo + g * n, cell, ev);
      gst(a.fxo + g * n, cell, fx);
      gst(a.fyo + g * n, cell, fy);
      gst(a.fzo + g * n, cell, fz);
    }
    gst(a.nhpluso, cell, nhplus);
    gst(a.einto, cell, eint);
    gst(a.tempo, cell, temp);
  }
  if (a.counters != nullptr) {
    // one atomic per wave that did work
    for (int o = 32; o > 0; o >>= 1) {
      nit_acc += __shfl_xor(nit_acc, o, 64);
      ncell_acc += __shfl_xor(ncell_acc, o, 64);
    }
    unsigned long long* slot = a.counters + (size_t)(blockIdx.x % kCounterSlots) * kCounterStride;
    if ((threadIdx.x & 63) == 0 && ncell_acc != 0u) {
      atomicAdd(slot, (unsigned long long)nit_acc);
      atomicAdd(slot + 2, (unsigned long long)ncell_acc);
    }
  }
}

// ------------------------------------------------------------------ COARSERAD transfers
// One thread per split cell of the coarse level and component (blockIdx.y: E,
// Fx, Fy, Fz of each group), which walks the cell's subtree depth first,
// children in index order like the reference's recursion (collectE,
// src_utils.c:94-123; distribE, rad_utils.c:26-45), so every sum has its order.
//
// Bound by the chain of dependent loads of the largest subtree: an oct's eight
// child entries and eight values (32 or 64 B, aligned) come in one round trip,
// and once more on the way back from each split child.  One thread per coarse
// cell, all components in turn and cell by cell, took 93 us up and 72 us down
// on a tree of 4,096 cells with 302 and 70 octs below them, three FP32 groups;
// now 15 and 18.  The coupled coarse step there 222 -> 81 us, of 32^3 cells
// with 1,500, 6,000 and 20,000 octs below them 2079 -> 379 us (FP64 2368 ->
// 442).
constexpr int kTransferThreads = 64;
template <typename R, bool Put>
__global__ __launch_bounds__(kTransferThreads) void coarse_transfer_kernel(TreeView<R> t) {
  __shared__ const int* sChild[kMaxLevels];
  __shared__ R* sVal[kMaxLevels];
  __shared__ long long sStack[kMaxLevels][kTransferThreads];  // oct * 16 + the next child to visit
  const int tid = (int)threadIdx.x, v = (int)blockIdx.y & 3, g = (int)blockIdx.y >> 2;
#pragma unroll
  for (int k = 0; k < kMaxLevels; k++) {
    if (tid == k) {
      sChild[k] = t.child[k];
      sVal[k] = (v == 0 ? t.e[k] : v == 1 ? t.fx[k] : v == 2 ? t.fy[k] : t.fz[k]) + (size_t)g * t.ncell[k];
    }
  }
  __syncthreads();
  const int i = (int)blockIdx.x * kTransferThreads + tid;
  if (i >= t.nsplit) return;
  const int cell0 = t.split[i];
  R acc = Put ? R(0) : sVal[0][cell0];
  int k = 1, oct = sChild[0][cell0], next = 0;
  while (true) {
    typedef int IntV __attribute__((ext_vector_type(4)));
    typedef R ValV __attribute__((ext_vector_type(16 / sizeof(R))));
    constexpr int kPer = 16 / sizeof(R);
    const IntV* pc = (const IntV*)(sChild[k] + (size_t)oct * 8);
    ValV* pv = (ValV*)(sVal[k] + (size_t)oct * 8);
    const IntV c0 = pc[0], c1 = pc[1];
    ValV x[8 / kPer];
    if (Put) {
#pragma unroll
      for (int q = 0; q < 8 / kPer; q++) x[q] = pv[q];
    }
    const R fact = (R)ldexp(1.0, -3 * k);  // pow(2, 3 (lcoarse - level))
    int down = -1, at = 8;
    bool stored = false;
    if (!Put) {
      const IntV m = c0 & c1;
      stored = next == 0 && (m[0] & m[1] & m[2] & m[3]) < 0;  // eight leaves
      if (stored) {
#pragma unroll
        for (int q = 0; q < 8 / kPer; q++) pv[q] = (ValV)acc;
      }
    }
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int ch = j < 4 ? c0[j & 3] : c1[j & 3];
      if (j >= next && at == 8) {
        if (ch >= 0) {
          if (k + 1 < t.nlev) {  // (else a split cell on the last level: no children stored)
            at = j;
            down = ch;
          }
        } else if (Put) {
          acc += x[j / kPer][j % kPer] * fact;
        } else if (!stored) {
          ((R*)pv)[j] = acc;
        }
      }
    }
    if (at < 8) {
      sStack[k][tid] = (long long)oct * 16 + at + 1;
      k++;
      oct = down;
      next = 0;
      continue;
    }
    // back to the nearest level with children left
    do {
      if (--k < 1) break;
      const long long s = sStack[k][tid];
      oct = (int)(s >> 4);
      next = (int)(s & 15);
    } while (next == 8);
    if (k < 1) break;
  }
  if (Put) sVal[0][cell0] = acc;
}

template <typename R, bool Put>
static hipError_t launch_transfer(const TreeView<R>& t, hipStream_t s) {
  if (t.nsplit == 0) return hipSuccess;
  const dim3 grid((t.nsplit + kTransferThreads - 1) / kTransferThreads, 4 * t.ng);
  hipLaunchKernelGGL((coarse_transfer_kernel<R, Put>), grid, dim3(kTransferThreads), 0, s, t);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_put_e2coarse(const TreeView<R>& t, hipStream_t s) {
  return launch_transfer<R, true>(t, s);
}

template <typename R>
hipError_t launch_distrib_e(const TreeView<R>& t, hipStream_t s) {
  return launch_transfer<R, false>(t, s);
}

template hipError_t launch_put_e2coarse<double>(const TreeView<double>&, hipStream_t);
template hipError_t launch_put_e2coarse<float>(const TreeView<float>&, hipStream_t);
template hipError_t launch_distrib_e<double>(const TreeView<double>&, hipStream_t);
template hipError_t launch_distrib_e<float>(const TreeView<float>&, hipStream_t);

// ------------------------------------------------------------------ photon budget
// FP64 sum over leaf cells of sum_g N_g * dx^3 (wavefront shuffles, one
// atomic per block)
template <typename R>
__global__ __launch_bounds__(256) void photon_sum_kernel(const R* e, const int* child, int ncell, int ng, double vol,
                                                         double* out) {
  double s = 0.;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < ncell; i += gridDim.x * 256) {
    if (child[i] < 0)
      for (int g = 0; g < ng; g++) s += (double)e[g * ncell + i];
  }
  s *= vol;
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(out, red[0] + red[1] + red[2] + red[3]);
}

// small fill kernel (used instead of hipMemsetAsync so that the work can sit
// inside a captured graph)
__global__ void fill_kernel(unsigned int* p, int n, unsigned int v) {
  int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}

// The end of a call: one work-group sums the counter slots (a slot per thread),
// reports them with the status words to the host and clears all call words for
// the next call.  The flag is stored last, at system scope.
__global__ __launch_bounds__(kCounterSlots) void call_end_kernel(int* status, unsigned long long* counters,
                                                                 int* defer_ctl, int ndefer, CallRecord* rec) {
  __shared__ unsigned long long red[3][kCounterSlots / 64];
  const int t = (int)threadIdx.x;
  if (counters != nullptr) {
    unsigned long long* slot = counters + (size_t)t * kCounterStride;
    unsigned long long v[3];
#pragma unroll
    for (int k = 0; k < 3; k++) v[k] = slot[k];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      slot[k] = 0ull;
      for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o, 64);
      if ((t & 63) == 0) red[k][t >> 6] = v[k];
    }
  }
  for (int i = t; i < ndefer; i += kCounterSlots) defer_ctl[i] = 0;
  __syncthreads();
  if (t == 0) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      unsigned long long sum = 0ull;
      if (counters != nullptr)
        for (int w = 0; w < kCounterSlots / 64; w++) sum += red[k][w];
      rec->counts[k] = sum;
      rec->status[k] = status[k];
      status[k] = 0;
    }
    __hip_atomic_store(&rec->flag, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// ------------------------------------------------------------------ persistent coarse step
// The schedule's read-only tables are read through the constant address
// space: at a wave-uniform index the loads are scalar loads, and the level
// step's arguments inside a StepDesc stay in SGPRs like kernel arguments.
#define EMMA_CONST __attribute__((address_space(4)))
template <typename T>
__device__ __forceinline__ const T& cref(const void* base, int i) {
  return *(const T*)((const EMMA_CONST T*)base + i);
}

__device__ __forceinline__ const SchedArgs& sched_args() {
  return *reinterpret_cast<const SchedArgs*>((const char*)__builtin_amdgcn_kernarg_segment_ptr());
}

// wait until ticket dt is done in this launch (epoch), bounded by wall-clock
// time: past the bound the wait is abandoned with EMMA_RT_ERR_SCHED, and
// once that status is raised no other wait starts, so that every work-group
// ends within about one bound
__device__ __forceinline__ void wait_done(const SchedArgs& s, int dt, int epoch) {
  if (__hip_atomic_load(s.done + dt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch) return;
  const long long t0 = (long long)__builtin_amdgcn_s_memrealtime();
  while (__hip_atomic_load(s.done + dt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != epoch) {
    if (__hip_atomic_load(s.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == kErrSched) return;
    __builtin_amdgcn_s_sleep(2);
    if ((long long)__builtin_amdgcn_s_memrealtime() - t0 > s.wait_ticks) {
      raise_status(s.status, kErrSched, -1, dt);
      return;
    }
  }
}

template <int G>
__device__ __forceinline__ TileLds<G>* tile_lds() {
  __shared__ TileLds<G> lds;
  return &lds;
}

// The thread index as a value the optimiser cannot see through: otherwise
// every address and mask the item derives from it alone is hoisted out of
// the work-group's ticket loop and held in registers across all items.
__device__ __forceinline__ int opaque_thread() {
  int t = (int)threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// one tile of an item: FillRad's block on the tile's cells, the tile's
// level step, the hydro injection of its cells.  Each thread fills and
// injects the cell it steps, so the three need no barrier between them;
// neighbours' cells are read only for their N, F and split flags, which
// FillRad does not touch.
template <typename R, int G, bool Tiled, bool Coupled>
__device__ __forceinline__ void run_item(const StepDesc<R>& D, int tile) {
  const int lc = opaque_thread();
  const int cell = tile * kTileCells + lc;
  if constexpr (Coupled)
    if (D.fill && cell < D.f.ncell) fill_cell<R>(D.f, cell);
  if constexpr (Tiled) {
    if (D.variant == kListed)
      tiled_step<G, kListed>(D.a, D.K, tile, *tile_lds<G>(), lc);
    else
      tiled_step<G, kPerDir>(D.a, D.K, tile, *tile_lds<G>(), lc);
  } else {
    cell_step<R, G, sizeof(R) == 4>(D.a, D.K, tile, lc);
  }
  if constexpr (Coupled)
    if (D.hydro && cell < D.h.ncell) to_hydro_cell(D.h, cell);
}

// Work-groups loop over tickets of their XCD's queue (the XCC_ID hardware
// register names the XCD): take the next one, wait for the tickets it
// depends on (lanes of wave 0, one dependency each), acquire at agent scope,
// run the item, release, mark the ticket done.  The release writes the L2
// back (agent scope) only for items with a dependent in another queue:
// within a queue the producer's stores are in the XCD's shared L2 once they
// have completed.  One wave of the work-group does the acquire and the
// release for all four.  Items on the schedule's critical path run at a
// raised wave priority so that the bandwidth-bound items sharing their SIMDs
// do not stretch the chain.  The last work-group to leave re-arms the queues
// (tickets 0, next epoch) for the next launch.  Coupled: FillRad's block and
// the hydro injection are compiled in (without them the kernel needs fewer
// registers).
//
// The work-group's own bookkeeping (ticket, done flag, exit count) is done
// by all of wave 0 under a wave-uniform branch, never by one lane: a
// lane-divergent block at each end of a loop that holds barriers lets the
// compiler split the loop by lane (thread 0 looping over tickets, the other
// lanes over the old ticket), which never ends.
template <typename R, int G, bool Tiled, bool Coupled>
__global__ __launch_bounds__(kTileCells) __attribute__((amdgpu_waves_per_eu(Tiled ? 4 : 1))) void persistent_step_kernel(
    SchedArgs s_by_value) {
  const SchedArgs& s = sched_args();
  __shared__ int sTicket, sEpoch;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = (int)threadIdx.x & 63;
  // the queue of this work-group's XCD
  int xcc;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
  const int q = s.xcc_queue[xcc & 15];
  // (an XCD the library did not see serves no queue)
  const int qb = q >= 0 ? cref<int>(s.qoff, q) : 0, qn = q >= 0 ? cref<int>(s.qoff, q + 1) - qb : 0;
  if (wave == 0) sEpoch = __hip_atomic_load(s.ctl + s.nq + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  int epoch = 0;
  for (;;) {
    if (wave == 0) {  // lane 0 adds one, the other lanes nothing
      const int old = q >= 0 ? atomicAdd(s.ctl + q, lane == 0 ? 1 : 0) : 0;
      sTicket = __builtin_amdgcn_readfirstlane(old);
    }
    __syncthreads();
    const int tq = __builtin_amdgcn_readfirstlane(sTicket);
    epoch = __builtin_amdgcn_readfirstlane(sEpoch);
    if (tq >= qn) break;
    const int t = qb + tq;
    const int flags = cref<unsigned char>(s.item_flags, t);
    const int d0 = cref<int>(s.dep_off, t), d1 = cref<int>(s.dep_off, t + 1);
    if (d1 > d0) {
      if (wave == 0) {
        for (int i = d0 + lane; i < d1; i += 64) wait_done(s, s.deps[i], epoch);
        // one acquire at agent scope for the work-group (its waves share
        // this CU's caches), also for dependencies on this XCD's items: an
        // L1-only invalidate (buffer_inv sc0) left same-XCD results stale in
        // measurements, the agent-scope invalidate does not
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      }
      __syncthreads();
    }
    const int step = cref<int>(s.item_step, t), tile = cref<int>(s.item_tile, t);
    const int ntile = cref<int>(s.item_ntile, t);
    const int prio = flags & kItemPrio;
    if (prio) __builtin_amdgcn_s_setprio(2);
    for (int k = 0; k < ntile; k++) {
      if (k > 0) __syncthreads();  // the tile step's LDS is reused
      run_item<R, G, Tiled, Coupled>(cref<StepDesc<R>>(s.steps, step), tile + k);
    }
    if (prio) __builtin_amdgcn_s_setprio(0);
    // every wave's stores have reached the L2 before wave 0 publishes the
    // ticket; for readers on other XCDs it writes the L2 back first (release
    // at agent scope)
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (wave == 0) {
      if (flags & kItemReleaseAgent) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      __hip_atomic_store(s.done + t, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (wave == 0) {
    const int left = __builtin_amdgcn_readfirstlane(atomicAdd(s.ctl + s.nq, lane == 0 ? 1 : 0));
    if (left == (int)gridDim.x - 1) {
      for (int i = lane; i < s.nq + 1; i += 64) s.ctl[i] = 0;
      if (lane == 0) s.ctl[s.nq + 1] = epoch + 1;
    }
  }
}

// ------------------------------------------------------------------ launchers
constexpr unsigned kCuLds = 160 * 1024;
static_assert(sizeof(TileLds<3>) < kCuLds / 4, "four work-groups a CU");
template <int G>
static void launch_split(LevelArgs<float> a, const ChemConst& K, hipStream_t s) {
  a.nblocks = ((a.ncell + kSplitCells - 1) / kSplitCells + 7) & ~7;
  hipLaunchKernelGGL((level_step_split<G>), dim3(a.nblocks), dim3(64 * G), 0, s, a, K);
}

hipError_t launch_stragglers(const LevelArgs<float>& a, const ChemConst& K, hipStream_t s) {
  // the list holds at most the level's cells
  const dim3 grid(std::min(kStragglerBlocks, (a.ncell + kStragglerThreads - 1) / kStragglerThreads));
  if (a.ng == 1)
    hipLaunchKernelGGL((chem_straggler_kernel<1>), grid, dim3(kStragglerThreads), 0, s, a, K);
  else
    hipLaunchKernelGGL((chem_straggler_kernel<3>), grid, dim3(kStragglerThreads), 0, s, a, K);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_level_step(const LevelArgs<R>& a0, const ChemConst& K, bool stragglers, hipStream_t s) {
  LevelArgs<R> a = a0;
  if constexpr (sizeof(R) == 4) {
    if (a.ng == 1 || a.ng == 3) {
      int nb = a.tiles ? a.ntiles : (a.ncell + kTileCells - 1) / kTileCells;
      nb = (nb + 7) & ~7;
      a.nblocks = nb;
      // sparse levels: per-direction halo faces
      const int v = a.variant;
      const bool defer = a.chem_budget > 0;
      if (defer && (a.defer_list == nullptr || a.defer_ctl == nullptr || a.defer_cap < a.ncell))
        return hipErrorInvalidValue;
      // beside smaller levels' launches: LDS beyond a quarter of a CU's, so that
      // three work-groups instead of four share it and the small ones start at once
      const unsigned share = a.leave_room ? kCuLds / 4 + 256 - (unsigned)sizeof(TileLds<3>) : 0u;
      if (a.ng == 1) {
        if (v == kLatency)
          launch_split<1>(a, K, s);
        else if (v == kPerDir)
          hipLaunchKernelGGL((level_step_tiled<1, true>), dim3(nb), dim3(kTileCells), 0, s, a, K);
        else
          hipLaunchKernelGGL((level_step_tiled<1, false>), dim3(nb), dim3(kTileCells), 0, s, a, K);
      } else {
        if (v == kLatency)
          launch_split<3>(a, K, s);
        else if (v == kPerDir)
          hipLaunchKernelGGL((level_step_tiled<3, true>), dim3(nb), dim3(kTileCells), share, s, a, K);
        else
          hipLaunchKernelGGL((level_step_tiled<3, false>), dim3(nb), dim3(kTileCells), share, s, a, K);
      }
      const hipError_t e = hipGetLastError();
      return e == hipSuccess && defer && stragglers ? launch_stragglers(a, K, s) : e;
    }
  }
  int nb = a.tiles ? a.ntiles : (a.ncell + kTileCells - 1) / kTileCells;
  nb = (nb + 7) & ~7;
  a.nblocks = nb;
  const dim3 grid(nb), block(kTileCells);
  constexpr bool fast = sizeof(R) == 4;
  if constexpr (!fast) {
    if (a.ng == 1) {
      hipLaunchKernelGGL(level_step_kernel, grid, block, 0, s, a, K);
      return hipGetLastError();
    }
  }
  const dim3 tgrid(nb, a.ng);
  bool three = false;
  if constexpr (!fast) {  // (three FP32 groups took the tiled kernel)
    three = a.ng == 3;
    if (three) hipLaunchKernelGGL((transport_kernel<R, 3, fast>), tgrid, block, 0, s, a, K);
  }
  if (!three) hipLaunchKernelGGL((transport_kernel<R, kMaxGrp, fast>), tgrid, block, 0, s, a, K);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  switch (a.ng) {
#define EMMA_CHEM(g) \
  case g: hipLaunchKernelGGL((chemistry_kernel<R, g, fast>), grid, block, 0, s, a, K); break
    EMMA_CHEM(2);
    EMMA_CHEM(4);
    EMMA_CHEM(5);
    EMMA_CHEM(6);
    EMMA_CHEM(7);
    EMMA_CHEM(8);
    EMMA_CHEM(9);
#undef EMMA_CHEM
    default:
      if constexpr (!fast) {
        if (a.ng == 3) {
          hipLaunchKernelGGL((chemistry_kernel<R, 3, fast>), grid, block, 0, s, a, K);
          break;
        }
      }
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

__global__ void xcc_probe_kernel(int* out, int n) {
  int xcc;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
  if (threadIdx.x == 0 && (int)blockIdx.x < n) out[blockIdx.x] = xcc & 15;
}

hipError_t launch_xcc_probe(int* out, int n, hipStream_t st) {
  hipLaunchKernelGGL(xcc_probe_kernel, dim3(n), dim3(64), 0, st, out, n);
  return hipGetLastError();
}

template <typename R, int G, bool Tiled>
static void* persistent_kernel_of(bool coupled) {
  return coupled ? reinterpret_cast<void*>(persistent_step_kernel<R, G, Tiled, true>)
                 : reinterpret_cast<void*>(persistent_step_kernel<R, G, Tiled, false>);
}
template <typename R>
static void* persistent_kernel(int ng, bool coupled) {
  if constexpr (sizeof(R) == 4) {
    if (ng == 1) return persistent_kernel_of<float, 1, true>(coupled);
    if (ng == 3) return persistent_kernel_of<float, 3, true>(coupled);
    return persistent_kernel_of<float, 0, false>(coupled);
  } else {
    if (ng == 1) return persistent_kernel_of<double, 1, false>(coupled);
    if (ng == 3) return persistent_kernel_of<double, 3, false>(coupled);
    return persistent_kernel_of<double, 0, false>(coupled);
  }
}

template <typename R>
int persistent_blocks_per_cu(int ng, bool coupled) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, persistent_kernel<R>(ng, coupled), kTileCells, 0) != hipSuccess)
    return 0;
  return n;
}

template <typename R>
hipError_t launch_persistent(const SchedArgs& s, int ng, bool coupled, int nblocks, hipStream_t st) {
  void* args[] = {const_cast<SchedArgs*>(&s)};
  return hipLaunchKernel(persistent_kernel<R>(ng, coupled), dim3(nblocks), dim3(kTileCells), args, 0, st);
}

template <typename R>
hipError_t launch_photon_sum(const R* e, const int* child, int ncell, int ng, double vol, double* out,
                             hipStream_t s) {
  int nb = (ncell + 255) / 256;
  if (nb > 2048) nb = 2048;
  if (nb < 1) nb = 1;
  hipLaunchKernelGGL((photon_sum_kernel<R>), dim3(nb), dim3(256), 0, s, e, child, ncell, ng, vol, out);
  return hipGetLastError();
}

hipError_t launch_fill(unsigned int* p, int n, unsigned int v, hipStream_t s) {
  hipLaunchKernelGGL(fill_kernel, dim3((n + 255) / 256), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

hipError_t launch_call_end(int* status, unsigned long long* counters, int* defer_ctl, int ndefer, CallRecord* rec,
                           hipStream_t s) {
  hipLaunchKernelGGL(call_end_kernel, dim3(1), dim3(kCounterSlots), 0, s, status, counters, defer_ctl, ndefer, rec);
  return hipGetLastError();
}

template hipError_t launch_level_step<double>(const LevelArgs<double>&, const ChemConst&, bool, hipStream_t);
template hipError_t launch_level_step<float>(const LevelArgs<float>&, const ChemConst&, bool, hipStream_t);
template int persistent_blocks_per_cu<double>(int, bool);
template int persistent_blocks_per_cu<float>(int, bool);
template hipError_t launch_persistent<double>(const SchedArgs&, int, bool, int, hipStream_t);
template hipError_t launch_persistent<float>(const SchedArgs&, int, bool, int, hipStream_t);
template hipError_t launch_photon_sum<double>(const double*, const int*, int, int, double, double*, hipStream_t);
template hipError_t launch_photon_sum<float>(const float*, const int*, int, int, double, double*, hipStream_t);

}  // namespace emma
