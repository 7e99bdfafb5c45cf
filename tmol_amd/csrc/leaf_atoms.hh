// Missing leaf atoms of a pose stack (hydrogens, carbonyl oxygens): each is
// built from three resolved ancestors and its ideal internal coordinates,
// with a backup ancestor set where the first is absent (gen_pose_leaf_atoms).
//
// Reference: tmol/io/details/compiled/gen_pose_leaf_atoms.impl.hh:25-336,
// leaf_atoms.hh:11-100; tmol/score/common/uaid_util.hh:110-205 (atoms named
// across inter-block connections), gen_coord.hh (build_coordinate).
#pragma once

#include "ljlk_common.hh"
#include "lkball.hh"

namespace tmol_ljlk {

// padded pose layout of the op boundary
struct LeafArgs {
  int P, NA, B, Amax, C;
  const uint8_t* block_missing;   // [P, B, Amax] atom not given
  const uint8_t* pose_missing;    // [P, NA]
  const int32_t* block_offset;    // [P, B]
  const int32_t* block_type;      // [P, B]
  const int32_t* irc;             // [P, B, C, 2] inter-block connections
  const int32_t* n_atoms;         // [T]
  const int32_t* downstream;      // [T, C, Amax] atoms downstream of each connection
  const int32_t* anc;             // [T, Amax, 3, 3] (atom, conn, bonds from conn)
  const int32_t* anc_backup;
  const void* geom;               // [T, Amax, 3] phi, theta, d
  const void* geom_backup;
};

// Bits of *failed, in the order the host reports them: every index that the
// kernels below follow lies inside its table.  The last two index with values
// that the first ones check, so they are tested only where those are sound
// (and reported only when none of the first failed).
//
// Bound by the two launches and the read-back of one word: the tables of
// 256 poses of 50-600 residues are 5 MB, read once.  The same checks as
// elementwise tensor operations took 60 launches, 300 us of device time and
// two read-backs per call.
constexpr uint32_t LEAF_BAD_TYPE = 1, LEAF_BAD_N = 2, LEAF_BAD_DOWN = 4, LEAF_BAD_ANC = 8,
                   LEAF_BAD_CONN = 32, LEAF_BAD_OFFSET = 64, LEAF_BAD_PARTNER = 128;

__device__ __forceinline__ bool leaf_outside(int v, int lo, int n) { return v < lo || v >= n; }

__global__ __launch_bounds__(256) void leaf_check_kernel(LeafArgs a, int T, uint32_t* failed) {
  const int64_t i0 = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t step = int64_t(gridDim.x) * blockDim.x;
  uint32_t bad = 0;
  for (int64_t t = i0; t < T; t += step)
    if (leaf_outside(a.n_atoms[t], 0, a.Amax + 1)) bad |= LEAF_BAD_N;
  for (int64_t i = i0; i < int64_t(T) * a.C * a.Amax; i += step)
    if (leaf_outside(a.downstream[i], -1, a.n_atoms[i / (int64_t(a.C) * a.Amax)]))
      bad |= LEAF_BAD_DOWN;
  for (int64_t i = i0; i < int64_t(T) * a.Amax * 3; i += step) {
    const int n = a.n_atoms[i / (int64_t(a.Amax) * 3)];
    for (int k = 0; k < 2; ++k) {
      const int32_t* u = (k ? a.anc_backup : a.anc) + 3 * i;
      if (leaf_outside(u[0], -1, n) || leaf_outside(u[1], -1, a.C) ||
          (u[1] >= 0 && leaf_outside(u[2], 0, a.Amax)))
        bad |= LEAF_BAD_ANC << k;
    }
  }
  for (int64_t q = i0; q < int64_t(a.P) * a.B; q += step) {
    const int bt = a.block_type[q];
    if (leaf_outside(bt, -1, T)) {
      bad |= LEAF_BAD_TYPE;
    } else if (bt >= 0) {
      const int off = a.block_offset[q];
      if (off < 0 || int64_t(off) + a.n_atoms[bt] > a.NA) bad |= LEAF_BAD_OFFSET;
    }
    const int32_t* row = a.block_type + (q / a.B) * a.B;
    for (int c = 0; c < a.C; ++c) {
      const int ob = a.irc[(q * a.C + c) * 2], oc = a.irc[(q * a.C + c) * 2 + 1];
      if (leaf_outside(ob, -1, a.B) || (ob >= 0 && leaf_outside(oc, 0, a.C)))
        bad |= LEAF_BAD_CONN;
      else if (ob >= 0 && row[ob] < 0)
        bad |= LEAF_BAD_PARTNER;
    }
  }
  if (bad) atomicOr(failed, bad);
}

// pose-wide index of an unresolved atom id of block b (-1: none)
__device__ __forceinline__ int leaf_resolve(const LeafArgs& a, int p, int b, const int32_t* u) {
  if (u[0] != -1) return a.block_offset[p * a.B + b] + u[0];
  if (u[1] == -1) return -1;
  const int32_t* c = a.irc + ((int64_t(p) * a.B + b) * a.C + u[1]) * 2;
  const int ob = c[0];
  if (ob == -1) return -1;
  const int obt = a.block_type[p * a.B + ob];
  const int idx = a.downstream[(int64_t(obt) * a.C + c[1]) * a.Amax + u[2]];
  if (idx < 0) return -1;
  return a.block_offset[p * a.B + ob] + idx;
}

// a row of an ancestor table: three atom ids (atom, conn, bonds from conn),
// loaded whole (two 16-byte loads and one word instead of nine words)
struct LeafRow {
  int32_t v[9];
  // an ancestor named across a connection
  __device__ __forceinline__ bool remote() const {
    return (v[0] == -1 && v[1] != -1) || (v[3] == -1 && v[4] != -1) || (v[6] == -1 && v[7] != -1);
  }
};
__device__ __forceinline__ LeafRow leaf_row(const int32_t* table, int64_t row) {
  LeafRow r;
  __builtin_memcpy(&r, table + row * 9, sizeof r);
  return r;
}

// the three ancestors (pose-local indices) of atom slot `at` of a block of
// type bt, for each its atom slot in the same block or -1 when named across a
// connection, and the geometry (phi, theta, d): the primary set, else the
// backup, else none (false)
template <typename Real>
__device__ __forceinline__ bool leaf_ancestors(const LeafArgs& a, int p, int b, int64_t row,
                                               const LeafRow& primary, int* anc, int* slot,
                                               Real* geom) {
  LeafRow u = primary;
  for (int k = 0; k < 2; ++k) {
    if (k) u = leaf_row(a.anc_backup, row);
    bool ok = true;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      anc[j] = leaf_resolve(a, p, b, u.v + 3 * j);
      slot[j] = u.v[3 * j];
      ok = ok && anc[j] != -1;
    }
    if (!ok) continue;
    const uint8_t* miss = a.pose_missing + int64_t(p) * a.NA;
    __builtin_memcpy(geom, (const Real*)(k ? a.geom_backup : a.geom) + row * 3, 3 * sizeof(Real));
    if (!(miss[anc[0]] | miss[anc[1]] | miss[anc[2]])) return true;
  }
  return false;
}

// what an atom slot's work starts from: loads that need the block's type
// alone, issued together (the kernels wait on chains of loads, not on
// bandwidth), and held by `ready` before the first branch on them
struct LeafSlot {
  int n_at, off, miss;
  LeafRow row;
  __device__ __forceinline__ LeafSlot(const LeafArgs& a, int q, int bt, int at) {
    n_at = a.n_atoms[bt];
    off = a.block_offset[q];
    miss = a.block_missing[int64_t(q) * a.Amax + at];
    row = leaf_row(a.anc, int64_t(bt) * a.Amax + at);
  }
  __device__ __forceinline__ void ready() {
    asm volatile("" : "+v"(n_at), "+v"(off), "+v"(miss), "+v"(row.v[0]), "+v"(row.v[4]),
                 "+v"(row.v[8]));
  }
};

template <typename Real>
__device__ __forceinline__ bool any_nan(Vec3<Real> v) {
  return v.x != v.x || v.y != v.y || v.z != v.z;
}

// Launch shape of all three kernels: one wave per workgroup (its barriers
// are wave barriers, reached by the whole workgroup whatever the wave's
// trip count).  Wave w owns the LEAF_BPW blocks q = LEAF_BPW w ... of the flat
// (pose, block) grid: it loads their types, keeps the real ones (a ballot)
// and takes them G = 64 / Amax at a time (Amax <= 64: lane = g * Amax + atom
// slot), or one at a time with lanes striding over the atom slots (Amax >
// 64).  Padding blocks cost one load per LEAF_BPW.
constexpr int LEAF_WAVE = 64;
// blocks whose types one wave loads.  The kernels wait on chains of dependent
// loads, so two passes per wave keep more chains in flight than sixteen
// blocks' eight; fewer repeat the launch and the type load.  Build / backward
// local / remote, 256 poses of 50-600 residues: 2 blocks 42 / 59 / 42 us, 4
// 38 / 54 / 39, 8 41 / 56 / 43, 16 46 / 59 / 54 (one after another with their
// loads instead of together: 51 / 64 / 52).
constexpr int LEAF_BPW = 4;
constexpr int LEAF_MAX_ATOMS = 2048;  // larger block types: ENOTSUP

struct LeafPass {
  int g;       // this lane's block of the pass (-1: none)
  int q;       // its flat (pose, block) index
  int bt;      // its block type
  int at0;     // first atom slot of this lane
  int stride;  // atom-slot stride (past Amax when one slot per lane)
};

__device__ __forceinline__ int leaf_blocks_per_pass(const LeafArgs& a) {
  return a.Amax <= LEAF_WAVE ? LEAF_WAVE / a.Amax : 1;
}

// this lane's block in the pass that takes the lowest blocks of `real`
__device__ __forceinline__ LeafPass leaf_pass(const LeafArgs& a, uint64_t real, int64_t q0,
                                              int bt_lane, int lane) {
  const int G = leaf_blocks_per_pass(a);
  LeafPass r;
  const bool small = a.Amax <= LEAF_WAVE;
  const int g = small ? lane / a.Amax : 0;
  r.at0 = small ? lane - g * a.Amax : lane;
  r.stride = small ? (1 << 30) : LEAF_WAVE;  // small: one slot per lane
  uint64_t m = real;
  for (int k = 0; k < g && m; ++k) m &= m - 1;
  const int pos = (g < G && m) ? __ffsll((unsigned long long)m) - 1 : -1;
  const int bt = __shfl(bt_lane, pos < 0 ? 0 : pos, LEAF_WAVE);
  r.g = pos < 0 ? -1 : g;
  r.q = pos < 0 ? -1 : int(q0 + pos);
  r.bt = pos < 0 ? -1 : bt;
  return r;
}

__device__ __forceinline__ uint64_t leaf_drop(const LeafArgs& a, uint64_t real) {
  const int G = leaf_blocks_per_pass(a);
  for (int k = 0; k < G && real; ++k) real &= real - 1;
  return real;
}

// given atoms are copied, missing ones built (NaN when no complete ancestor
// set exists)
template <typename Real>
__global__ __launch_bounds__(LEAF_WAVE) void leaf_atoms_kernel(LeafArgs a, const Real* orig,
                                                               Real* out) {
  const int lane = threadIdx.x;
  const int64_t nblk = int64_t(a.P) * a.B;
  for (int64_t w = blockIdx.x; w * LEAF_BPW < nblk; w += gridDim.x) {
    const int64_t q0 = w * LEAF_BPW;
    const int bt_lane = lane < LEAF_BPW && q0 + lane < nblk ? a.block_type[q0 + lane] : -1;
    uint64_t real = __ballot(bt_lane >= 0);
    while (real) {
      const LeafPass r = leaf_pass(a, real, q0, bt_lane, lane);
      real = leaf_drop(a, real);
      if (r.g < 0) continue;
      const int p = r.q / a.B, b = r.q - p * a.B;
      for (int at = r.at0; at < a.Amax; at += r.stride) {
        LeafSlot s(a, r.q, r.bt, at);
        s.ready();
        if (at >= s.n_at) continue;
        const int64_t dst = int64_t(p) * a.NA + s.off + at;
        Real* o = out + 3 * dst;
        if (!s.miss) {
          o[0] = orig[3 * dst];
          o[1] = orig[3 * dst + 1];
          o[2] = orig[3 * dst + 2];
          continue;
        }
        int anc[3], slot[3];
        Real g[3];
        Vec3<Real> W = {Real(NAN), Real(NAN), Real(NAN)};
        if (leaf_ancestors(a, p, b, int64_t(r.bt) * a.Amax + at, s.row, anc, slot, g)) {
          const Real* base = orig + 3 * int64_t(p) * a.NA;
          const Vec3<Real> A = v3(base + 3 * anc[0]), B = v3(base + 3 * anc[1]),
                           C = v3(base + 3 * anc[2]);
          if (!any_nan(A) && !any_nan(B) && !any_nan(C)) {
            Vec3<Real> e0, e1, e2;
            water_frame(A, B, C, e0, e1, e2);
            const WaterCoef<Real> c = water_coef(g[2], g[1], g[0]);
            W = {A.x + c.k0 * e0.x + c.k1 * e1.x + c.k2 * e2.x,
                 A.y + c.k0 * e0.y + c.k1 * e1.y + c.k2 * e2.y,
                 A.z + c.k0 * e0.z + c.k1 * e1.z + c.k2 * e2.z};
          }
        }
        o[0] = W.x;
        o[1] = W.y;
        o[2] = W.z;
      }
    }
  }
}

// the ancestor shares of the atom at slot `at` of block q if it is built
// (false otherwise, or without ancestors or with an absent coordinate; with
// REMOTE_ONLY also when every ancestor is in the same block)
template <typename Real, bool REMOTE_ONLY>
__device__ __forceinline__ bool leaf_shares(const LeafArgs& a, const Real* orig,
                                            const Real* dnew, int q, int bt, int at,
                                            const LeafSlot& s, int* anc, int* slot,
                                            Vec3<Real>* gs) {
  if (!s.miss) return false;
  const int p = q / a.B, b = q - p * a.B;
  Real g[3];
  if (!leaf_ancestors(a, p, b, int64_t(bt) * a.Amax + at, s.row, anc, slot, g)) return false;
  if (REMOTE_ONLY && slot[0] >= 0 && slot[1] >= 0 && slot[2] >= 0) return false;
  const int64_t base = int64_t(p) * a.NA;
  const Vec3<Real> A = v3(orig + 3 * (base + anc[0])), B = v3(orig + 3 * (base + anc[1])),
                   C = v3(orig + 3 * (base + anc[2]));
  if (any_nan(A) || any_nan(B) || any_nan(C)) return false;
  const int64_t dst = base + s.off + at;
  build_coord_vjp(A, B, C, water_coef(g[2], g[1], g[0]), v3(dnew + 3 * dst), gs[0], gs[1],
                  gs[2]);
  return true;
}

// Backward, first kernel: a pass's blocks sum the shares their built atoms
// send to ancestors in the same block in LDS (dynamic, 3 x max(64, Amax)
// per wave), then write each atom once: its own gradient if given, plus the
// sum.  Shares sent across a connection are added by the second kernel,
// with global atomics, after the first has written every atom.
template <typename Real>
__global__ __launch_bounds__(LEAF_WAVE) void leaf_atoms_backward_local_kernel(
    LeafArgs a, const Real* orig, const Real* dnew, Real* dorig) {
  extern __shared__ unsigned char leaf_lds[];
  Real* acc = (Real*)leaf_lds;
  const int lane = threadIdx.x;
  const int W = a.Amax <= LEAF_WAVE ? LEAF_WAVE : a.Amax;  // entries per component
  const int64_t nblk = int64_t(a.P) * a.B;
  for (int64_t w = blockIdx.x; w * LEAF_BPW < nblk; w += gridDim.x) {
    const int64_t q0 = w * LEAF_BPW;
    const int bt_lane = lane < LEAF_BPW && q0 + lane < nblk ? a.block_type[q0 + lane] : -1;
    uint64_t real = __ballot(bt_lane >= 0);
    while (real) {
      const LeafPass r = leaf_pass(a, real, q0, bt_lane, lane);
      real = leaf_drop(a, real);
      for (int i = lane; i < 3 * W; i += LEAF_WAVE) acc[i] = Real(0);
      __syncthreads();
      const int gbase = r.g < 0 ? 0 : r.g * a.Amax;
      const int n_slots = r.g < 0 ? 0 : a.Amax;
      for (int at = r.at0; at < n_slots; at += r.stride) {
        LeafSlot s(a, r.q, r.bt, at);
        s.ready();
        if (at >= s.n_at) continue;
        int anc[3], slot[3];
        Vec3<Real> gs[3];
        if (!leaf_shares<Real, false>(a, orig, dnew, r.q, r.bt, at, s, anc, slot, gs)) continue;
        for (int j = 0; j < 3; ++j) {
          if (slot[j] < 0) continue;
          const int e = gbase + slot[j];
          atomicAdd(&acc[e], gs[j].x);
          atomicAdd(&acc[W + e], gs[j].y);
          atomicAdd(&acc[2 * W + e], gs[j].z);
        }
      }
      __syncthreads();
      if (r.g >= 0) {
        const int p = r.q / a.B;
        const int64_t off = int64_t(p) * a.NA + a.block_offset[r.q];
        const int n_at = a.n_atoms[r.bt];
        for (int at = r.at0; at < n_at; at += r.stride) {
          const int64_t dst = off + at;
          const int e = gbase + at;
          const bool given = !a.block_missing[int64_t(r.q) * a.Amax + at];
          dorig[3 * dst] = (given ? dnew[3 * dst] : Real(0)) + acc[e];
          dorig[3 * dst + 1] = (given ? dnew[3 * dst + 1] : Real(0)) + acc[W + e];
          dorig[3 * dst + 2] = (given ? dnew[3 * dst + 2] : Real(0)) + acc[2 * W + e];
        }
      }
      __syncthreads();
    }
  }
}

template <typename Real>
__global__ __launch_bounds__(LEAF_WAVE) void leaf_atoms_backward_remote_kernel(
    LeafArgs a, const Real* orig, const Real* dnew, Real* dorig) {
  const int lane = threadIdx.x;
  const int64_t nblk = int64_t(a.P) * a.B;
  for (int64_t w = blockIdx.x; w * LEAF_BPW < nblk; w += gridDim.x) {
    const int64_t q0 = w * LEAF_BPW;
    const int bt_lane = lane < LEAF_BPW && q0 + lane < nblk ? a.block_type[q0 + lane] : -1;
    uint64_t real = __ballot(bt_lane >= 0);
    while (real) {
      const LeafPass r = leaf_pass(a, real, q0, bt_lane, lane);
      real = leaf_drop(a, real);
      if (r.g < 0) continue;
      const int64_t base = int64_t(r.q / a.B) * a.NA;
      for (int at = r.at0; at < a.Amax; at += r.stride) {
        LeafSlot s(a, r.q, r.bt, at);
        const LeafRow backup = leaf_row(a.anc_backup, int64_t(r.bt) * a.Amax + at);
        s.ready();
        // most atoms hang from their own block whichever set they take: the
        // tables say so before any ancestor is looked up
        if (at >= s.n_at || !(s.row.remote() || backup.remote())) continue;
        int anc[3], slot[3];
        Vec3<Real> gs[3];
        if (!leaf_shares<Real, true>(a, orig, dnew, r.q, r.bt, at, s, anc, slot, gs)) continue;
        for (int j = 0; j < 3; ++j) {
          if (slot[j] >= 0) continue;
          Real* d = dorig + 3 * (base + anc[j]);
          unsafeAtomicAdd(&d[0], gs[j].x);
          unsafeAtomicAdd(&d[1], gs[j].y);
          unsafeAtomicAdd(&d[2], gs[j].z);
        }
      }
    }
  }
}

}  // namespace tmol_ljlk
