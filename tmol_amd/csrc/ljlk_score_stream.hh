// Streaming scoring kernel (blocks of at most 32 atoms; whole-pose energies
// and the weighted gradient): one wave walks one row of the work list -- block
// g1 against its neighbor blocks g2 > g1 -- but treats the row's g2 atoms as
// one stream instead of block pair by block pair.
//
//   descriptors  64 neighbor blocks at a time, one per lane: type, atom
//                offset, atom count, minimum bond separation and, for blocks
//                within 4 bonds, the connection separations; an exclusive scan
//                of the atom counts places each block's atoms in the stream
//   raw chunk    64 consecutive stream atoms, one per lane: the lane finds its
//                block from per-chunk start markers and a ballot, loads the
//                atom and culls it against g1's sphere (an atom farther than
//                r1 + max_dis from g1's centre reaches no atom of g1); the
//                survivors are staged into the current test chunk
//   test chunk   32 survivors held in LDS ring slots (three chunks of 32 live
//                at a time); lanes 0..31 and 32..63 hold the same 32 atoms
//                and test them against g1 atoms t and t + 1: squared
//                distance and, only in chunks holding atoms within 4 bonds
//                of g1, the count-pair separation from precombined path
//                bytes.  In-range pairs of non-zero weight are
//                ballot-compacted into the pair FIFO
//   phase B      64 FIFO entries at a time, one per lane: LJ, and elec in the
//                fused mode (its 5.5 A reach lies inside LJ's 6 A, so a pair's
//                distance, LDS reads and gradient sums are shared); the
//                heavy-heavy entries among them, about a quarter, are
//                compacted again into the LK FIFO, evaluated 64 at a time.
//                Gradients accumulate in LDS as 64-bit fixed point and a ring
//                chunk is flushed to global memory when its slots are reused,
//                g1 at row end
//
// Per block pair the row kernel pays staging, a cull of both blocks and
// bookkeeping; here that work is per 64 atoms of the stream, and the pair
// tests read g2 atoms from registers and g1 atoms by LDS broadcast.  The
// separation of a pair is min(5, min_c1 pd1[c1] + q[c1]) with
// q[c1] = min_c2 cs[c1][c2] + pd2[c2] combined once per g2 atom (absent
// connections carry path distance 6, so their sums never reach below 5), the
// count-pair rule of impl.hh:47-67 / count_pair.hh:162-207.
//
// A wave takes a part of a row: A.part_shift > 0 splits every row's items into
// 2^part_shift parts, so that a batch with fewer rows than resident waves
// still fills the chip (see row_part_shift).
//
// Bound: VALU issue.  LDS (40 KB a workgroup: four of them fill a CU's 160 KB)
// and 128 VGPRs both hold the gradient modes at 4 waves per SIMD.
#pragma once

#include "ljlk_score_rows.hh"

namespace tmol_ljlk {

constexpr int SCH = 32;                // atoms per test chunk
constexpr int SRING = 3 * SCH;         // ring slots
constexpr int SSLOTS = TILE + SRING;   // g1 slots 0..31, ring 32..127
constexpr int SLIST = 128;             // FIFO capacity (drained at 64)
constexpr uint32_t Q_NONE = 0x64646464u;  // q bytes of blocks more than 4 bonds apart (100)
constexpr uint32_t Q_LIG = 0x00800000u;   // bit 7 of byte 2: ligand-fragment block

// Gradient accumulators: one entry per slot, and a second copy of g1's for odd
// lanes: LDS atomics on one address serialize, and consecutive FIFO entries
// share their g1 atom.  Ring slots stay single (a second copy of them costs a
// workgroup per CU).  All in one row per component, so an entry's three
// atomics differ by constant offsets.
constexpr int GROW = SSLOTS + TILE;

// FIFO entry: g1 slot (5 bits) | second slot (7 bits) | LJ / LK weight code
// << 12 | elec weight code << 14; code 0: weight 1, 1: 0.2, 2: no contribution
constexpr int CODE_LJ = 12, CODE_EL = 14;
constexpr int CODE_NONE = 2;

template <typename Real, int MODE>
struct StreamLDS {
  using C = RowCtx<Real, MODE>;
  using T = typename LdsAcc<Real>::T;
  static constexpr int NGP = C::NG > 0 ? C::NG : 1;
  T grad[NGP][3][C::DERIV ? GROW : 1];
  alignas(4 * sizeof(Real)) Real pos[SSLOTS][4];  // x, y, z, lj_radius
  alignas(4 * sizeof(Real)) Real prm[SSLOTS][4];  // K, 1/lambda^2, lk_volume, charge
  alignas(2 * sizeof(Real)) Real lj2[SSLOTS][2];  // sqrt(lj_wdepth), flags (pack_flags)
  uint16_t lj[SLIST];    // pair FIFO; its upper half holds the test chunk's tq
  uint16_t lk[SLIST];    // LK FIFO; its upper half holds the raw chunk's marks
  int32_t atom[SRING];   // global atom of each ring slot
  uint32_t pd1[TILE];    // g1 atoms' connection path distances, byte per connection
  uint32_t epd1[C::ELEC ? TILE : 1];  // elec's
  uint32_t teq[C::ELEC ? SCH : 1];    // test chunk atoms: elec's connection bytes
  // both FIFOs hold fewer than 64 entries outside phase B and the test loop
  // (which reads tq before it appends)
  __device__ __forceinline__ uint32_t* tq() { return (uint32_t*)(lj + WAVE); }
  __device__ __forceinline__ uint8_t* mark() { return (uint8_t*)(lk + WAVE); }
};
static_assert(SCH * 4 <= 2 * (SLIST - WAVE) && WAVE <= 2 * (SLIST - WAVE), "aliased FIFO halves");

__device__ __forceinline__ float pack_flags(int f, float) { return __int_as_float(f); }
__device__ __forceinline__ double pack_flags(int f, double) { return double(f); }
__device__ __forceinline__ int unpack_flags(float v) { return __float_as_int(v); }
__device__ __forceinline__ int unpack_flags(double v) { return int(v); }

// count-pair weight of a 2-bit code
template <typename Real>
__device__ __forceinline__ Real code_weight(int code) {
  return code == 0 ? Real(1) : (code == 1 ? Real(0.2) : Real(0));
}

// smallest of the four 7-bit byte fields of v, capped at 5 (the count-pair
// separation from packed sums)
__device__ __forceinline__ int min_sep_bytes(uint32_t v) {
  const int b0 = v & 127, b1 = (v >> 8) & 127, b2 = (v >> 16) & 127, b3 = (v >> 24) & 127;
  const int m = min(min(b0, b1), min(b2, b3));
  return m < 5 ? m : 5;
}

// q[c1] = min_c2 (cs[c1][c2] + pd2[c2]) as bytes, cs row c1 packed (byte c2)
__device__ __forceinline__ uint32_t combine_q(const uint32_t cs[MAX_CONN], uint32_t pd2) {
  uint32_t q = 0;
#pragma unroll
  for (int c1 = 0; c1 < MAX_CONN; ++c1) {
    const uint32_t s = cs[c1] + pd2;  // bytes <= 12: no carries
    const uint32_t b0 = s & 255, b1 = (s >> 8) & 255, b2 = (s >> 16) & 255, b3 = s >> 24;
    const uint32_t m = min(min(b0, b1), min(b2, b3));
    q |= m << (8 * c1);
  }
  return q;
}

// gradient gs (x1 - x2) of an entry's pair: + to the g1 atom's slot s1 (odd
// lanes: its second copy), - to slot s2 (a ring slot, or a g1 slot for
// intra-block pairs)
template <typename Real, int MODE>
__device__ __forceinline__ void stream_scatter(StreamLDS<Real, MODE>& L, int term, int s1, int s2,
                                               Real gs, Real dx, Real dy, Real dz, int odd) {
  using Acc = LdsAcc<Real>;
  using T = typename Acc::T;
  const Real g = gs * Acc::SCALE;
  const T ex = Acc::enc_scaled(g * dx), ey = Acc::enc_scaled(g * dy), ez = Acc::enc_scaled(g * dz);
  T* b1 = &L.grad[term][0][s1 + odd];
  T* b2 = &L.grad[term][0][s2];
  atomicAdd(b1, ex);
  atomicAdd(b1 + GROW, ey);
  atomicAdd(b1 + 2 * GROW, ez);
  Acc::sub(b2, ex);
  Acc::sub(b2 + GROW, ey);
  Acc::sub(b2 + 2 * GROW, ez);
}

// one atom's accumulated gradient component to global memory
template <typename Real, int MODE>
__device__ __forceinline__ void flush_value(const ScoreArgs<Real>& A, int t, int64_t i,
                                            typename LdsAcc<Real>::T acc) {
  using C = RowCtx<Real, MODE>;
  if (C::DET) {
    if (acc != 0) atomicAdd(&A.fixed[int64_t(t) * A.n_atoms * 3 + i], acc);
    return;
  }
  const Real v = LdsAcc<Real>::dec(acc);
  if (v != Real(0)) {
    if (C::DVDX)
      unsafeAtomicAdd(&A.dvdx[int64_t(t) * A.n_atoms * 3 + i], v);
    else
      unsafeAtomicAdd(&A.grad[i], v);
  }
}

// flush the gradients of ring chunk r (n atoms, slots TILE + SCH r ...) to
// their atoms and zero them; lane l takes component l % 3 of atom l / 3
template <typename Real, int MODE>
__device__ __forceinline__ void flush_chunk(StreamLDS<Real, MODE>& L, const ScoreArgs<Real>& A,
                                            int r, int n, int lane) {
  using C = RowCtx<Real, MODE>;
  if (!C::DERIV) return;
  for (int i = lane; i < 3 * n; i += WAVE) {
    const int a = i / 3, k = i - 3 * a;
    const int64_t atom = L.atom[SCH * r + a];
#pragma unroll
    for (int t = 0; t < C::NG; ++t) {
      auto* g = &L.grad[t][k][TILE + SCH * r + a];
      const auto acc = *g;
      *g = 0;
      flush_value<Real, MODE>(A, t, atom * 3 + k, acc);
    }
  }
}

// g1's atoms [0, n) (slots 0..n-1 and their copies, contiguous atoms from atom0)
template <typename Real, int MODE>
__device__ __forceinline__ void flush_g1(StreamLDS<Real, MODE>& L, const ScoreArgs<Real>& A, int n,
                                         int64_t atom0, int lane) {
  using C = RowCtx<Real, MODE>;
  if (!C::DERIV) return;
  for (int i = lane; i < 3 * n; i += WAVE) {
    const int a = i / 3, k = i - 3 * a;
#pragma unroll
    for (int t = 0; t < C::NG; ++t) {
      auto* g = &L.grad[t][k][a];
      const auto acc = g[0] + g[SSLOTS];
      g[0] = g[SSLOTS] = 0;
      flush_value<Real, MODE>(A, t, atom0 * 3 + i, acc);
    }
  }
}

// running energies of one lane's entries
struct StreamEnergies {
  LaneSum atr, rep, lk, el;
};

// LK entries [0, consume) of the FIFO, consume <= 64, one per lane
template <typename Real, int MODE>
__device__ __forceinline__ void stream_lk(StreamLDS<Real, MODE>& L, int consume,
                                          const GlobalParams<Real>& gp, const Real* wrow,
                                          StreamEnergies& en, int lane, int odd) {
  using C = RowCtx<Real, MODE>;
  using V = typename V4<Real>::T;
  if (lane >= consume) return;
  const int e = L.lk[lane];
  const int s1 = e & 31, s2 = (e >> 5) & 127;
  const Real wcp = (e >> CODE_LJ) & 1 ? Real(0.2) : Real(1);
  const V p1 = *(const V*)L.pos[s1], p2 = *(const V*)L.pos[s2];
  const V q1 = *(const V*)L.prm[s1], q2 = *(const V*)L.prm[s2];
  const int f1 = unpack_flags(L.lj2[s1][1]), f2 = unpack_flags(L.lj2[s2][1]);
  const Real dx = p1.x - p2.x, dy = p1.y - p2.y, dz = p1.z - p2.z;
  const Real d2 = dx * dx + dy * dy + dz * dz;
  const Real inv_d = fast_rsqrt(d2);
  const Real dist = d2 > Real(0) ? d2 * inv_d : Real(0);  // coincident atoms: d = 0
  const Real sigma = lj_sigma(f1, f2, p1.w, p2.w, gp);
  const bool cc = (f1 & F_CARBON_LK) && (f2 & F_CARBON_LK);
  Real d_min, cdmin, cdmax;
  lk_knots(sigma, cc, d_min, cdmin, cdmax);
  const LkSide<Real> side[2] = {{-q2.z * q1.x, p1.w, q1.y}, {-q1.z * q2.x, p2.w, q2.y}};
  Real v, dv;
  lk_sides<Real, C::DERIV>(dist, d_min, cdmin, cdmax, side, gp, v, dv);
  if (!C::NOE) en.lk.add(wcp * v);
  if (C::DERIV && dist > Real(0)) {
    Real gs = wcp * dv;
    if (gs != Real(0)) {
      gs *= inv_d;
      if (C::WGRAD) gs *= wrow[2];
      stream_scatter<Real, MODE>(L, C::DVDX ? 2 : 0, s1, s2, gs, dx, dy, dz, odd);
    }
  }
}

// pair entries [0, consume) of the FIFO, consume <= 64, one per lane: LJ (and
// elec); returns whether this lane's entry (in *entry) goes on to LK
template <typename Real, int MODE>
__device__ __forceinline__ bool stream_pairs(StreamLDS<Real, MODE>& L, int consume,
                                             const GlobalParams<Real>& gp,
                                             const ElecConst<Real>& ek, const Real* wrow, Real wel,
                                             StreamEnergies& en, int lane, int odd, int* entry) {
  using C = RowCtx<Real, MODE>;
  using V = typename V4<Real>::T;
  if (lane >= consume) return false;
  const int e = L.lj[lane];
  *entry = e;
  const int s1 = e & 31, s2 = (e >> 5) & 127;
  const V p1 = *(const V*)L.pos[s1], p2 = *(const V*)L.pos[s2];
  const Real se1 = L.lj2[s1][0], se2 = L.lj2[s2][0];
  const int f1 = unpack_flags(L.lj2[s1][1]), f2 = unpack_flags(L.lj2[s2][1]);
  const int code = C::ELEC ? (e >> CODE_LJ) & 3 : (e >> CODE_LJ) & 1;
  const Real dx = p1.x - p2.x, dy = p1.y - p2.y, dz = p1.z - p2.z;
  const Real d2 = dx * dx + dy * dy + dz * dz;
  const Real inv_d = fast_rsqrt(d2);
  const Real dist = d2 > Real(0) ? d2 * inv_d : Real(0);  // coincident atoms: d = 0
  const Real sigma = lj_sigma(f1, f2, p1.w, p2.w, gp);
  const Real wcp = C::ELEC ? code_weight<Real>(code) : (code ? Real(0.2) : Real(1));
  Real atr, rep, dlj;
  lj_pair<Real, C::DERIV>(dist, sigma, se1 * se2, wcp, gp, atr, rep, dlj);
  if (!C::NOE) {
    en.atr.add(atr);
    en.rep.add(rep);
  }
  const bool inside = dist < sigma;
  Real gs = dlj;
  if (C::WGRAD) gs *= inside ? wrow[1] : wrow[0];
  if (C::ELEC) {
    const Real qq = code_weight<Real>(e >> CODE_EL) * (L.prm[s1][3] * L.prm[s2][3]);
    Real v, dv;
    elec_unit<Real, C::DERIV>(dist, ek, v, dv);
    if (!C::NOE) en.el.add(qq * v);
    if (C::DERIV) gs += wel * (qq * dv);
  }
  if (C::DERIV && gs != Real(0) && dist > Real(0))
    stream_scatter<Real, MODE>(L, C::DVDX && inside ? 1 : 0, s1, s2, gs * inv_d, dx, dy, dz, odd);
  return (f1 & f2 & F_HEAVY) && (!C::ELEC || code != CODE_NONE);
}

template <int MODE, int OCC>
constexpr int stream_waves_per_simd() {
  return OCC > 0 ? OCC : 4;
}

template <typename Real, int MODE, int OCC = 0>
__global__ __launch_bounds__(256, (stream_waves_per_simd<MODE, OCC>())) void score_stream_kernel(
    ScoreArgs<Real> A) {
  using C = RowCtx<Real, MODE>;
  using V = typename V4<Real>::T;
  static_assert(!C::BP && !(C::ELEC && (C::DVDX || C::DET)), "modes of the row kernel");
  __shared__ StreamLDS<Real, MODE> lds_all[WAVES_PER_WG];
  const int lane = lane_id();
  StreamLDS<Real, MODE>& L = lds_all[uni(threadIdx.x / WAVE)];
  const GlobalParams<Real> gp = load_global_params(A.global_params);
  const ElecConst<Real> ek = A.ek;
  const StackView& s = A.s;
  const BTView& bt = A.bt;
  const int shift = A.part_shift;
  RowQueue queue(A.row_cursor, int64_t(s.G) << shift, A.row_grab);
  const Real cull_pad = gp.max_dis + Real(1e-3);
  // in a scalar register: the fused gradient mode is at its 128 VGPRs
  const Real cut2 = wave_lane(C::ELEC && ek.cull2 > gp.max_dis2 ? ek.cull2 : gp.max_dis2, 0);
  const int u = lane & (SCH - 1), half = lane >> 5;
  const int odd = (lane & 1) ? SSLOTS : 0;

  if (C::DERIV) {
    auto* g = &L.grad[0][0][0];
    for (int i = lane; i < L.NGP * 3 * GROW; i += WAVE) g[i] = 0;
  }
  wave_sync();

  for (int64_t unit = queue.next(); unit >= 0; unit = queue.next()) {
    const int64_t row = unit >> shift;
    const int n_row = uni((int)min<int64_t>(A.w.row_count[row], A.w.row_cap));
    // this part's items [k_lo, n_items) of the row
    const int64_t part = unit - (row << shift);
    const int k_lo = int((n_row * part) >> shift);
    const int n_items = int((n_row * (part + 1)) >> shift);
    if (n_items == k_lo) continue;
    const int g1 = (int)row;
    const int t1 = uni(s.block_type[g1]);
    const int n1 = uni(bt.n_atoms[t1]);
    const int o1 = uni(s.block_atom_offset[g1]);
    const int p = uni(s.pose_of(g1));
    const int nc1 = uni(bt.n_conn[t1]);
    const bool lig1 = bt.is_ligand[t1] != 0;
    const V sph1 = *(const V*)(A.spheres + 4 * int64_t(g1));
    Real wrow[3] = {Real(0), Real(0), Real(0)};
    if (C::WGRAD) {
      wrow[0] = A.weights[p];
      wrow[1] = A.weights[s.P + p];
      wrow[2] = A.weights[2 * s.P + p];
    }
    const Real wel = (C::ELEC && C::WGRAD) ? A.weights[3 * s.P + p] : Real(0);
    const Real reach1 = sph1.w + cull_pad;
    const Real reach1_2 = reach1 * reach1;
    auto stage = [&](int slot, const AtomRegs<Real>& R) {
      V pp, pq;
      pp.x = R.x; pp.y = R.y; pp.z = R.z; pp.w = R.r0.x;
      pq.x = R.r0.z; pq.y = R.r0.w; pq.z = R.vol; pq.w = C::ELEC ? R.q : Real(0);
      *(V*)L.pos[slot] = pp;
      *(V*)L.prm[slot] = pq;
      L.lj2[slot][0] = R.r0.y;
      L.lj2[slot][1] = pack_flags(R.flags, Real(0));
    };
    // ---- stage g1 into slots 0..31
    if (lane < n1) {
      AtomRegs<Real> R;
      load_atom<Real, C::ELEC>(R, A, t1, o1, lane);
      stage(lane, R);
      L.pd1[lane] = R.pd;
      if (C::ELEC) L.epd1[lane] = R.epd;
    }
    StreamEnergies en;
    int n_lj = 0, n_lk = 0, seq_lj = 0, done_lj = 0;
    int end_lj[3] = {0, 0, 0};
    int cnt[3] = {0, 0, 0};  // atoms held by each ring chunk (0: free)
    int cur = 0;             // ring chunk being filled
    int fill = 0;            // its atoms so far
    bool cur_cp = false, cur_lig = false;  // it holds atoms within 4 bonds / ligand atoms
    wave_sync();

    auto drain_lk = [&]() {
      const int c = min(n_lk, WAVE);
      stream_lk<Real, MODE>(L, c, gp, wrow, en, lane, odd);
      wave_sync();
      fifo_shift(L.lk, c, n_lk, lane);
      n_lk -= c;
    };
    // one batch of the pair FIFO; its heavy-heavy entries join the LK FIFO
    auto drain = [&]() {
      const int c = min(n_lj, WAVE);
      int e = 0;
      const bool hv = stream_pairs<Real, MODE>(L, c, gp, ek, wrow, wel, en, lane, odd, &e);
      const uint64_t m = __ballot(hv);
      if (hv) L.lk[n_lk + lanes_below(m)] = (uint16_t)(e & ((1 << CODE_EL) - 1));
      n_lk += __popcll(m);
      wave_sync();
      fifo_shift(L.lj, c, n_lj, lane);
      n_lj -= c;
      done_lj += c;
      if (n_lk >= WAVE) drain_lk();
    };
    auto append = [&](bool in, int e) {
      const uint64_t m = __ballot(in);
      if (in) L.lj[n_lj + lanes_below(m)] = (uint16_t)e;
      n_lj += __popcll(m);
      seq_lj += __popcll(m);
      wave_sync();
      if (n_lj >= WAVE) drain();
    };
    // ring chunk r no longer referenced: evaluate what still points at it,
    // flush its atoms (LK entries are in ring order, so the oldest pending one
    // tells whether any is left)
    auto retire = [&](int r) {
      if (cnt[r] == 0) return;
      if (end_lj[r] > done_lj) drain();
      if (n_lk > 0) {
        const int head = (uni((int)L.lk[0]) >> 10) & 3;  // 0: intra-block, 1 + ring chunk
        if (head == 0 || head == r + 1) drain_lk();
      }
      flush_chunk<Real, MODE>(L, A, r, cnt[r], lane);
      cnt[r] = 0;
    };
    // phase A of the current chunk (fill atoms), then the next ring chunk
    auto test_chunk = [&]() {
      const int r = cur;
      const int n = fill;
      const V tr = *(const V*)L.pos[TILE + SCH * r + u];
      const uint32_t qb = L.tq()[u];
      const uint32_t eqb = C::ELEC ? L.teq[u] : 0;
      const bool lig2 = (qb & Q_LIG) != 0;
      const bool ok_u = u < n;
      const int ebase = (TILE + SCH * r + u) << 5;
      wave_sync();
      for (int t = 0; t < n1; t += 2) {
        const int ta = t + half;
        const int tl = ta < n1 ? ta : t;
        const V P1 = *(const V*)L.pos[tl];
        const Real dx = P1.x - tr.x, dy = P1.y - tr.y, dz = P1.z - tr.z;
        const Real d2 = dx * dx + dy * dy + dz * dz;
        bool in = ok_u && ta < n1 && d2 < cut2;
        int e = ebase | ta;
        if (cur_cp) {
          int sep = min_sep_bytes(qb + L.pd1[tl]);
          if (cur_lig && lig1 && lig2 && (sep == 3 || sep == 4)) sep = 5;
          const int code = sep > 4 ? 0 : (sep == 4 ? 1 : CODE_NONE);
          if (C::ELEC) {
            int sep_e = min_sep_bytes(eqb + L.epd1[tl]);
            if (cur_lig && lig1 && lig2 && (sep_e == 3 || sep_e == 4)) sep_e = 5;
            const int code_e = sep_e > 4 ? 0 : (sep_e == 4 ? 1 : CODE_NONE);
            in = in && (code != CODE_NONE || code_e != CODE_NONE);
            e |= code_e << CODE_EL;
          } else {
            in = in && code != CODE_NONE;
          }
          e |= code << CODE_LJ;
        }
        append(in, e);
      }
      end_lj[r] = seq_lj;
      cnt[r] = n;
      cur = cur == 2 ? 0 : cur + 1;
      fill = 0;
      cur_cp = cur_lig = false;
      retire(cur);  // the chunk two before: its entries are consumed by now
    };

    int k0 = k_lo;
    if (k_lo == 0 && uni(A.w.row_items[row * A.w.row_cap]) == g1) {
      // ---- intra-block pairs a1 < a2 of non-zero weight (prepared tables)
      auto intra = [&](int n_ip, const uint16_t* ip, Real cut2, int code_other, int code_shift) {
        for (int j0 = 0; j0 < n_ip; j0 += WAVE) {
          bool in = false;
          int e = 0;
          if (j0 + lane < n_ip) {
            const int w = ip[j0 + lane];
            const int a1 = w & 31, a2 = (w >> 5) & 31;
            const V pa = *(const V*)L.pos[a1], pb = *(const V*)L.pos[a2];
            const Real dx = pa.x - pb.x, dy = pa.y - pb.y, dz = pa.z - pb.z;
            in = dx * dx + dy * dy + dz * dz < cut2;
            e = a1 | (a2 << 5) | code_other | (((w >> 10) & 1) << code_shift);
          }
          append(in, e);
        }
      };
      intra(uni(A.intra_count[t1]), A.intra_pairs + int64_t(t1) * INTRA_MAX, gp.max_dis2,
            C::ELEC ? CODE_NONE << CODE_EL : 0, CODE_LJ);
      // elec's own table (representative separations, charged atoms only)
      if (C::ELEC)
        intra(uni(A.e_intra_count[t1]), A.e_intra_pairs + int64_t(t1) * INTRA_MAX, ek.cull2,
              CODE_NONE << CODE_LJ, CODE_EL);
      k0 = 1;
    }

    for (int c0 = k0; c0 < n_items; c0 += WAVE) {
      // ---- descriptors: one neighbor block per lane
      const int nb = min(WAVE, n_items - c0);
      int d_t2 = 0, d_o2 = 0, d_n2 = 0, d_info = 0;
      uint32_t cs[MAX_CONN] = {0, 0, 0, 0};  // read for blocks within 4 bonds only
      if (lane < nb) {
        const int g2 = A.w.row_items[row * A.w.row_cap + c0 + lane];
        if (g2 != g1) {
          d_t2 = s.block_type[g2];
          d_o2 = s.block_atom_offset[g2];
          d_n2 = bt.n_atoms[d_t2];
          const int nc2 = bt.n_conn[d_t2];
          const int ms = pair_separations(s, g1, g2, nc1, nc2, cs);
          const bool lig2 = lig1 && bt.is_ligand[d_t2] != 0;
          d_info = (ms <= 4 ? 1 : 0) | (lig2 ? 2 : 0) | (d_n2 << 8);
        }
      }
      // exclusive scan of the atom counts: the stream position of each block
      int incl = d_n2;
#pragma unroll
      for (int o = 1; o < WAVE; o <<= 1) {
        const int y = __shfl_up(incl, o, WAVE);
        if (lane >= o) incl += y;
      }
      const int d_pre = incl - d_n2;
      const int total = uni(__shfl(incl, WAVE - 1, WAVE));

      for (int q0 = 0; q0 < total; q0 += WAVE) {
        // ---- raw chunk: lane -> (block, atom) through start markers
        L.mark()[lane] = 0;
        wave_sync();
        if (d_n2 > 0 && d_pre >= q0 && d_pre < q0 + WAVE) L.mark()[d_pre - q0] = 1;
        wave_sync();
        const uint64_t M = __ballot(L.mark()[lane] != 0);
        // blocks with atoms that start at or before q0, less one: the block
        // holding stream position q0 (in lane order over blocks with atoms)
        const int kfirst = __popcll(__ballot(d_n2 > 0 && d_pre <= q0)) - 1;
        const int rank = kfirst + lanes_below(M) + int((M >> lane) & 1ull) - int(M & 1ull);
        // every listed block but g1 itself (row position 0, skipped) has
        // atoms, so the rank-th block with atoms is descriptor lane `rank`
        const int k = rank;
        const int q = q0 + lane;
        const bool valid = q < total;  // (and a within its block, checked below)
        const int pre_k = __shfl(d_pre, k, WAVE);
        const int o2 = __shfl(d_o2, k, WAVE), t2 = __shfl(d_t2, k, WAVE);
        const int info = __shfl(d_info, k, WAVE);
        const int a = q - pre_k;
        AtomRegs<Real> R;
        bool near = false;
        if (valid && a >= 0 && a < (info >> 8)) {
          load_atom<Real, C::ELEC>(R, A, t2, o2, a);
          const Real ex = R.x - sph1.x, ey = R.y - sph1.y, ez = R.z - sph1.z;
          near = ex * ex + ey * ey + ez * ez < reach1_2;
        }
        const uint64_t mnear = __ballot(near);
        const int n_surv = __popcll(mnear);
        if (n_surv == 0) continue;
        // combined connection bytes q (count pair) for atoms within 4 bonds
        uint32_t qv = Q_NONE, eqv = Q_NONE;
        const uint64_t mcp = __ballot(near && (info & 1));
        if (mcp) {
          uint32_t csk[MAX_CONN];
#pragma unroll
          for (int c1 = 0; c1 < MAX_CONN; ++c1) csk[c1] = (uint32_t)__shfl((int)cs[c1], k, WAVE);
          if (info & 1) {
            qv = combine_q(csk, R.pd);
            if (C::ELEC) eqv = combine_q(csk, R.epd);
          }
        }
        qv |= (info & 2) ? Q_LIG : 0u;
        const bool any_lig = __ballot(near && (info & 2)) != 0;
        const int rk = lanes_below(mnear);
        // stage the survivors into test chunks of 32
        int done = 0;
        while (done < n_surv) {
          const int take = min(n_surv - done, SCH - fill);
          const bool mine = near && rk >= done && rk < done + take;
          if (mine) {
            const int pos = fill + rk - done;
            stage(TILE + SCH * cur + pos, R);
            L.tq()[pos] = qv;
            if (C::ELEC) L.teq[pos] = eqv;
            L.atom[SCH * cur + pos] = o2 + a;
          }
          cur_cp = cur_cp || (__ballot(mine && (info & 1)) != 0);
          cur_lig = cur_lig || (any_lig && __ballot(mine && (info & 2)) != 0);
          fill += take;
          done += take;
          wave_sync();
          if (fill == SCH) test_chunk();
        }
      }
    }
    // ---- row end: test the partial chunk, evaluate the rest, flush
    if (fill > 0) test_chunk();
    if (n_lj > 0) drain();
    if (n_lk > 0) drain_lk();
    for (int r = 0; r < 3; ++r)
      if (cnt[r] > 0) {
        flush_chunk<Real, MODE>(L, A, r, cnt[r], lane);
        cnt[r] = 0;
      }
    flush_g1<Real, MODE>(L, A, n1, o1, lane);
    if (!C::NOE) {
      const double ea = wave_sum(en.atr.value());
      const double er = wave_sum(en.rep.value());
      const double el = wave_sum(en.lk.value());
      if (lane == 0 && C::DET) {
        auto* e = (unsigned long long*)A.energies64;
        atomicAdd(&e[p], det_energy_enc(ea));
        atomicAdd(&e[s.P + p], det_energy_enc(er));
        atomicAdd(&e[2 * s.P + p], det_energy_enc(el));
      } else if (lane == 0) {
        unsafeAtomicAdd(&A.energies64[p], ea);
        unsafeAtomicAdd(&A.energies64[s.P + p], er);
        unsafeAtomicAdd(&A.energies64[2 * s.P + p], el);
      }
      if (C::ELEC) {
        const double ee = wave_sum(en.el.value());
        if (lane == 0) unsafeAtomicAdd(&A.energies64[3 * s.P + p], ee);
      }
    }
    wave_sync();
  }
}

}  // namespace tmol_ljlk
