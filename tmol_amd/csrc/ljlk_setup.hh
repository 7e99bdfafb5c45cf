// First launch of a call: block-type tables, bounding spheres and the clears
// of the neighbor pass (and of the scoring pass where both run in one call).
//
// Bound: launch count.  Each piece takes 4-13 us by itself, most of it the
// latency of starting; as separate launches (two fills, records, intra-block
// table, elec tables, spheres) they cost a small protein's call more than its
// pairs.  The first T workgroups build one block type's tables each (they hold
// the longest chains), the others take spheres and clears.
#pragma once

#include "ljlk_elec.hh"
#include "ljlk_neighbors.hh"

namespace tmol_ljlk {

template <typename Real>
struct SetupArgs {
  StackView s;  // s.G spheres
  BTView bt;
  const Real* coords;
  Real* spheres;
  // LJ+LK tables (records null: none)
  const Real* type_params;
  int n_atom_types;
  Real* records;
  uint8_t* conn_pd;
  int32_t* intra_count;  // null: no intra-block table
  uint16_t* intra_pairs;
  // elec tables (epd null: none)
  const Real* charge;
  const int32_t* inter_rpd;
  const int32_t* intra_rpd;
  uint32_t* epd;
  int32_t* e_intra_count;
  uint16_t* e_intra_pairs;
  ClearList clear;
  int type_jobs;  // leading workgroups that build tables: T, or 0
};

template <typename Real>
__global__ __launch_bounds__(256) void setup_kernel(SetupArgs<Real> A) {
  const int tid = threadIdx.x;
  if (int(blockIdx.x) < A.type_jobs) {
    const int t = blockIdx.x, lane = lane_id(), wave = tid / WAVE;
    if (A.records)
      for (int a = tid; a < A.bt.Amax; a += 256)
        prepare_record(A.bt, t, a, A.type_params, A.n_atom_types, A.records, A.conn_pd);
    if (A.intra_count && wave == 0) prepare_intra(A.bt, t, lane, A.intra_count, A.intra_pairs);
    if (A.epd && wave == 1)
      elec_prepare(A.bt, t, lane, A.charge, A.inter_rpd, A.intra_rpd, A.epd, A.e_intra_count,
                   A.e_intra_pairs);
    return;
  }
  const int64_t i0 = int64_t(blockIdx.x - A.type_jobs) * 256 + tid;
  const int64_t stride = int64_t(gridDim.x - A.type_jobs) * 256;
  for (int64_t g = i0; g < A.s.G; g += stride)
    block_sphere(A.s, A.bt, int(g), A.coords, A.spheres);
  clear_ranges(A.clear, i0, stride);
}

}  // namespace tmol_ljlk
