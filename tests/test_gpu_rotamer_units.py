"""Rotamer work units and the rotamer-sphere cull: blocks whose rotamer counts
lie at the edges of the unit rule (as many b1 rotamers, up to four, as make
32 rotamer pairs) and of a window of 64, with every other rotamer of two
blocks moved out of reach, in float64 against the f64 oracles."""

import numpy
import pytest
import torch

from oracle import oracle as orc
from rotamer_cases import dense_case, densify_rotamers
from tmol_amd.rotamers import rotamer_op_args
from tmol_amd.score.elec_energy_term import ElecEnergyTerm
from tmol_amd.score.ljlk_energy_term import LJLKEnergyTerm

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("counts", [(1, 2, 3, 4, 5, 7), (8, 9, 10, 11, 16, 17), (31, 32, 33, 63, 64, 65)])
@pytest.mark.parametrize("away", [0.0, 9.0])
@pytest.mark.parametrize("name", ["ljlk", "elec"])
def test_units_at_the_edges_of_the_rule(name, counts, away):
    import tmol_amd.ops as ops

    print("rotamer units", name, counts, away, flush=True)
    term, op, oracle = {
        "ljlk": (LJLKEnergyTerm(), torch.ops.tmol_ljlk.ljlk_rotamer_scores, orc.oracle_rotamer_scores),
        "elec": (ElecEnergyTerm(), ops.elec_rotamer_scores, orc.oracle_elec_rotamer_scores)}[name]
    ps, rs = dense_case()[torch.float64]
    nat = ps.packed_block_types.n_atoms.numpy()
    rs = densify_rotamers(rs, {(0, 1 + i): n for i, n in enumerate(counts)}, nat, seed=3)
    if away:
        off, bt = rs.coord_offset_for_rot.numpy(), rs.block_type_ind_for_rot.numpy()
        for b in (2, 4):
            first = int(rs.rot_offset_for_block[0, b])
            for r in range(first + 1, first + int(rs.n_rots_for_block[0, b]), 2):
                rs.coords[off[r]: off[r] + nat[bt[r]], 0] += away
    a = rotamer_op_args(ps, rs, term)
    for i in ((16, 22) if name == "elec" else (23, 24)):
        a[i] = a[i].double()
    d = [x.to(DEV) if torch.is_tensor(x) else x for x in a]
    d[0] = d[0].clone().requires_grad_(True)
    s, idx = op(*d)
    w = torch.rand(s.shape, generator=torch.Generator().manual_seed(2), dtype=torch.float64)
    (s * w.to(DEV)).sum().backward()
    out = oracle(*a, dTdV=w.numpy())
    assert numpy.array_equal(idx.cpu().numpy(), out[1])
    # the same formulas in float64, sums in another order: the bounds of the
    # dense rotamer tests
    E = s.detach().cpu().numpy()
    assert (numpy.abs(E - out[0]) / numpy.maximum(1.0, numpy.abs(out[0]))).max() < 1e-10
    assert numpy.abs(d[0].grad.cpu().numpy() - out[-1]).max() < 1e-10 * max(1.0, numpy.abs(out[-1]).max())
