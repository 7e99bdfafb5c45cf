"""GPU tests of the ragged persistent scorer: parity with the oracle on the
same poses, hipGraph replays, census consistency, overflow detection."""

import sys

import numpy
import pytest
import torch

from oracle import oracle as orc
from tmol_amd.generator import generate_poses
from tmol_amd.io_pdb import pose_from_pdb
from tmol_amd.pose import PoseStack, RaggedPoseStack
from tmol_amd.score.ljlk_energy_term import LJLKEnergyTerm, pose_op_args

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
W = numpy.array([1.0, 0.55, 1.0])


def _say(msg):
    print("[gpu-case] " + msg, flush=True)
    sys.stdout.flush()


def _poses(ubq_pdb):
    return [pose_from_pdb(ubq_pdb), pose_from_pdb(ubq_pdb, (20, 50))] + generate_poses(
        6, (10, 150), seed=5, log_uniform=True
    )


def _oracle(poses, dtype=numpy.float64):
    ps = PoseStack(poses, dtype=torch.float64 if dtype == numpy.float64 else torch.float32)
    a = pose_op_args(ps, LJLKEnergyTerm())
    if dtype == numpy.float64:
        a[23] = a[23].double()
        a[24] = a[24].double()
    s, _, dv, _ = orc.oracle_pose_scores(*a, require_grad=True, dtype=dtype)
    # padded atom order -> ragged atom order (poses concatenated without padding)
    A = ps.max_n_atoms
    keep = numpy.concatenate([p * A + numpy.arange(pose.n_atoms) for p, pose in enumerate(poses)])
    return s, dv[:, keep]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_ragged_energy_and_grad(ubq_pdb, dtype):
    from tmol_amd.scorer import LJLKRaggedScorer

    poses = _poses(ubq_pdb)
    _say("ragged energy+grad %s" % dtype)
    stack = RaggedPoseStack(poses, dtype=dtype)
    term = LJLKEnergyTerm(device=DEV)
    sc = LJLKRaggedScorer(stack, term, device=DEV, dtype=dtype)
    x = stack.coords.to(DEV)
    e, g = sc.energy_and_grad(x, torch.tensor(W))
    e = e.double().cpu().numpy()
    g = g.double().cpu().numpy()
    s64, dv64 = _oracle(poses)
    og = (dv64 * W[:, None, None]).sum(0)
    if dtype == torch.float64:
        numpy.testing.assert_allclose(e, s64, rtol=1e-9, atol=1e-9)
        numpy.testing.assert_allclose(g, og, rtol=1e-8, atol=1e-8)
    else:
        rel = numpy.abs(e - s64) / numpy.maximum(numpy.abs(s64), 1.0)
        assert rel.max() < 1e-4, rel.max()
        assert numpy.abs(g - og).max() / numpy.abs(og).max() < 1e-5
    # per-term planes agree with the weighted gradient
    _, dv = sc.per_term_gradients(x)
    g2 = (dv.double().cpu().numpy() * W[:, None, None]).sum(0)
    assert numpy.abs(g2 - og).max() / numpy.abs(og).max() < (1e-12 if dtype == torch.float64 else 1e-5)


def test_graph_replays_match_eager(ubq_pdb):
    from tmol_amd.scorer import LJLKRaggedScorer

    poses = _poses(ubq_pdb)
    _say("graph replay")
    stack = RaggedPoseStack(poses)
    sc = LJLKRaggedScorer(stack, LJLKEnergyTerm(device=DEV), device=DEV)
    x = stack.coords.to(DEV)
    e0, g0 = [t.clone() for t in sc.energy_and_grad(x, torch.tensor(W))]
    sc.capture(x, torch.tensor(W))
    rng = torch.Generator().manual_seed(0)
    for k in range(4):
        xk = x + 0.01 * k * torch.randn(x.shape, generator=rng).to(DEV)
        ee, ge = [t.clone() for t in sc.energy_and_grad(xk, torch.tensor(W))]
        torch.cuda.synchronize()
        er, gr = sc.replay(xk)
        torch.cuda.synchronize()
        torch.testing.assert_close(er, ee, rtol=1e-6, atol=1e-4)
        torch.testing.assert_close(gr, ge, rtol=1e-5, atol=1e-4)
    er, gr = sc.replay(x)
    torch.testing.assert_close(er, e0, rtol=1e-6, atol=1e-4)


def test_census_counts(ubq_pdb):
    from tmol_amd.scorer import LJLKRaggedScorer

    poses = _poses(ubq_pdb)[:4]
    _say("census")
    stack = RaggedPoseStack(poses)
    sc = LJLKRaggedScorer(stack, LJLKEnergyTerm(device=DEV), device=DEV)
    x = stack.coords.to(DEV)
    c = sc.census(x)
    n = sc.check_capacity()
    items = sc.ws.pairs(sc.cstack, sc.bt.c).numpy()
    assert items.shape[0] == n
    bt = stack.block_type.numpy()
    pbt = stack.packed_block_types
    nat = pbt.n_atoms.numpy()
    nh = pbt.ljlk_n_heavy_atoms_in_tile.numpy().sum(1)
    lj = lk = 0
    for g1, g2 in items:
        n1, n2 = nat[bt[g1]], nat[bt[g2]]
        h1, h2 = nh[bt[g1]], nh[bt[g2]]
        if g1 == g2:
            lj += n1 * (n1 - 1) // 2
            lk += h1 * (h1 - 1) // 2
        else:
            lj += n1 * n2
            lk += h1 * h2
    assert c["items"] == len(items)
    assert c["lj_pairs"] == lj and c["lk_pairs"] == lk
    lj_parts = sum(c[k] for k in ("lj_cp0", "lj_far", "lj_linear", "lj_126", "lj_spline"))
    lk_parts = sum(c[k] for k in ("lk_cp0", "lk_far", "lk_const", "lk_close", "lk_fdesolv", "lk_spline"))
    assert lj_parts == lj and lk_parts == lk


def test_overflow_is_reported(ubq_pdb):
    from tmol_amd.ops import LJLKLibraryError
    from tmol_amd.scorer import LJLKRaggedScorer

    poses = _poses(ubq_pdb)[:2]
    _say("overflow")
    stack = RaggedPoseStack(poses)
    sc = LJLKRaggedScorer(stack, LJLKEnergyTerm(device=DEV), device=DEV, capacity=16)
    sc.neighbors(stack.coords.to(DEV))
    with pytest.raises(LJLKLibraryError):
        sc.check_capacity()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_rows_kernel_matches_general_kernel(ubq_pdb, dtype):
    """The fast rows kernel and the general kernel evaluate the same work
    list; energies, per-term gradients and weighted gradients agree."""
    from tmol_amd import ops
    from tmol_amd.scorer import LJLKRaggedScorer

    poses = _poses(ubq_pdb)
    _say("rows vs general %s" % dtype)
    stack = RaggedPoseStack(poses, dtype=dtype)
    sc = LJLKRaggedScorer(stack, LJLKEnergyTerm(device=DEV), device=DEV, dtype=dtype)
    x = stack.coords.to(DEV)
    w = sc._weights(torch.tensor(W))
    sc.neighbors(x)
    out = {}
    for name, extra in (("rows", 0), ("general", ops.GENERAL_KERNEL)):
        e = torch.empty((3, sc.P), dtype=dtype, device=DEV)
        g = torch.empty((sc.NA, 3), dtype=dtype, device=DEV)
        dv = torch.empty((3, sc.NA, 3), dtype=dtype, device=DEV)
        e2 = torch.empty((3, sc.P), dtype=dtype, device=DEV)
        sc.score(x, ops.WGRAD | extra, weights=w, energies=e, grad=g)
        sc.score(x, ops.DVDX | extra, energies=e2, dvdx=dv)
        out[name] = [t.double().cpu() for t in (e, g, dv, e2)]
    tol = dict(rtol=1e-10, atol=1e-9) if dtype == torch.float64 else dict(rtol=2e-5, atol=2e-4)
    for a, b in zip(out["rows"], out["general"]):
        torch.testing.assert_close(a, b, **tol)


@pytest.mark.parametrize("general", [False, True])
def test_item_energies_sum_to_pose_energies(ubq_pdb, general):
    """Per-block-pair energies of a ragged stack ([3, G, capacity], one entry
    per work-list pair) sum per pose to the whole-pose energies, and are zero
    past each row's count."""
    from tmol_amd import ops
    from tmol_amd.scorer import LJLKRaggedScorer

    poses = _poses(ubq_pdb)
    _say("item energies general=%s" % general)
    stack = RaggedPoseStack(poses, dtype=torch.float64)
    sc = LJLKRaggedScorer(stack, LJLKEnergyTerm(device=DEV), device=DEV, dtype=torch.float64)
    x = stack.coords.to(DEV)
    if general:
        out = torch.empty((3, sc.G, sc.capacity), dtype=torch.float64, device=DEV)
        sc.neighbors(x)
        sc.score(x, ops.BLOCK_PAIR | ops.GENERAL_KERNEL, energies=out)
    else:
        out = sc.item_energies(x)
    cnt, _ = sc.ws.rows(sc.cstack, sc.bt.c)
    cnt = cnt.cpu().long().clamp(max=sc.capacity)
    past = torch.arange(sc.capacity)[None, :] >= cnt[:, None]
    assert float(out.cpu()[:, past].abs().max()) == 0.0
    per_block = out.sum(2).cpu()  # [3, G]
    per_pose = torch.zeros(3, sc.P, dtype=torch.float64).index_add_(
        1, stack.block_pose.long(), per_block)
    e = sc.energies_only(x).cpu()
    torch.testing.assert_close(per_pose, e, rtol=1e-10, atol=1e-8)


def test_f32_rounding_against_f64():
    """Float32 energies and gradients against the same kernels in float64 on
    the same inputs, as norms over 40 poses.  The gradients' 2.4e-7 is the
    rounding of the distance and of a pair's few products; 4e-7 lies below
    what sigma * rcp(x), off by 2-3 ulp, gives in the sixth power on the
    linear piece (5.1e-7).  Energies: 4e-8, and 9e-8 with it."""
    from tmol_amd.scorer import LJLKRaggedScorer

    _say("f32 rounding")
    poses = generate_poses(40, (50, 300), seed=19)
    x = RaggedPoseStack(poses, dtype=torch.float32).coords.to(DEV)
    out = {}
    for dt in (torch.float32, torch.float64):
        st = RaggedPoseStack(poses, dtype=dt)
        sc = LJLKRaggedScorer(st, LJLKEnergyTerm(device=DEV), device=DEV, dtype=dt)
        out[dt] = [t.double().clone() for t in sc.energy_and_grad(x.to(dt), torch.tensor(W))]
    for got, want, bound in zip(out[torch.float32], out[torch.float64], (7e-8, 4e-7)):
        assert (got - want).norm() <= bound * want.norm()
