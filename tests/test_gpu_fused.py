"""GPU tests of the fused LJ+LK+elec pass (``LJLKElecRaggedScorer``,
``tmol_ljlk_elec_score``): one neighbor pass and one scoring launch give the
same per-pose energies and weighted gradient as the two terms scored
separately, and as the two oracles; hipGraph replays match eager calls."""

import sys

import numpy
import pytest
import torch

from oracle import oracle as orc
from tmol_amd.generator import generate_poses, workload_poses
from tmol_amd.io_pdb import pose_from_pdb
from tmol_amd.pose import PoseStack, RaggedPoseStack
from tmol_amd.score.elec_energy_term import ElecEnergyTerm, elec_op_args
from tmol_amd.score.ljlk_energy_term import LJLKEnergyTerm, pose_op_args

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
W4 = numpy.array([1.0, 0.55, 1.0, 0.8])


def _say(msg):
    print("[gpu-case] " + msg, flush=True)
    sys.stdout.flush()


def _poses(ubq_pdb):
    return [pose_from_pdb(ubq_pdb), pose_from_pdb(ubq_pdb, (20, 50))] + generate_poses(
        6, (10, 150), seed=21, log_uniform=True)


def _scorers(poses, dtype):
    from tmol_amd.scorer import ElecRaggedScorer, LJLKElecRaggedScorer, LJLKRaggedScorer

    st = RaggedPoseStack(poses, dtype=dtype)
    lj = LJLKEnergyTerm(device=DEV)
    el = ElecEnergyTerm()
    return (st, LJLKElecRaggedScorer(st, lj, el, device=DEV, dtype=dtype),
            LJLKRaggedScorer(st, lj, device=DEV, dtype=dtype),
            ElecRaggedScorer(st, el, device=DEV, dtype=dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_fused_equals_separate_terms_and_oracles(ubq_pdb, dtype):
    poses = _poses(ubq_pdb)
    _say("fused vs separate %s" % dtype)
    st, fused, lj, el = _scorers(poses, dtype)
    x = st.coords.to(DEV)
    w = torch.tensor(W4)
    e4, g4 = [t.double().cpu().numpy() for t in fused.energy_and_grad(x, w)]
    e3, g3 = [t.double().cpu().numpy() for t in lj.energy_and_grad(x, w[:3])]
    e1, g1 = [t.double().cpu().numpy() for t in el.energy_and_grad(x, float(W4[3]))]
    tol = 1e-10 if dtype == torch.float64 else 1e-5
    scale = numpy.maximum(1.0, numpy.abs(e4))
    assert (numpy.abs(e4[:3] - e3) / scale[:3]).max() < tol
    assert (numpy.abs(e4[3] - e1) / scale[3]).max() < tol
    g = g3 + g1
    assert numpy.abs(g4 - g).max() / max(1.0, numpy.abs(g).max()) < tol
    # the gradient-only pass gives the same gradient
    grad = torch.empty_like(fused.grad)
    fused.neighbors(x)
    fused.score(x, 4 | 16, weights=fused._weights(w), grad=grad)
    assert numpy.abs(grad.double().cpu().numpy() - g4).max() <= 1e-12 * max(1.0, numpy.abs(g4).max()) \
        or dtype == torch.float32
    if dtype == torch.float64:
        # both oracles on the padded stack of the same poses
        ps = PoseStack(poses, dtype=torch.float64)
        a = pose_op_args(ps, LJLKEnergyTerm())
        a[23], a[24] = a[23].double(), a[24].double()
        s3, _, dv3, _ = orc.oracle_pose_scores(*a, require_grad=True)
        b = elec_op_args(ps, ElecEnergyTerm())
        b[16], b[22] = b[16].double(), b[22].double()
        s1, _, dv1, _ = orc.oracle_elec_scores(*b, require_grad=True)
        A = ps.max_n_atoms
        keep = numpy.concatenate([p * A + numpy.arange(pose.n_atoms) for p, pose in enumerate(poses)])
        og = (dv3[:, keep] * W4[:3, None, None]).sum(0) + W4[3] * dv1[0, keep]
        oe = numpy.concatenate([s3, s1], axis=0)
        assert (numpy.abs(e4 - oe) / numpy.maximum(1.0, numpy.abs(oe))).max() < 1e-9
        assert numpy.abs(g4 - og).max() / max(1.0, numpy.abs(og).max()) < 1e-9


def test_fused_graph_replays_match_eager(ubq_pdb):
    poses = _poses(ubq_pdb)
    _say("fused graph replay")
    st, fused, _, _ = _scorers(poses, torch.float32)
    x = st.coords.to(DEV)
    e0, g0 = [t.clone() for t in fused.energy_and_grad(x)]
    fused.capture(x)
    for k in range(3):
        e, g = fused.replay()
        torch.cuda.synchronize()
        assert torch.equal(e, e0) or (e - e0).abs().max().item() < 1e-4
        assert (g - g0).abs().max().item() <= 1e-5 * max(1.0, g0.abs().max().item())
        _ = fused.energy_and_grad(x)  # eager work between replays
        torch.cuda.synchronize()


def test_fused_on_the_512_pose_batch():
    """The headline batch: fused energies and gradient against the two
    separate passes (float32)."""
    poses = workload_poses("ragged_512x50_1200")
    _say("fused 512 poses")
    st, fused, lj, el = _scorers(poses, torch.float32)
    x = st.coords.to(DEV)
    e4, g4 = [t.double() for t in fused.energy_and_grad(x)]
    e3, g3 = [t.double() for t in lj.energy_and_grad(x, torch.tensor([1.0, 0.55, 1.0]))]
    e1, g1 = [t.double() for t in el.energy_and_grad(x, 1.0)]
    assert (e4[:3] - e3).abs().max().item() < 1e-5 * max(1.0, e3.abs().max().item())
    assert (e4[3] - e1).abs().max().item() < 1e-4
    g = g3 + g1
    assert ((g4 - g).norm() / g.norm()).item() < 1e-6


@pytest.mark.parametrize("n,lo,hi", [(1, 2, 2), (1, 9, 9), (2, 33, 35), (9, 40, 90), (220, 2, 7),
                                     (420, 5, 5), (1100, 4, 6)])
@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
def test_split_rows_equal_the_oracles(n, lo, hi, dt):
    """Rows are split into parts when a batch has at most half as many rows as
    resident waves (4096 of the fused float32 kernel on 256 CUs, 2048 of the
    float64 one): per-pose energies, the weighted gradient and the drop-in
    ops' per-term derivatives from one residue pair over 1000 rows (split in
    two and in four), 2100 (just above half of 4096, and above 2048) to 5500."""
    poses = generate_poses(n, (lo, hi), seed=11 + n)
    _say("split rows %d x %d-%d %s" % (n, lo, hi, dt))
    ps = PoseStack(poses, dtype=torch.float64)

    def f64(args):  # the oracles in float64, on the values that the kernels are given
        return [t.to(dt).double() if torch.is_tensor(t) and t.is_floating_point() else t
                for t in args]

    a = f64(pose_op_args(ps, LJLKEnergyTerm()))
    b = f64(elec_op_args(ps, ElecEnergyTerm()))
    s3, _, dv3, _ = orc.oracle_pose_scores(*a, require_grad=True)
    s1, _, dv1, _ = orc.oracle_elec_scores(*b, require_grad=True)
    keep = numpy.concatenate([p * ps.max_n_atoms + numpy.arange(q.n_atoms)
                              for p, q in enumerate(poses)])
    st, fused, _, _ = _scorers(poses, dt)
    e4, g4 = [t.double().cpu().numpy()
              for t in fused.energy_and_grad(st.coords.to(DEV), torch.tensor(W4))]
    oe = numpy.concatenate([s3, s1], axis=0)
    og = (dv3 * W4[:3, None, None]).sum(0) + W4[3] * dv1[0]
    # float64 on both sides: the bounds of the fused test above.  float32: a
    # pair is off by up to 1e-6 of its own size, and a pose's elec energy is
    # the remainder of pairs that cancel to a part in a hundred, so 1e-4 of it
    # (as in the edge cases' tests); an atom's gradient stays within ten pairs
    # of the largest
    tol, etol = (1e-9, 1e-9) if dt == torch.float64 else (1e-5, 1e-4)
    assert (numpy.abs(e4 - oe) / numpy.maximum(1.0, numpy.abs(oe))).max() < etol
    assert numpy.abs(g4 - og[keep]).max() / max(1.0, numpy.abs(og).max()) < tol
    from tmol_amd.ops import elec_pose_scores, ljlk_pose_scores

    for op, args, want, w in ((ljlk_pose_scores, a, dv3, W4[:3]),
                              (elec_pose_scores, b, dv1, W4[3:])):
        for bp in (False, True):
            d = [t.to(DEV, dt if t.is_floating_point() else None) if torch.is_tensor(t) else t
                 for t in args[:-1]] + [bp]
            x = d[0].clone().requires_grad_(True)
            out = op(x, *d[1:])
            scores = out[0] if isinstance(out, (tuple, list)) else out
            wt = torch.tensor(w, device=DEV).view([-1] + [1] * (scores.dim() - 1))
            (scores * wt).sum().backward()
            go = (want * w[:, None, None]).sum(0)
            err = numpy.abs(x.grad.double().cpu().numpy() - go).max()
            assert err <= tol * max(1.0, numpy.abs(go).max()), (op, bp, err)
