"""Missing-leaf-atom building on the GPU (``gen_pose_leaf_atoms`` drop-in,
tmol_leaf_atoms_build / _backward) against the oracle, float32 and float64;
the canonical-form ingest end to end (heavy atoms of 1ubq and 6DMZ in,
hydrogens built, LJ+LK scored); and size-independent properties at a large
batch (idempotence, given atoms passing through)."""

import os

import numpy
import pytest
import torch

from oracle import leaf_oracle as lo
from tmol_amd import ingest

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")
# float64: the same formulas in another order; float32: hardware sin / cos
# and sqrt, float atomics in the backward sums
TOL = {torch.float64: 1e-11, torch.float32: 2e-5}


@pytest.fixture(scope="module")
def co():
    return ingest.CanonicalOrdering()


def _pdb(name):
    with open(os.path.join(GOLDEN, name)) as f:
        return f.read()


def _random_missing(co, dtype, seed=11, frac=0.6, names=("1ubq.pdb", "6DMZ_A.pdb")):
    lays = []
    for name in names:
        ch, rt, xyz = ingest.canonical_form_from_pdb(_pdb(name), co)
        lays += ingest.block_layout_from_canonical_form(co, ch, rt, xyz)
    ps = ingest.pose_stack_from_layouts(lays, dtype)
    _, tab = ingest.leaf_op_args(ps, co.db, lays)
    rng = numpy.random.default_rng(seed)
    for L in lays:
        for b, r in enumerate(L["rts"]):
            lf = tab.is_leaf[ps.packed_block_types.index[r.name]][: r.n_atoms]
            L["missing"][b][:] = lf & (rng.random(r.n_atoms) < frac)
    args, _ = ingest.leaf_op_args(ps, co.db, lays)
    return ps, args


def _dev(args):
    return [a.cuda() if torch.is_tensor(a) else a for a in args]


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("frac", [0.6, 1.0])
def test_leaf_atoms_match_oracle(co, dt, frac):
    """Forward (NaN placement exact) and backward of the HIP op against the
    oracle's autograd; frac=1 drops every leaf, O and OXT together (both
    unbuildable: NaN), every terminus on its backup ancestors."""
    print("leaf atoms", dt, frac, flush=True)
    ps, args = _random_missing(co, dt, frac=frac)
    args = [a.to(dt) if a.is_floating_point() else a for a in args]
    X = args[0].cuda().requires_grad_(True)
    da = _dev(args)
    da[0] = X
    out = ingest.gen_pose_leaf_atoms(*da)
    Xo = args[0].clone().requires_grad_(True)
    ao = list(args)
    ao[0] = Xo
    ref = lo.oracle_leaf_atoms(*ao)
    o = out.detach().cpu()
    assert torch.equal(torch.isnan(o), torch.isnan(ref))
    assert int(args[1].sum()) > 500
    scale = float(ref.detach().abs().nan_to_num(0).max())
    assert float((o - ref.detach()).abs().nan_to_num(0).max()) <= TOL[dt] * scale
    w = torch.randn(ref.shape, dtype=dt, generator=torch.Generator().manual_seed(4))
    (out.nan_to_num(0) * w.cuda()).sum().backward()
    (ref.nan_to_num(0) * w).sum().backward()
    g = X.grad.cpu()
    gs = max(1.0, float(Xo.grad.abs().max()))
    assert float((g - Xo.grad).abs().max()) <= 10 * TOL[dt] * gs


@pytest.mark.parametrize("pdb", ["1ubq.pdb", "6DMZ_A.pdb"])
def test_ingest_heavy_atoms_then_score(co, pdb):
    """Hydrogens stripped from the canonical form, rebuilt on the GPU by
    pose_stack_from_canonical_form: every rebuilt atom within 0.1 A of the
    deposited one (the reference test's bound) and the LJ+LK energies of
    the rebuilt pose close to those of the deposited one."""
    import tmol_amd.ops  # noqa: F401  (registers torch.ops.tmol_ljlk)
    from tmol_amd.score.ljlk_energy_term import LJLKEnergyTerm, pose_op_args

    ljlk_pose_scores = torch.ops.tmol_ljlk.ljlk_pose_scores
    print("ingest", pdb, flush=True)
    ch, rt, xyz = ingest.canonical_form_from_pdb(_pdb(pdb), co)
    full = ingest.pose_stack_from_layouts(
        ingest.block_layout_from_canonical_form(co, ch, rt, xyz))
    heavy = xyz.clone()
    for r in range(rt.shape[1]):
        t = int(rt[0, r])
        for name, k in co.atom_index[t].items():
            if name.startswith("H") or (len(name) > 1 and name[0].isdigit() and name[1] == "H"):
                heavy[0, r, k] = float("nan")
    ps = ingest.pose_stack_from_canonical_form(co, ch, rt, heavy, device="cuda")
    assert ps.coords.is_cuda and ps.block_type_ind.is_cuda
    assert ps.coords.shape == full.coords.shape
    dev = (ps.coords[0].cpu() - full.coords[0]).norm(dim=-1)
    assert not torch.isnan(ps.coords).any()
    assert float(dev.max()) < 1e-1 and float(dev.mean()) < 1e-3
    from tmol_amd.pose import PoseStack

    term = LJLKEnergyTerm(device="cuda")
    e_full, _ = ljlk_pose_scores(*pose_op_args(PoseStack(full.poses, device="cuda"), term))
    e_built, _ = ljlk_pose_scores(*pose_op_args(ps, term))
    assert torch.allclose(e_built.cpu(), e_full.cpu(), rtol=2e-3, atol=2e-2)


def test_large_batch_properties(co):
    """512 poses (256 copies each of 1ubq and 6DMZ with different random
    masks): building twice is idempotent, given atoms pass through
    bit-exactly, and every pose's output matches that of the same pose
    built alone."""
    print("leaf atoms batch 512", flush=True)
    lays = []
    for name in ("1ubq.pdb", "6DMZ_A.pdb"):
        ch, rt, xyz = ingest.canonical_form_from_pdb(_pdb(name), co)
        lays += ingest.block_layout_from_canonical_form(co, ch, rt, xyz)
    base = ingest.pose_stack_from_layouts(lays)
    _, tab = ingest.leaf_op_args(base, co.db, lays)
    rng = numpy.random.default_rng(5)
    big = []
    for k in range(512):
        L = lays[k % 2]
        m = []
        for b, r in enumerate(L["rts"]):
            lf = tab.is_leaf[base.packed_block_types.index[r.name]][: r.n_atoms]
            m.append(lf & (rng.random(r.n_atoms) < 0.8))
        big.append(dict(L, missing=m))
    ps = ingest.pose_stack_from_layouts(big)
    args, _ = ingest.leaf_op_args(ps, co.db, big)
    da = _dev(args)
    out = ingest.gen_pose_leaf_atoms(*da)
    given = ~args[2].cuda()
    real = torch.zeros_like(given)
    for p, L in enumerate(big):
        real[p, : sum(r.n_atoms for r in L["rts"])] = True
    keep = given & real
    assert torch.equal(out[keep], da[0][keep])
    da2 = list(da)
    da2[0] = out.clone()
    out2 = ingest.gen_pose_leaf_atoms(*da2)
    assert torch.equal(torch.isnan(out2), torch.isnan(out))
    assert torch.equal(out2.nan_to_num(0), out.nan_to_num(0))
    for p in (0, 1, 257, 510):
        one = [big[p]]
        ps1 = ingest.pose_stack_from_layouts(one)
        a1, _ = ingest.leaf_op_args(ps1, co.db, one)
        o1 = ingest.gen_pose_leaf_atoms(*_dev(a1))
        n = o1.shape[1]
        assert torch.equal(o1[0].nan_to_num(0), out[p, :n].nan_to_num(0))


@pytest.mark.parametrize("amax", [64, 100])
def test_wide_block_type_tables(co, amax):
    """The same poses with the block-type tables padded to ``amax`` atom
    slots (one block per wave pass, lanes striding over the slots when
    amax > 64): forward and backward identical to the unpadded call."""
    print("leaf atoms amax", amax, flush=True)
    ps, args = _random_missing(co, torch.float32, seed=7)
    A0 = args[1].shape[2]

    def pad(t, dim, value):
        shape = list(t.shape)
        shape[dim] = amax - A0
        return torch.cat([t, torch.full(shape, value, dtype=t.dtype)], dim=dim)

    wide = list(args)
    wide[1] = pad(args[1], 2, False)
    wide[7] = pad(args[7], 2, -1)
    wide[8] = pad(args[8], 1, -1)
    wide[9] = pad(args[9], 1, 0.0)
    wide[10] = pad(args[10], 1, -1)
    wide[11] = pad(args[11], 1, 0.0)
    outs, grads = [], []
    for a in (args, wide):
        X = a[0].cuda().requires_grad_(True)
        da = _dev(a)
        da[0] = X
        out = ingest.gen_pose_leaf_atoms(*da)
        w = torch.randn(out.shape, generator=torch.Generator().manual_seed(2)).cuda()
        (out.nan_to_num(0) * w).sum().backward()
        outs.append(out.detach().cpu())
        grads.append(X.grad.cpu())
    assert torch.equal(outs[0].nan_to_num(0), outs[1].nan_to_num(0))
    assert torch.equal(torch.isnan(outs[0]), torch.isnan(outs[1]))
    assert torch.allclose(grads[0], grads[1], rtol=1e-6, atol=1e-6)


def test_pose_stack_from_pdb(co):
    """The top-level entry from a file name with a residue range: the
    interior residues' atoms (hydrogens included, as given) equal the
    deposited ones and the new termini are built and finite."""
    print("pose_stack_from_pdb 1ubq 10..40", flush=True)
    ps = ingest.pose_stack_from_pdb(os.path.join(GOLDEN, "1ubq.pdb"), "cuda",
                                    residue_start=10, residue_end=40, co=co)
    assert ps.n_poses == 1 and ps.max_n_blocks == 30
    assert not torch.isnan(ps.coords).any()
    rts = ps.poses[0].residue_types
    assert rts[0].is_nterm and rts[-1].is_cterm
    full = ingest.pose_stack_from_layouts(ingest.block_layout_from_canonical_form(
        co, *ingest.canonical_form_from_pdb(_pdb("1ubq.pdb"), co)))
    for b in range(1, 29):
        assert numpy.allclose(ps.poses[0].coords[b], full.poses[0].coords[b + 10], atol=1e-4)


@pytest.mark.parametrize("key,value", [
    ("btype", "T"), ("btype", -2), ("bt_n", "A1"), ("bt_n", -1), ("down", "n"), ("down", -2),
    ("anc0", "n"), ("anc1", "C"), ("anc2", "A"), ("anc_b0", -2), ("anc_b1", -2), ("irc0", "B"),
    ("irc0", -2), ("irc1", "C"), ("boff", "NA"), ("boff", -1), ("pad", 0)])
@pytest.mark.parametrize("at", [0, -1])
def test_table_check_equals_the_tensor_checks(co, key, value, at):
    """One table entry out of range, first or last of its table: the kernel's
    check raises what the tensor form of the checks raises on the host."""
    _same_refusal(co, [(key, value)], at)


@pytest.mark.parametrize("faults", [
    [("boff", -1), ("anc0", -2)], [("pad", 0), ("bt_n", "A1")], [("boff", "NA"), ("pad", 0)],
    [("btype", "T"), ("boff", -1)], [("down", "n"), ("irc0", "B")], [("anc2", "A"), ("anc_b0", -2)]],
    ids=lambda f: "+".join(k for k, _ in f))
@pytest.mark.parametrize("at", [0, -1])
def test_several_tables_out_of_range(co, faults, at):
    """Two tables at once: every range check that fails is named, in order,
    and the checks that index with checked values only where none failed."""
    _same_refusal(co, faults, at)


def _same_refusal(co, faults, at):
    _, args = _random_missing(co, torch.float64)
    keys = ("orig", "bmiss", "pmiss", "boff", "btype", "irc", "bt_n", "down", "anc",
            "geom", "anc_b", "geom_b")
    k = {n: (torch.as_tensor(t).clone()) for n, t in zip(keys, args)}
    P, NA = k["orig"].shape[:2]
    B, A = k["bmiss"].shape[1:]
    C, T = k["irc"].shape[2], k["bt_n"].shape[0]
    for key, value in faults:
        name = key.rstrip("012")
        v = {"T": T, "A1": A + 1, "n": A, "A": A, "C": C, "B": B, "NA": NA}.get(value, value)
        if key == "pad":  # a connection to a block that does not exist
            pose = int((k["btype"] < 0).any(dim=1).nonzero()[0, 0])
            k["irc"][pose, 0, 0, 0] = int((k["btype"][pose] < 0).nonzero()[at, 0])
            k["irc"][pose, 0, 0, 1] = 0
        elif key == "boff":
            b = (k["btype"].view(-1) >= 0).nonzero()[at, 0]
            k["boff"].view(-1)[b] = v
        elif key[-1] in "012":
            row = k[name].view(-1, k[name].shape[-1])[at]
            row[1 if key.startswith("anc") and key[-1] == "2" else 0] = 0
            row[int(key[-1])] = v
        else:
            k[name].view(-1)[at] = v
    with pytest.raises(ingest.ops.LJLKLibraryError) as want:
        ingest._validate_leaf_tables(k, P, NA, B, A, C)
    with pytest.raises(ingest.ops.LJLKLibraryError) as got:
        ingest.gen_pose_leaf_atoms(*[k[n].cuda() for n in keys])
    assert str(got.value) == str(want.value)


@pytest.mark.parametrize("mask_dtype", [torch.bool, torch.uint8])
def test_masks_cleared_between_forward_and_backward(co, mask_dtype):
    """A program that marks the built atoms as present before it calls
    backward gets the gradient of the atoms that the forward built."""
    _, args = _random_missing(co, torch.float64)
    grads = []
    for clear in (False, True):
        da = _dev(args)
        da[1], da[2] = da[1].to(mask_dtype), da[2].to(mask_dtype)
        X = da[0] = da[0].clone().requires_grad_(True)
        out = ingest.gen_pose_leaf_atoms(*da)
        if clear:
            da[1].zero_()
            da[2].zero_()
        w = torch.randn(out.shape, dtype=out.dtype, generator=torch.Generator().manual_seed(4))
        (out.nan_to_num(0) * w.cuda()).sum().backward()
        grads.append(X.grad)
    # the same kernels on the same inputs; atomic sums in another order
    assert torch.allclose(grads[0], grads[1], rtol=1e-12, atol=1e-12)


def _reshaped(args, name):
    a = list(args)
    if name == "bt_n":  # [T, 2]
        a[6] = torch.cat([a[6], a[6]]).view(-1, 2)
    elif name == "boff":  # [B, P]
        a[3] = a[3].t().contiguous()
    else:  # irc [P, B * C, 1, 2]
        a[5] = a[5].flatten(1, 2).unsqueeze(2)
    return a


@pytest.mark.parametrize("name", ["bt_n", "boff", "irc"])
def test_table_shapes_refused(co, name):
    """Tables of the right size in another shape are refused, not read in
    the order of their words."""
    _, args = _random_missing(co, torch.float32)
    assert args[3].shape[0] != args[3].shape[1]
    with pytest.raises((RuntimeError, IndexError)):
        ingest.gen_pose_leaf_atoms(*_dev(_reshaped(args, name)))


def test_block_offsets_with_a_leading_one(co):
    """[1, P, B] block offsets are the [P, B] table."""
    _, args = _random_missing(co, torch.float32)
    want = ingest.gen_pose_leaf_atoms(*_dev(args))
    args[3] = args[3].unsqueeze(0)
    got = ingest.gen_pose_leaf_atoms(*_dev(args))
    assert torch.equal(got.nan_to_num(0), want.nan_to_num(0))
