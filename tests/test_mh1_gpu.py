"""MH-1 (MACE_Nonlinear) on the GPU against the float64 oracle
(oracle/mh1_oracle.py, pinned in tests/test_mh1_oracle.py).

The HIP path runs in FP32; the bars are the north star's: energy 1e-5
eV/atom, forces 1e-4 eV/A, stress 1e-6 eV/A^3, with the reference's own
MH-1 float32 comparisons (test_mh1.py:429-463, 1e-3 absolute on generated
float32 paths) far looser.  Models: cutoff on the features (l_max 2 and 3),
cutoff on the weights with Agnesi distances, a linear bias and ZBL, and the
64/32-channel l_max-3 member.  Stage checks (up-projection, messages,
density, layer features, edge weights) localise a failure.
"""

import json

import numpy as np
import pytest

from oracle import mh1_oracle as mo
from oracle import oracle
from symmetrix import random_mh1, systems

pytestmark = pytest.mark.gpu

# mh1_tiny_l2e (2e node and edge features in the second interaction) is
# outside the family's compiled convolution structures: its convolutions run
# the table-driven kernels; mh1_tiny_mlp32 (one 32-wide LayerNorm stage) and
# mh1_tiny_mlp4 (four stages: the LDS-tile MLP kernels) cover the edge-MLP forms
TINY = ["mh1_tiny", "mh1_tiny_l3", "mh1_tiny_raw", "mh1_tiny_l2e", "mh1_tiny_mlp32", "mh1_tiny_mlp4"]


@pytest.fixture(scope="module")
def paths(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("mh1gpu"))
    return {n: random_mh1.cached_mh1(n, directory=d) for n in TINY + ["mh1_medium"]}


def _say(msg):
    print(msg, flush=True)


def _random_system(model, n, L, seed, min_dist=1.2):
    rng = np.random.default_rng(seed)
    pos = np.zeros((n, 3))
    for i in range(n):
        while True:
            p = rng.random(3) * L
            d = pos[:i] - p
            d -= L * np.rint(d / L)
            if i == 0 or np.min(np.linalg.norm(d, axis=1)) > min_dist:
                pos[i] = p
                break
    nums = rng.choice(model.atomic_numbers, n)
    return pos, np.eye(3) * L, model.types_of(nums)


def _graph(model, pos, cell):
    g = oracle.neighbor_graph(pos, cell, model.r_cut)
    xyz, r = oracle.prepared_geometry(g, cell, pos, pos, 1e3)
    return g, xyz, r


def _gpu(path, types, g, xyz, r):
    from symmetrix.mace_nonlinear import MACENonlinearKokkosFloat
    ev = MACENonlinearKokkosFloat(path)
    src = g["sources"]
    ev.compute_node_energies_forces(len(types), types, g["num_neigh"], src, types[src], xyz, r)
    return ev, ev.node_energies, ev.node_forces.reshape(-1, 3)


def _compare(model, path, pos, cell, types, stages=False):
    g, xyz, r = _graph(model, pos, cell)
    n = len(types)
    _say("mh1 case: %s, %d atoms, %d edges" % (path.split("/")[-1], n, len(r)))
    e_ref, f_ref = model.evaluate(types, g["receivers"], g["sources"], xyz)
    ev, e, f = _gpu(path, types, g, xyz, r)
    vol = abs(np.linalg.det(cell))
    F = mo.reduce_forces(n, g["receivers"], g["sources"], f)
    F_ref = mo.reduce_forces(n, g["receivers"], g["sources"], f_ref)
    S = mo.reduce_stress(f, xyz, vol)
    S_ref = mo.reduce_stress(f_ref, xyz, vol)
    de = abs(e.sum() - e_ref.sum()) / n
    dn = np.abs(e - e_ref).max()
    dF = np.abs(F - F_ref).max()
    dS = np.abs(S - S_ref).max()
    _say("  |dE|/atom %.2e  max|dE_i| %.2e  max|dF| %.2e (|F| %.2f)  max|dS| %.2e" %
         (de, dn, dF, np.abs(F_ref).max(), dS))
    if stages:
        st = model.stages["states"]
        for k in range(len(st)):
            for name, ref in (("up", st[k]["up"]), ("msg", st[k]["msg"]), ("density", st[k]["density"]),
                              ("w", st[k]["wraw"]), ("features", model.stages["layer_features"][k])):
                got = ev._stage("%s%d" % (name, k)).reshape(np.shape(ref))
                err = np.abs(got - ref).max() / max(1.0, np.abs(ref).max())
                _say("  stage %s%d: scaled max err %.2e" % (name, k, err))
                assert err < 2e-5, (name, k, err)
    assert de < 1e-5
    assert dn < 1e-4
    assert dF < 1e-4
    assert dS < 1e-6
    return ev


@pytest.mark.parametrize("name", TINY)
def test_mh1_matches_oracle(paths, name):
    model = mo.MH1Oracle(paths[name])
    pos, cell, types = _random_system(model, 40, 8.0, seed=3)
    _compare(model, paths[name], pos, cell, types, stages=True)


def test_mh1_medium_member_matches_oracle(paths):
    model = mo.MH1Oracle(paths["mh1_medium"])
    s = systems.irregular_box(120, seed=2)
    pos, cell = np.asarray(s["positions"]), np.asarray(s["cell"])
    _compare(model, paths["mh1_medium"], pos, cell, model.types_of(s["numbers"]))


def test_mh1_repeat_calls_and_graph_changes(paths):
    """Two calls on one evaluator (workspace reuse, a smaller second graph),
    then the first graph again: identical results."""
    path = paths["mh1_tiny"]
    model = mo.MH1Oracle(path)
    pos, cell, types = _random_system(model, 40, 8.0, seed=5)
    g, xyz, r = _graph(model, pos, cell)
    from symmetrix.mace_nonlinear import MACENonlinearKokkosFloat
    ev = MACENonlinearKokkosFloat(path)
    src = g["sources"]
    ev.compute_node_energies_forces(len(types), types, g["num_neigh"], src, types[src], xyz, r)
    e1, f1 = ev.node_energies.copy(), ev.node_forces.copy()
    pos2, cell2, types2 = _random_system(model, 12, 6.0, seed=6)
    g2, xyz2, r2 = _graph(model, pos2, cell2)
    ev.compute_node_energies_forces(len(types2), types2, g2["num_neigh"], g2["sources"], types2[g2["sources"]],
                                    xyz2, r2)
    e_ref, _ = model.evaluate(types2, g2["receivers"], g2["sources"], xyz2)
    assert np.abs(ev.node_energies - e_ref).max() < 1e-4
    ev.compute_node_energies_forces(len(types), types, g["num_neigh"], src, types[src], xyz, r)
    assert np.array_equal(ev.node_energies, e1) and np.array_equal(ev.node_forces, f1)


def test_mh1_isolated_atoms_and_empty_graph(paths):
    """Atoms without neighbours get their atomic energy plus the readouts of
    the embedding alone; an empty graph is valid."""
    path = paths["mh1_tiny"]
    model = mo.MH1Oracle(path)
    types = np.array([0, 1, 2], dtype=np.int32)
    empty = np.zeros((0, 3))
    from symmetrix.mace_nonlinear import MACENonlinearKokkosFloat
    ev = MACENonlinearKokkosFloat(path)
    ev.compute_node_energies_forces(3, types, np.zeros(3, np.int32), np.zeros(0, np.int32),
                                    np.zeros(0, np.int32), empty, np.zeros(0))
    e_ref, _ = model.evaluate(types, np.zeros(0, np.int64), np.zeros(0, np.int64), empty)
    assert np.abs(ev.node_energies - e_ref).max() < 1e-5
    assert ev.node_forces.size == 0


def test_mh1_rejects_bad_graphs(paths):
    from symmetrix.mace_nonlinear import MACENonlinearKokkosFloat
    ev = MACENonlinearKokkosFloat(paths["mh1_tiny"])
    t = np.array([0, 1], dtype=np.int32)
    xyz = np.array([[1.0, 0.0, 0.0], [-1.0, 0.0, 0.0]])
    r = np.ones(2)
    ok = dict(num_nodes=2, node_types=t, num_neigh=[1, 1], neigh_indices=[1, 0], neigh_types=[1, 0], xyz=xyz, r=r)
    ev.compute_node_energies_forces(**ok)
    for bad in (dict(neigh_types=[0, 0]), dict(neigh_indices=[2, 0]), dict(num_neigh=[2, 1]),
                dict(r=np.array([1.0, np.nan])), dict(node_types=np.array([0, 9], np.int32))):
        args = dict(ok)
        args.update(bad)
        with pytest.raises(ValueError):
            ev.compute_node_energies_forces(**args)
    # the evaluator still works after the refusals
    ev.compute_node_energies_forces(**ok)
    assert np.all(np.isfinite(ev.node_energies))


def test_mh1_family_facts(paths):
    from symmetrix.mace_nonlinear import MACENonlinearKokkosFloat
    ev = MACENonlinearKokkosFloat(paths["mh1_medium"])
    assert ev.is_mh1_family and ev.mh1_family_rejection_reason == ""
    assert (ev.mh1_node_channels, ev.mh1_edge_channels, ev.mh1_radial_size, ev.mh1_l_max) == (64, 32, 8, 3)
    assert ev.atomic_numbers == [1, 6, 7, 8, 13, 14, 22, 26, 29, 38]
    model = mo.MH1Oracle(paths["mh1_medium"])
    assert np.allclose(ev.atomic_energies, model.atomic_energies)


def _oracle_system(model, pos, cell, pbc, types):
    """Oracle E, F, S (3x3) on the graph r < r_cut (brute force over the
    images that can reach the cutoff)."""
    n = len(pos)
    recv, src, vec = [], [], []
    rng = [range(-2, 3) if p else range(0, 1) for p in pbc]
    for i in range(n):
        for j in range(n):
            for a in rng[0]:
                for b in rng[1]:
                    for c in rng[2]:
                        d = pos[j] - pos[i] + np.array([a, b, c]) @ cell
                        r = np.linalg.norm(d)
                        if 0.0 < r < model.r_cut:
                            recv.append(i)
                            src.append(j)
                            vec.append(d)
    recv, src, vec = np.array(recv), np.array(src), np.array(vec).reshape(-1, 3)
    order = np.argsort(recv, kind="stable")
    recv, src, vec = recv[order], src[order], vec[order]
    e, f = model.evaluate(types, recv, src, vec)
    F = mo.reduce_forces(n, recv, src, f)
    vol = abs(np.linalg.det(cell)) if all(pbc) else None
    S = mo.reduce_stress(f, vec, vol) if vol else None
    return e.sum(), F, S


def test_mh1_calculator_matches_oracle_and_reuses_its_graph(paths):
    from symmetrix.calculator import Symmetrix, full_3x3_to_voigt_6_stress
    path = paths["mh1_tiny_raw"]
    model = mo.MH1Oracle(path)
    pos, cell, types = _random_system(model, 24, 7.5, seed=11)
    numbers = np.array(model.atomic_numbers)[types]
    calc = Symmetrix(path, neighbor_skin=0.5)
    for step in range(3):
        # moves well inside half the skin: the graph is reused
        p = pos + 0.02 * step * np.random.default_rng(step).normal(size=pos.shape)
        res = calc.calculate({"numbers": numbers, "positions": p, "cell": cell, "pbc": [True] * 3},
                             ["energy", "forces", "stress"])
        e, F, S = _oracle_system(model, p, cell, [True] * 3, types)
        _say("mh1 calculator step %d: |dE| %.2e max|dF| %.2e max|dS| %.2e" %
             (step, abs(res["energy"] - e), np.abs(res["forces"] - F).max(),
              np.abs(res["stress"] - full_3x3_to_voigt_6_stress(S)).max()))
        assert abs(res["energy"] - e) / len(p) < 1e-5
        assert np.abs(res["forces"] - F).max() < 1e-4
        assert np.abs(res["stress"] - full_3x3_to_voigt_6_stress(S)).max() < 1e-6
    assert calc.neighbor_cache_build_count == 1 and calc.neighbor_cache_reuse_count == 2


def test_mh1_calculator_open_cluster(paths):
    from symmetrix.calculator import Symmetrix
    path = paths["mh1_tiny_l3"]
    model = mo.MH1Oracle(path)
    pos, _, types = _random_system(model, 16, 6.0, seed=12)
    numbers = np.array(model.atomic_numbers)[types]
    calc = Symmetrix(path)
    res = calc.calculate({"numbers": numbers, "positions": pos, "cell": np.zeros((3, 3)), "pbc": [False] * 3},
                         ["energy", "forces"])
    e, F, _ = _oracle_system(model, pos, np.eye(3), [False] * 3, types)
    assert abs(res["energy"] - e) / len(pos) < 1e-5
    assert np.abs(res["forces"] - F).max() < 1e-4


def test_mh1_convolution_kernel_choice(paths):
    """Family convolutions run the compiled-structure kernels; a structure
    outside them (2e edge features) runs the table-driven ones."""
    from symmetrix.mace_nonlinear import MACENonlinearKokkosFloat
    for name, table in (("mh1_tiny_l3", False), ("mh1_tiny_l2e", True)):
        model = mo.MH1Oracle(paths[name])
        pos, cell, types = _random_system(model, 12, 6.0, seed=13)
        g, xyz, r = _graph(model, pos, cell)
        ev = MACENonlinearKokkosFloat(paths[name])
        ev._set_kernel_timing(True)
        ev.compute_node_energies_forces(len(types), types, g["num_neigh"], g["sources"], types[g["sources"]], xyz, r)
        names = set(ev._kernel_timing())
        assert ("mh1_tp_forward_table" in names) == table
        assert ("mh1_tp_reverse_table" in names) == table
        assert "mh1_tp_forward" in names if not table else True


def _neighbor_arrays(ev, pos, cell):
    from symmetrix.neighbors import neighbor_list_ijS
    recv, src, shifts = neighbor_list_ijS(pos, cell, np.array([True] * 3), ev.r_cut)
    xyz = pos[src] - pos[recv] + shifts @ cell
    r = np.sqrt(np.einsum("ij,ij->i", xyz, xyz))
    keep = r < ev.r_cut
    return recv[keep], src[keep], np.ascontiguousarray(xyz[keep]), r[keep]


def _gpu_system(ev, numbers, pos, cell):
    lut = {z: i for i, z in enumerate(ev.atomic_numbers)}
    types = np.array([lut[int(z)] for z in numbers], np.int32)
    recv, src, xyz, r = _neighbor_arrays(ev, pos, cell)
    n = len(types)
    ev.compute_node_energies_forces(n, types, np.bincount(recv, minlength=n).astype(np.int32), src, types[src],
                                    xyz.reshape(-1), r)
    nf = ev.node_forces.reshape(-1, 3)
    F = mo.reduce_forces(n, recv, src, nf)
    S = mo.reduce_stress(nf, xyz, abs(np.linalg.det(cell)))
    return ev.node_energies.copy(), F, S, len(r)


def test_mh1_benchmark_size_unperturbed_crystal(paths):
    """The bench's 5,000-atom SrTiO3 cell without displacements: every site
    is an inversion centre, so each atom's energy equals its site's energy in
    the oracle's 3x3x3 cell, all forces vanish and the stress equals the
    oracle's (r_cut 6.0 A: 369k edges through every MH-1 kernel)."""
    from symmetrix.mace_nonlinear import MACENonlinearKokkosFloat
    path = paths["mh1_medium"]
    model = mo.MH1Oracle(path)
    small = systems.srtio3_supercell(3, sigma=0.0)
    ps, cs = np.asarray(small["positions"]), np.asarray(small["cell"])
    ts = model.types_of(small["numbers"])
    g, xyz, r = _graph(model, ps, cs)
    e_ref, f_ref = model.evaluate(ts, g["receivers"], g["sources"], xyz)
    S_ref = mo.reduce_stress(f_ref, xyz, abs(np.linalg.det(cs)))
    site = {int(z): e_ref[np.asarray(small["numbers"]) == z].mean() for z in set(small["numbers"])}
    big = systems.srtio3_supercell(10, sigma=0.0)
    ev = MACENonlinearKokkosFloat(path)
    e, F, S, E = _gpu_system(ev, big["numbers"], np.asarray(big["positions"]), np.asarray(big["cell"]))
    want = np.array([site[int(z)] for z in big["numbers"]])
    _say("mh1 unperturbed 10x10x10: %d edges, max|dE_i| %.2e, max|F| %.2e, max|dS| %.2e"
         % (E, np.abs(e - want).max(), np.abs(F).max(), np.abs(S - S_ref).max()))
    assert E > 300000
    assert np.abs(e - want).max() < 1e-4
    assert abs(e.sum() - want.sum()) / len(e) < 1e-5
    assert np.abs(F).max() < 1e-4
    assert np.abs(S - S_ref).max() < 1e-6


def test_mh1_benchmark_size_rotation_and_translation(paths):
    """The perturbed 5,000-atom cell rotated and shifted as a whole: node
    energies unchanged and forces rotated, within the FP32 bars."""
    from symmetrix import e3
    from symmetrix.mace_nonlinear import MACENonlinearKokkosFloat
    ev = MACENonlinearKokkosFloat(paths["mh1_medium"])
    s = systems.srtio3_supercell(10, sigma=0.05, seed=0)
    pos, cell = np.asarray(s["positions"]), np.asarray(s["cell"])
    e0, F0, _, _ = _gpu_system(ev, s["numbers"], pos, cell)
    R = e3.random_rotation(np.random.default_rng(21))
    e1, F1, _, _ = _gpu_system(ev, s["numbers"], pos @ R.T + np.array([0.7, -1.3, 2.1]), cell @ R.T)
    _say("mh1 rotated 10x10x10: max|dE_i| %.2e, |dE|/atom %.2e, max|dF| %.2e (|F| %.2f)"
         % (np.abs(e1 - e0).max(), abs(e1.sum() - e0.sum()) / len(e0), np.abs(F1 - F0 @ R.T).max(),
            np.abs(F0).max()))
    # the bar is the energy per atom; single node energies carry the FP32
    # rounding of their own sums (two different rounding patterns here)
    assert abs(e1.sum() - e0.sum()) / len(e0) < 1e-5
    assert np.abs(e1 - e0).max() < 5e-4
    assert np.abs(F1 - F0 @ R.T).max() < 1e-4


@pytest.mark.parametrize("name", ["mh1_tiny", "mh1_tiny_mlp32", "mh1_medium"])
@pytest.mark.parametrize("n", [2, 3, 5, 6, 9])
def test_mh1_edge_mlp_at_tile_edges(paths, name, n):
    """Edge MLP outputs and forces of few edges (2, 6, 20, 30, 72: parts of a
    16-edge tile, whole tiles and a remainder).  Bound of a weight: each of at
    most four linears rounds a sum of at most 64 terms in FP32, 64 * 2^-24 of
    its scale, and 1e-6 in the root mean square (four linears, LayerNorm and
    SiLU of 1e-7 to 2e-7 each).  One linear without its weights' third bf16
    part exceeds that: the oracle on such weights is 1.4e-6 to 4.9e-6 off, and
    its forces mostly over 1.5e-6, their bound here."""
    model = mo.MH1Oracle(paths[name])
    rng = np.random.default_rng(n)
    sites = np.stack(np.meshgrid(*(np.arange(3),) * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    pos = sites * 1.4 + rng.uniform(-0.1, 0.1, size=(n, 3))
    cell = np.eye(3) * 30.0
    types = rng.integers(0, len(model.atomic_numbers), size=n).astype(np.int32)
    g, xyz, r = _graph(model, pos, cell)
    _, f_ref = model.evaluate(types, g["receivers"], g["sources"], xyz)
    ev, _, f = _gpu(paths[name], types, g, xyz, r)
    for k, state in enumerate(model.stages["states"]):
        ref = np.asarray(state["wraw"])
        got = ev._stage("w%d" % k).reshape(ref.shape)
        assert np.abs(got - ref).max() <= 4 * 64 * 2.0 ** -24 * max(1.0, np.abs(ref).max())
        assert np.mean((got - ref) ** 2) <= 1e-6 ** 2 * np.mean(ref ** 2)
    assert np.abs(f - f_ref).max() < 1e-4 * max(1.0, np.abs(f_ref).max())
    assert np.mean((f - f_ref) ** 2) <= 1.5e-6 ** 2 * np.mean(f_ref ** 2)


@pytest.mark.parametrize("name", ["mh1_tiny_mlp32", "mh1_medium"])
def test_mh1_edge_mlp_weight_beyond_bf16(paths, name, tmp_path):
    """A final-linear weight of 3.4e38, which rounds to infinity in bf16, gives
    what FP32 products give."""
    with open(paths[name]) as f:
        d = json.load(f)
    last = d["interactions"][0]["conv_tp_weights"]["layers"][-1]["weight"]
    cols, hidden = int(last["shape"][0]), int(last["shape"][1])
    last["values"][3 * hidden + 1] = 3.4e38
    path = str(tmp_path / "huge.json")
    with open(path, "w") as f:
        json.dump(d, f)
    model = mo.MH1Oracle(path)
    pos, cell, types = _random_system(model, 7, 8.0, 5)
    g, xyz, r = _graph(model, pos, cell)
    with np.errstate(all="ignore"):
        model.evaluate(types, g["receivers"], g["sources"], xyz)
    ev, _, _ = _gpu(path, types, g, xyz, r)
    ref = np.asarray(model.stages["states"][0]["wraw"]).reshape(-1, cols)
    got = ev._stage("w0").reshape(-1, cols)
    fits = np.abs(ref[:, 3]) < 3e38
    assert fits.sum() > len(r) // 2 and np.abs(ref[fits, 3]).max() > 1e37
    np.testing.assert_allclose(got[fits, 3], ref[fits, 3], rtol=4e-5)
    rest = np.arange(cols) != 3
    np.testing.assert_allclose(got[:, rest], ref[:, rest], rtol=0, atol=4 * 64 * 2.0 ** -24 * np.abs(ref[:, rest]).max())
