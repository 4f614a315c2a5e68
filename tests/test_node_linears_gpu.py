"""Node linears on the GPU against float64 products of the kernels' own inputs.

A0 = Phi0 W per (type, l), H1 = M0 W and A1 = Phi1 W per l, and the reverse of
A1 (dPhi1 = A1_adj W^T): row counts at the edges of 16-row tiles and of the
workgroups' 64 and 128 rows, and sizes that take each form of the kernel, which
a case names: FP32 waves of 32, 64 and 128 columns, the FP32 workgroup, and at
256 channels the workgroups on bf16 parts.

Bound (test_bf16_parts.ROUNDING, which tells a lost product of parts): the root
mean square of the error is at most 1.5 * 2^-24 of that of sum |x w|.
"""

import functools
import json

import numpy as np
import pytest

from test_bf16_parts import ROUNDING

pytestmark = pytest.mark.gpu

# form of a linear: (kind, columns, rows) of a workgroup
W32, W64, W128 = (0, 32, 16), (0, 64, 16), (0, 128, 16)
SHARED = (1, 128, 128)
P64, P128_64, P128 = (2, 64, 64), (2, 128, 64), (2, 128, 128)


@functools.lru_cache(maxsize=None)
def _model(path):
    with open(path) as f:
        d = json.load(f)
    C = d["num_channels"]

    def f32(w):
        return np.asarray(w, np.float32).astype(np.float64)

    return (C, [[f32(b).reshape(C, C) for b in w] for w in d["A0_weights"]], f32(d["H1_weights"]).reshape(-1, C, C),
            [f32(w).reshape(-1, C) for w in d["A1_weights"]])


def _sparse(n, seed, choice):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0) - 1e-9))
    sites = np.stack(np.meshgrid(*(np.arange(m),) * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    return sites * 4.6 + rng.uniform(-0.4, 0.4, size=(n, 3)), np.eye(3) * 4.6 * m, rng.choice(choice, size=n)


def _error(y, x, w):
    """rms of y - x w over rms of |x| |w|"""
    ref, scale = x @ w, np.abs(x) @ np.abs(w)
    return np.sqrt(np.mean((y - ref) ** 2) / np.mean(scale ** 2))


# model, atoms, forms of A0, H1, A1 and the reverse of A1
CASES = [
    ("tiny", 1, W32, W32, W32, W32),
    ("tiny", 16, W32, W32, W32, W32),
    ("tiny", 43, W32, W32, W32, W32),
    ("tiny", 16451, W32, W32, W32, W32),
    ("medium", 1, W64, W64, W64, W64),
    ("medium", 15, W64, W64, W64, W64),
    ("medium", 17, W64, W64, W64, W64),
    ("medium", 128, W64, W64, W64, W64),
    ("medium", 1303, W64, W64, W64, W64),
    ("medium", 5003, W64, W64, W64, W128),
    ("medium", 12001, W128, W64, W64, SHARED),
    ("wide", 1, P64, P64, P64, P64),
    ("wide", 15, P64, P64, P64, P64),
    ("wide", 65, P64, P64, P64, P64),
    ("wide", 129, P64, P64, P64, P64),
    ("wide", 1203, P128_64, P64, P128_64, P128),
    ("wide", 2501, P128, P128_64, P128, P128),
    ("wide", 4003, P128, P128, P128, P128),
]


@pytest.mark.parametrize("model,n,a0,h1,a1,a1r", CASES)
def test_linears_against_float64(request, model, n, a0, h1, a1, a1r):
    from symmetrix.mace_kokkos import MACEKokkosFloat
    path = request.getfixturevalue(model + "_model_path")
    C, A0w, H1w, A1w = _model(path)
    ev = MACEKokkosFloat(path)
    pos, cell, numbers = _sparse(n, n, [1, 8] if model == "wide" else [8, 22, 38])
    lut = {z: i for i, z in enumerate(ev.atomic_numbers)}
    types = np.array([lut[int(z)] for z in numbers], np.int32)
    g = ev._prepare_periodic_factorized_graph(types, pos, cell, np.linalg.inv(cell), ev.r_cut + 0.5)
    ev._compute_prepared_factorized_positions(g["generation"], pos)
    forms = [tuple(int(v) for v in f) for f in ev._stage("linear_forms").reshape(4, 3)]
    print(model, n, forms, flush=True)
    assert forms == [a0, h1, a1, a1r]

    def stage(name):
        return ev._stage(name).reshape(n, -1, C).astype(np.float64)

    phi0, A0, m0, H1 = (stage(s) for s in ("Phi0", "A0", "M0", "H1"))
    phi1, A1, A1_adj, dphi1 = (stage(s) for s in ("Phi1", "A1", "A1_adj", "dPhi1"))
    errors, base = {}, 0
    for l in range(ev.l_max + 1):
        rows = slice(l * l, (l + 1) ** 2)
        for t in np.unique(types):
            errors["A0", l, t] = _error(A0[types == t][:, rows], phi0[types == t][:, rows], A0w[t][l])
        if l <= ev.L_max:
            errors["H1", l] = _error(H1[:, rows], m0[:, rows], H1w[l])
        K = len(A1w[l])
        cols = slice(base, base + (2 * l + 1) * K // C)  # Phi1 rows of an l: m, then its paths
        base = cols.stop
        errors["A1", l] = _error(A1[:, rows], phi1[:, cols].reshape(n, 2 * l + 1, K), A1w[l])
        errors["A1 reverse", l] = _error(dphi1[:, cols].reshape(n, 2 * l + 1, K), A1_adj[:, rows], A1w[l].T)
    print("largest rms error %.2e (%s)" % max((e, k) for k, e in errors.items()), flush=True)
    assert max(errors.values()) <= ROUNDING


def test_values_beyond_bf16_and_infinities_at_256_channels(wide_model_path, tmp_path):
    """An A0 weight of 3.4e38, which rounds to infinity in bf16, in one column:
    A0 is the float64 product, and where the product basis overflows on it, H1
    is infinite or NaN as FP32 sums are."""
    from symmetrix.mace_kokkos import MACEKokkosFloat
    with open(wide_model_path) as f:
        d = json.load(f)
    C, k, n = d["num_channels"], 7, 21
    for w in d["A0_weights"]:
        w[0][k * C + n] = 3.4e38
    path = str(tmp_path / "huge.json")
    with open(path, "w") as f:
        json.dump(d, f)
    ev = MACEKokkosFloat(path)
    rng = np.random.default_rng(2)
    pos = np.stack(np.meshgrid(*(np.arange(3),) * 3, indexing="ij"), -1).reshape(-1, 3) * 2.5
    pos = pos + rng.uniform(-0.3, 0.3, size=pos.shape)
    cell, types = np.eye(3) * 20.0, rng.integers(0, len(ev.atomic_numbers), size=27).astype(np.int32)
    g = ev._prepare_periodic_factorized_graph(types, pos, cell, np.linalg.inv(cell), ev.r_cut + 0.5)
    ev._compute_prepared_factorized_positions(g["generation"], pos)
    NY, NH = (ev.l_max + 1) ** 2, (ev.L_max + 1) ** 2
    phi, a0 = (ev._stage(s).reshape(27, NY, C).astype(np.float64) for s in ("Phi0", "A0"))
    w = np.asarray([x[0] for x in d["A0_weights"]]).reshape(-1, C, C)[types]
    ref = np.einsum("ak,akn->an", phi[:, 0], w)
    fits = np.abs(ref[:, n]) < 3e38
    assert fits.sum() > 13 and np.abs(ref[fits, n]).max() > 1e36
    np.testing.assert_allclose(a0[fits, 0, n], ref[fits, n], rtol=1e-5)
    other = np.arange(C) != n
    np.testing.assert_allclose(a0[:, 0, other], ref[:, other], rtol=0, atol=1e-6 * np.abs(ref[:, other]).max())
    # H1 per degree: an infinity in one channel of a row is one of its sign in every output, a NaN is NaN
    m0, h1 = (ev._stage(s).reshape(27, NH, C) for s in ("M0", "H1"))
    w1 = np.asarray(d["H1_weights"]).reshape(ev.L_max + 1, C, C)
    inf = np.isinf(m0[..., n])
    assert inf.any() and np.isfinite(m0[..., other]).all()
    for l in range(ev.L_max + 1):
        rows = slice(l * l, (l + 1) ** 2)
        sign = np.sign(m0[:, rows, n])[..., None] * np.sign(w1[l][n])
        np.testing.assert_array_equal(h1[:, rows][inf[:, rows]], (sign * np.inf)[inf[:, rows]])
        assert np.isnan(h1[:, rows][np.isnan(m0[:, rows, n])]).all()
