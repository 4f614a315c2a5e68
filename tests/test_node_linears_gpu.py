"""Node linears on the GPU against float64 products of the kernel's own inputs.

H1 = M0 H1_w per degree (the linear whose rows are every node's): row counts
at the edges of its 16-row tiles and 128-row sets, and sizes that take each
form of the kernel (FP32 waves of 32 and 64 columns, workgroups of 32, 64 and
128 columns on bf16 parts).

Bound: a sum over K inputs rounds an FP32 accumulator K times (FP32 products)
or 6 K / 32 times (products of parts, which drop less than 2^-25 |x w| too),
each time by at most 2^-24 of a partial sum, itself at most sum |x w|.
"""

import functools
import json

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@functools.lru_cache(maxsize=None)
def _h1_weights(path):
    with open(path) as f:
        return np.asarray(json.load(f)["H1_weights"])


def _sparse(n, seed):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0) - 1e-9))
    sites = np.stack(np.meshgrid(*(np.arange(m),) * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    return sites * 4.6 + rng.uniform(-0.4, 0.4, size=(n, 3)), np.eye(3) * 4.6 * m, rng.choice([8, 22, 38], size=n)


@pytest.mark.parametrize("model,n", [("tiny", 1), ("tiny", 16), ("tiny", 43), ("tiny", 129), ("tiny", 12001),
                                     ("medium", 1), ("medium", 15), ("medium", 17), ("medium", 128), ("medium", 1303),
                                     ("medium", 3001), ("medium", 5003), ("medium", 17001)])
def test_h1_linear_against_float64(model, n, tiny_model_path, medium_model_path):
    from symmetrix.mace_kokkos import MACEKokkosFloat
    path = tiny_model_path if model == "tiny" else medium_model_path
    pos, cell, numbers = _sparse(n, n)
    ev = MACEKokkosFloat(path)
    lut = {z: i for i, z in enumerate(ev.atomic_numbers)}
    types = np.array([lut[int(z)] for z in numbers], np.int32)
    g = ev._prepare_periodic_factorized_graph(types, pos, cell, np.linalg.inv(cell), ev.r_cut + 0.5)
    ev._compute_prepared_factorized_positions(g["generation"], pos)
    C, L = ev.num_channels, ev.L_max
    m0 = ev._stage("M0").reshape(n, (L + 1) ** 2, C).astype(np.float64)
    h1 = ev._stage("H1").reshape(n, (L + 1) ** 2, C)
    w = _h1_weights(path).reshape(L + 1, C, C)
    assert np.abs(m0).max() > 0
    for l in range(L + 1):
        x = m0[:, l * l:(l + 1) ** 2]
        bound = (C + 1) * 2.0 ** -24 * (np.abs(x) @ np.abs(w[l])) + 1e-30
        assert np.all(np.abs(h1[:, l * l:(l + 1) ** 2] - x @ w[l]) <= bound)


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
