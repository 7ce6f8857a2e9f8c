"""Parity of the gfx950 reinitialisation (dcl_reinitialize, LevelSetReinitialize)
with the oracle: phi bit for bit over the whole window and the band in the
same order (both run the reference's heap with its comparisons and the same
second-order updates in the same operand order).  Cases: a scaled sphere, a
perturbed sphere (many second-order / first-order switches and near-ties),
an axis plane (exact ties along the plane), a 2D circle, a band that
touches the window's edge, a batch of level sets of different sizes run
side by side, an empty record list, and a heap too small (an error)."""
import numpy as np
import pytest
import torch

import oracle as O
import dcell_amd as D
from dcell_amd import metrics as M
from helpers import owin, to_dev, to_np

pytestmark = pytest.mark.gpu


def _case(phi, win, width=8.0):
    recs = O.irregular_nodes(phi, owin(win), O.band_compact(phi, owin(win), width))
    dev_recs = torch.from_numpy(recs.view(np.uint8).reshape(-1).copy()).to("cuda:0")
    return recs, dev_recs


def _check(phi, win, recs, got_phi, got_band):
    ref_phi, ref_band = O.reinitialize(phi, owin(win), recs)
    assert to_np(got_phi).tobytes() == ref_phi.tobytes()
    np.testing.assert_array_equal(to_np(got_band), ref_band)


def _sphere(n, c, r, scale, noise=0.0, seed=0):
    z, y, x = np.meshgrid(*(np.arange(n, dtype=float),) * 3, indexing="ij")
    sdf = np.sqrt((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2) - r
    return scale * sdf + noise * np.random.default_rng(seed).normal(size=sdf.shape)


@pytest.mark.parametrize("noise", [0.0, 0.3])
def test_reinit_sphere_bit_exact(dev, noise):
    n = 48
    win = D.GridWindow((2, -3, 5), (n, n, n), (1.0, 1.0, 1.0))
    phi = _sphere(n, (23.3, 22.6, 24.2), 13.4, 2.0, noise, seed=4)
    recs, drecs = _case(phi, win)
    dphi = to_dev(phi)
    (band,) = M.reinitialize([(dphi, win, drecs, len(recs))])
    _check(phi, win, recs, dphi, band)


def test_reinit_plane_and_edge(dev):
    n = 40
    win = D.GridWindow((0, 0, 0), (n, n, 24), (1.0, 1.0, 1.0))
    z, y, x = np.meshgrid(np.arange(24.0), np.arange(float(n)), np.arange(float(n)), indexing="ij")
    phi = 3.0 * (y - 20.3)  # a plane; the band reaches the x and z faces of the window
    recs, drecs = _case(phi, win)
    dphi = to_dev(phi)
    (band,) = M.reinitialize([(dphi, win, drecs, len(recs))])
    _check(phi, win, recs, dphi, band)


def test_reinit_circle_2d(dev):
    n = 96
    win = D.GridWindow((0, 0, 0), (n, n, 1), (1.0, 1.0, 1.0))
    y, x = np.meshgrid(np.arange(float(n)), np.arange(float(n)), indexing="ij")
    phi = 2.0 * (np.hypot(x - 47.3, y - 49.1) - 30.2)
    recs, drecs = _case(phi, win)
    dphi = to_dev(phi)
    (band,) = M.reinitialize([(dphi, win, drecs, len(recs))])
    _check(phi, win, recs, dphi, band)


def test_reinit_batch(dev):
    cells, host = [], []
    for i, n in enumerate((24, 40, 33, 56)):
        win = D.GridWindow((i, -i, 2 * i), (n, n + 1, n - 1), (1.0, 1.0, 1.0))
        phi = np.ascontiguousarray(_sphere(n, (n / 2 + 0.3, n / 2 - 0.2, n / 2), n / 4 + 0.1, 1.5, 0.1, seed=i)
                                   [: n - 1, :, :])
        phi = np.concatenate([phi, phi[:, :1, :]], axis=1)  # (n-1, n+1, n)
        recs, drecs = _case(phi, win)
        dphi = to_dev(phi)
        cells.append((dphi, win, drecs, len(recs)))
        host.append((phi, win, recs))
    bands = M.reinitialize(cells)
    for (phi, win, recs), (dphi, _, _, _), band in zip(host, cells, bands):
        _check(phi, win, recs, dphi, band)


@pytest.mark.parametrize("n", [(112, 112, 112), (128, 7, 24), (9, 61, 4), (301, 9, 1), (6, 5, 1), (7, 1, 9)])
def test_reinit_heap_levels_and_faces(dev, n):
    """A sphere whose heap is deeper than the part of it in LDS, and windows
    so thin that every node's stencil leaves them."""
    win = D.GridWindow((-3, 4, 1 if n[2] > 1 else 0), n, (1.0, 1.0, 1.0))
    if min(n) > 100:
        phi = _sphere(n[0], (55.3, 54.6, 56.2), 40.4, 1.7)
    else:
        z, y, x = np.meshgrid(*(np.arange(float(k)) for k in n[::-1]), indexing="ij")
        phi = 1.7 * (0.8 * (x - 0.47 * n[0]) + 0.5 * (y - 0.4 * n[1]) + 0.3 * (z - 0.6 * n[2]))
        phi = phi if n[2] > 1 else phi[0]
    phi = np.ascontiguousarray(phi)
    recs, drecs = _case(phi, win)
    dphi = to_dev(phi)
    (band,) = M.reinitialize([(dphi, win, drecs, len(recs))])
    _check(phi, win, recs, dphi, band)


def test_reinit_infinite_tentative_values(dev):
    """Tentative values that overflow to infinity fill a heap deeper than its
    part in LDS while ordinary nodes are accepted: the last entry, moved down at
    each pop, is infinite where the heap has no child.  A node between P along
    x and Q along y gets (2 P + 2 Q + sqrt((2 P + 2 Q)^2 - 8 (P^2 + Q^2))) / 4,
    whose first square rounds past the largest number for these two and the
    second sum does not."""
    P, Q = np.nextafter(2.0 ** 510, 0), 2.0 ** 510
    B = -2.0 * P - 2.0 * Q
    with np.errstate(over="ignore"):
        assert np.isinf(np.float64(B) * B) and np.isfinite(8.0 * (-1.0 + P * P + Q * Q))
    nx, ny = 260, 300
    win = D.GridWindow((0, 0, 0), (nx, ny, 1), (1.0, 1.0, 1.0))
    y, x = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    low = x == 5                                        # an ordinary front, pushed first
    high = (x >= 20) & ((x + y) % 2 == 0)
    phi = np.ones((ny, nx))
    at = np.concatenate([np.argwhere(low), np.argwhere(high)])
    recs = np.zeros(len(at), dtype=M.IRREGULAR_DTYPE)
    recs["pos"][:, 0], recs["pos"][:, 1] = at[:, 1], at[:, 0]
    recs["axis"] = recs["shift"] = -1
    recs["sign_center"] = 1
    recs["op"][:, 0] = np.where(at[:, 1] == 5, 0.25, np.where(at[:, 0] % 2 == 0, P, Q))
    drecs = torch.from_numpy(recs.view(np.uint8).reshape(-1).copy()).to("cuda:0")
    dphi = to_dev(phi)
    (band,) = M.reinitialize([(dphi, win, drecs, len(recs))], 6.0, 2.0 ** 600, heap_capacity=8 * len(recs))
    ref_phi, ref_band = O.reinitialize(phi, owin(win), recs, 6.0, 2.0 ** 600)
    assert len(ref_band) > len(recs) + 5 * ny           # the front was marched
    assert to_np(dphi).tobytes() == ref_phi.tobytes()
    np.testing.assert_array_equal(to_np(band), ref_band)


def test_reinit_empty_and_heap_error(dev):
    n = 20
    win = D.GridWindow((0, 0, 0), (n, n, n), (1.0, 1.0, 1.0))
    phi = _sphere(n, (9.5, 9.5, 9.5), 5.2, 1.0)
    dphi = to_dev(phi)
    empty = torch.zeros(0, dtype=torch.uint8, device="cuda:0")
    (band,) = M.reinitialize([(dphi, win, empty, 0)])
    assert band.shape[0] == 0
    assert np.array_equal(to_np(dphi), np.where(phi > 0, 7.5, -7.5))
    recs, drecs = _case(phi, win)
    with pytest.raises(RuntimeError, match="heap full"):
        M.reinitialize([(to_dev(phi), win, drecs, len(recs))], heap_capacity=8)
