"""The precision form at the edges of its kernels: fewer spheres than a group
of lanes or a block, the smallest grids (three cells per axis for the stencil,
five for the list), 2D, and the device conversions between float64 positions
and integer cell + float32 offset (equal to the host's, value by value)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from jaxdem_amd import _lib as L
from jaxdem_amd import precision as PR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
def test_conversions_equal_the_host(device, dim):
    rng = np.random.Generator(np.random.PCG64(dim))
    box = np.array([7.3, 11.9, 5.1])[:dim]
    pos = rng.uniform(-3.0, 4.0, (4099, dim)) * box
    pos[:6] = [[0.0] * dim, box, -box, np.nextafter(box, 0.0), box * (1.0 - 1e-9), box * 1e-12]
    dims = np.array([5, 8, 3])[:dim]
    c, o = PR.to_cell_offset(pos, box, dims)
    hi, _, h = PR.cell_edges(box, dims)
    ctx = L.context_for(device)
    tp = torch.as_tensor(pos, device=device).contiguous()
    tc = torch.empty(pos.shape, dtype=torch.int32, device=device)
    to = torch.empty(pos.shape, dtype=torch.float32, device=device)
    edge, d32 = dims * h, dims.astype(np.int32)
    conv = (len(pos), dim, edge.ctypes.data, h.ctypes.data, hi.ctypes.data, d32.ctypes.data)
    ctx.check(ctx.lib.jdem_precise_import(ctx.ptr, tp.data_ptr(), *conv, tc.data_ptr(), to.data_ptr()), "import")
    assert np.array_equal(tc.cpu().numpy(), c) and np.array_equal(to.cpu().numpy(), o)
    ctx.check(ctx.lib.jdem_precise_export(ctx.ptr, tc.data_ptr(), to.data_ptr(), *conv, tp.data_ptr()), "export")
    assert np.array_equal(tp.cpu().numpy(), PR.from_cell_offset(c, o, box, dims))


def forces64(pos, rad, box):
    """float64 forces, energy and virial of unit springs, all pairs."""
    d = pos[:, None, :] - pos[None, :, :]
    d -= box * np.rint(d / box)
    r = np.sqrt((d * d).sum(-1))
    np.fill_diagonal(r, np.inf)
    s = np.maximum(rad[:, None] + rad[None, :] - r, 0.0)
    f = (s / r)[..., None] * np.where(np.isfinite(r)[..., None], d, 0.0)
    return f.sum(1), 0.25 * (s * s).sum(), 0.5 * np.einsum("ijk,ijl->kl", d, f)


@pytest.mark.parametrize("skin", [0.0, 0.05, 0.3])
@pytest.mark.parametrize("dim,N,phi", [(3, 9, 0.25), (3, 65, 0.6), (3, 257, 0.66), (2, 15, 0.7), (2, 63, 0.84),
                                       (3, 900, 2.5), (2, 700, 4.0)])
def test_small_systems_against_float64(device, dim, N, phi, skin):
    """A few FIRE steps; the forces, energy and virial reported for the final
    configuration are those of its float64 positions: a pair's float32 force
    is off by some 1e-7 of the overlap's sum of radii (1e-6 below), the sums
    of up to a hundred of them by no more than that times their number."""
    print(f"[precision] dim={dim} N={N} phi={phi} skin={skin}", flush=True)
    rng = np.random.Generator(np.random.PCG64(N))
    rad = np.where(np.arange(N) % 2 == 0, 0.5, 0.7)
    vol = (4.0 / 3.0 * np.pi * rad**3 if dim == 3 else np.pi * rad**2).sum()
    L0 = (vol / phi) ** (1.0 / dim)
    box = np.maximum(np.full(dim, L0), 4.25)
    kw = dict(max_steps=11, pe_tol=0.0, pe_diff_tol=-1.0, skin=skin, device=device, max_neighbors=400 if skin else None)
    r = PR.minimize_precise(rng.uniform(0.0, 1.0, (N, dim)) * box, rad, box, **kw)
    assert r["steps"] == 11
    F, e, W = forces64(r["pos"], rad.astype(np.float32).astype(np.float64), box)
    got = r["force"].cpu().numpy().astype(np.float64)
    assert np.abs(got - F).max() <= 1e-6 * 100
    assert np.abs(got - F).max() <= 1e-5 * max(np.abs(F).max(), 1.0)
    assert abs(r["pe"] * N - e) <= 1e-5 * max(e, 1e-3)
    assert np.abs(r["virial"] - W).max() <= 1e-5 * max(np.abs(W).max(), 1e-3)
    assert r["max_grad"] == np.abs(r["force"].cpu().numpy()).max()


@pytest.mark.parametrize("skin", [0.0, 0.05])
@pytest.mark.parametrize("max_steps", [0, 63, 64, 65, 2**63 - 2, 2**63 - 1])
def test_step_limits(device, max_steps, skin):
    """A limit at the edges of the loop's chunks, and none at all: the largest
    integers that the argument holds (the loop stops by its energy test)."""
    print(f"[precision] max_steps={max_steps} skin={skin}", flush=True)
    rng = np.random.Generator(np.random.PCG64(2))
    rad = np.where(np.arange(200) % 2 == 0, 0.5, 0.7)
    kw = dict(pe_tol=0.0, skin=skin, device=device)
    p, box = rng.uniform(0.0, 6.5, (200, 3)), np.full(3, 6.5)
    if max_steps < 100:
        r = PR.minimize_precise(p, rad, box, max_steps=max_steps, pe_diff_tol=-1.0, **kw)
        assert r["steps"] == max_steps
        return
    r = PR.minimize_precise(p, rad, box, max_steps=max_steps, pe_diff_tol=1e-3, **kw)
    want = PR.minimize_precise(p, rad, box, max_steps=5000, pe_diff_tol=1e-3, **kw)
    assert 0 < r["steps"] == want["steps"] < 5000 and np.array_equal(r["pos"], want["pos"])


@pytest.mark.parametrize("dim", [2, 3])
def test_points_among_spheres(device, dim):
    """A wavefront of points whose radius is minus zero, inside larger
    spheres: the list finds every partner that the stencil finds."""
    print(f"[precision] points dim={dim}", flush=True)
    rng = np.random.Generator(np.random.PCG64(dim))
    rad = np.concatenate([np.full(64, -0.0), rng.uniform(0.4, 0.6, 136)])
    box = np.full(dim, 12.0 if dim == 2 else 6.0)
    pos = rng.uniform(0.0, 1.0, (200, dim)) * box
    kw = dict(max_steps=0, device=device, max_neighbors=200)
    r = PR.minimize_precise(pos, rad, box, skin=0.05, **kw)
    F, e, _ = forces64(r["pos"], rad.astype(np.float32).astype(np.float64), box)
    assert np.abs(r["force"].cpu().numpy() - F).max() <= 1e-6 * 100  # as for the small systems above
    assert np.abs(F[:64]).max() > 0.01 and abs(r["pe"] * 200 - e) <= 1e-5 * e
