"""GPU tests of the operators on particles in no order, at the sizes where
their dispatch or their indexing changes: the tile sort's one-workgroup and
general offset scans, waves that name more tiles than are matched one by one,
the binned deposits on a sorted copy and through the permutation, and the
gathers across the right and upper edges.  Integer results and the FP32 pushes
are compared bit for bit."""
import ctypes as C

import numpy as np
import pytest
import torch

from arcwarden_amd import _lib as L

from gpu_util import Ctx, DevParticles, dev, host, random_particles, stream

pytestmark = pytest.mark.gpu


# ntiles 1, 192 (the counters' groups do not divide the workgroup), 1024 (the
# scan's largest), 1056 (past it), and 1024 tiles x 80 blocks (past its counters)
@pytest.mark.parametrize("nx,ny,t,n", [(16, 16, 16, 1), (16, 16, 16, 70_001),
                                       (256, 192, 16, 63), (256, 192, 16, 300_001),
                                       (256, 256, 8, 65_536), (256, 256, 8, 65_537),
                                       (264, 256, 8, 200_000), (256, 256, 8, 5_200_000)])
def test_tile_bins_any_order(gpu, nx, ny, t, n):
    rng = np.random.default_rng(n + nx)
    x = rng.uniform(0, nx, n).astype(np.float32)
    y = rng.uniform(0, ny, n).astype(np.float32)
    x[x >= nx] = 0
    y[y >= ny] = 0
    # a stretch in tile order: waves of one tile beside waves of sixty
    h = n // 3
    x[:h] = np.sort(x[:h])
    g = L.grid(nx, ny, float(nx), float(ny))
    with Ctx(g, t, t) as ctx:
        z = np.zeros(n, np.float32)
        p = DevParticles({"x": x, "y": y, "ux": z, "uy": z, "uz": z})
        off = torch.full((ctx.ntiles + 1,), -1, dtype=torch.int32, device="cuda")
        idx = torch.full((n,), -1, dtype=torch.int32, device="cuda")
        L.call("aw_bin_tiles", ctx.h, C.byref(p.struct()), C.c_void_p(off.data_ptr()),
               C.c_void_p(idx.data_ptr()), stream())
        key = (np.floor(y).astype(np.int64) // t) * ctx.ntx + np.floor(x).astype(np.int64) // t
        want = np.searchsorted(np.sort(key), np.arange(ctx.ntiles + 1))
        assert np.array_equal(host(off), want)
        assert np.array_equal(host(idx), np.argsort(key, kind="stable"))


def _fields(rng, k, nx, ny):
    return [rng.normal(0, 0.3, (ny, nx)).astype(np.float32) for _ in range(k)]


def _edge_particles(rng, nx, ny, n):
    """Random particles, a third of them in the last column or row."""
    st = random_particles(rng, nx, ny, n)
    st["x"][: n // 6] = (nx - rng.uniform(0.01, 1, n // 6)).astype(np.float32)
    st["y"][n // 6: n // 3] = (ny - rng.uniform(0.01, 1, n // 3 - n // 6)).astype(np.float32)
    return st


@pytest.mark.parametrize("nx,ny,n", [(1, 1, 100), (1, 7, 1000), (2, 3, 1000), (33, 20, 255),
                                     (33, 20, 50_000)])
@pytest.mark.parametrize("back", [False, True])
def test_push_es_edges(gpu, oracle, nx, ny, n, back):
    rng = np.random.default_rng(n + nx + back)
    st = _edge_particles(rng, nx, ny, n)
    E = _fields(rng, 2, nx, ny)
    g = L.grid(nx, ny, 0.5 * nx, 0.5 * ny)
    B0 = (0.2, 0.0, 0.4)
    rp = L.run_params(dt=0.1, qm=-1.0, B0=B0)
    og, pp = oracle.grid(nx, ny, 0.5, 0.5), oracle.push_params(-1.0, 0.1, B0, True)
    ref = (oracle.half_back_f32(og, pp, st, *E) if back  # takes -dt/2 itself
           else oracle.push_es_f32(og, pp, st, *E, False))
    with Ctx(g) as ctx:
        p = DevParticles(st, w_uniform=1.0)
        Ed = [dev(a.ravel()) for a in E]
        L.call("aw_half_step_back" if back else "aw_push_es", ctx.h, C.byref(p.struct()),
               Ed[0].data_ptr(), Ed[1].data_ptr(), C.byref(rp), 1, stream())
        got = p.numpy()
    for k in ("x", "y", "ux", "uy", "uz"):
        assert np.array_equal(got[k], ref[k]), k


@pytest.mark.parametrize("nx,ny,n", [(1, 1, 100), (1, 7, 1000), (2, 3, 1000), (33, 20, 50_000)])
def test_push_boris_em_edges(gpu, oracle, nx, ny, n):
    rng = np.random.default_rng(n + nx)
    st = _edge_particles(rng, nx, ny, n)
    F = _fields(rng, 6, nx, ny)
    g = L.grid(nx, ny, 0.5 * nx, 0.5 * ny)
    rp = L.run_params(dt=0.1, qm=-1.0)
    ref = oracle.push_em_f32(oracle.grid(nx, ny, 0.5, 0.5), -1.0, 0.1, st, F[:3], F[3:])
    with Ctx(g) as ctx:
        p = DevParticles(st, w_uniform=1.0)
        Fd = [dev(a.ravel()) for a in F]
        f = L.AwFields()
        for name, t in zip(("Ex", "Ey", "Ez", "Bx", "By", "Bz"), Fd):
            setattr(f, name, t.data_ptr())
        L.call("aw_push_boris_em", ctx.h, C.byref(p.struct()), C.byref(f), C.byref(rp), stream())
        got = p.numpy()
    for k in ("x", "y", "ux", "uy", "uz"):
        assert np.array_equal(got[k], ref[k]), k


def _binned_deposits(ctx, st, w, x1, y1, Fd, nc):
    """rho, the Darwin moments, dcu and the Esirkepov current, binned."""
    wu = 0.0 if w is not None else 0.25
    p = DevParticles(st, w=w, w_uniform=wu)
    moved = DevParticles({**st, "x": x1, "y": y1}, w=w, w_uniform=wu)
    f = L.AwFields()
    for name, t in zip(("Ex", "Ey", "Ez", "Bx", "By", "Bz"), Fd):
        setattr(f, name, t.data_ptr())
    out = [torch.zeros(nc, dtype=torch.float32, device="cuda") for _ in range(15)]
    src = L.AwSources()
    for name, t in zip(("rho", "Jx", "Jy", "Jz", "amu0", "amu1", "amu2", "amu3", "dcux", "dcuy",
                        "dcuz"), out):
        setattr(src, name, t.data_ptr())
    L.call("aw_deposit_rho_j_amu", ctx.h, C.byref(p.struct()), -1.0, C.byref(src), stream())
    L.call("aw_deposit_dcu", ctx.h, C.byref(p.struct()), -1.0, C.byref(f), C.byref(src), stream())
    L.call("aw_deposit_rho", ctx.h, C.byref(p.struct()), -1.0, L.AW_DEPOSIT_BINNED,
           out[11].data_ptr(), stream())
    L.call("aw_deposit_esirkepov", ctx.h, p.t["x"].data_ptr(), p.t["y"].data_ptr(),
           C.byref(moved.struct()), -1.0, 0.1, L.AW_DEPOSIT_BINNED,
           *(t.data_ptr() for t in out[12:]), stream())
    return [host(t) for t in out]


# tiles of 2x2 on 512x512: 65536, whose counters do not fit LDS, so the
# particles are read through the radix sort's permutation; 16x16: from a copy
# in tile order.  The sums are integers: the same bits.
@pytest.mark.parametrize("per_w", [False, True])
def test_binned_deposits_copy_and_permutation(gpu, per_w):
    nx = ny = 512
    n = 150_003
    rng = np.random.default_rng(17 + per_w)
    st = _edge_particles(rng, nx, ny, n)
    x1 = np.mod(st["x"] + rng.uniform(-0.9, 0.9, n).astype(np.float32), np.float32(nx))
    y1 = np.mod(st["y"] + rng.uniform(-0.9, 0.9, n).astype(np.float32), np.float32(ny))
    x1[x1 >= nx], y1[y1 >= ny] = 0, 0
    w = rng.uniform(0.1, 0.4, n).astype(np.float32) if per_w else None
    g = L.grid(nx, ny, 0.5 * nx, 0.5 * ny)
    Fd = [dev(a.ravel()) for a in _fields(rng, 6, nx, ny)]
    got = []
    for t in (16, 2):
        with Ctx(g, t, t) as ctx:
            assert (ctx.ntiles > 40960) == (t == 2)
            got.append(_binned_deposits(ctx, st, w, x1, y1, Fd, nx * ny))
    for q, (a, b) in enumerate(zip(*got)):
        assert np.abs(a).max() > 0 and np.array_equal(a, b), q
