"""GPU tests of the split current deposit: moves that stay in their cell are
deposited on the spot with the 8 contributions that are not zero, the others
are set aside and take the general stencil (esk_device.hpp).

The tile-ordered Yee step does so.  The unsorted one deposits every move with
the general stencil on a grid of several rows whose current fits LDS: fields
and particles must be the same bits at every share of moves that leave their
cell, on one-column and ragged grids, with uniform and per-particle weights.
On one row the unsorted step splits the moves too (its own kernel): there both
are compared with the FP64 current of the same moves as well."""
import numpy as np
import pytest

from arcwarden_amd import _lib as L
from arcwarden_amd.maxwell import MaxwellSimulation
from arcwarden_amd.sim import SimConfig, Simulation

pytestmark = pytest.mark.gpu


def _run(tile_sort, nx, ny, step, per_w, n, steps=3):
    dx, dt = 0.5, 0.05
    rp = L.run_params(dt=dt, qm=-1.0, eps0=1.0, c=6.0)
    rp.B0[0], rp.B0[2], rp.tile_sort = 0.3, 0.2, tile_sort
    rng = np.random.default_rng(nx * 1000 + ny)
    st = {"x": rng.uniform(0, nx, n).astype(np.float32),
          "y": rng.uniform(0, ny, n).astype(np.float32)}
    # positions on cell edges and denormally close to the origin
    st["x"][:64] = np.floor(st["x"][:64])
    st["y"][32:96] = np.floor(st["y"][32:96])
    st["x"][96:112], st["y"][112:128] = 1e-30, 1e-12
    for k in ("ux", "uy", "uz"):  # at most `step` cells a step
        st[k] = (rng.uniform(-1, 1, n) * step * dx / dt).astype(np.float32)
    sim = MaxwellSimulation(L.grid(nx, ny, nx * dx, ny * dx), rp)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32) * (dx * dx / 16) if per_w else None
    sim.set_particles(st, w=w, **({} if per_w else {"w_uniform": dx * dx / 16}))
    for _ in range(steps):
        sim.step()
    sim.synchronize()
    M, P = sim.mesh_flat(), sim.particles()
    sim.close()
    cols = np.stack([P[k] for k in ("x", "y", "ux", "uy", "uz")])
    return M, cols[:, np.lexsort(cols[::-1])]


@pytest.mark.parametrize("step", [0.0, 0.02, 0.5, 0.98])
@pytest.mark.parametrize("nx,ny,per_w", [(48, 40, False), (33, 17, True), (300, 1, False),
                                         (17, 1, True), (2, 40, False), (1, 24, False)])
def test_split_deposit_matches_the_general_stencil(gpu, nx, ny, per_w, step):
    n = max(5000, 20 * nx * ny) + 37
    M0, P0 = _run(0, nx, ny, step, per_w, n)
    M1, P1 = _run(1, nx, ny, step, per_w, n)
    assert step == 0.0 or np.abs(M0[-3 * nx * ny:]).max() > 0
    assert np.array_equal(M0, M1)
    assert np.array_equal(P0, P1)


@pytest.mark.parametrize("tile_sort", [0, 1])
@pytest.mark.parametrize("step", [0.02, 0.5, 0.98])
@pytest.mark.parametrize("nx,per_w", [(300, False), (17, True), (2, False)])
def test_one_row_split_deposit_matches_fp64(gpu, oracle, nx, per_w, step, tile_sort):
    """One step without fields: the particles keep their velocities, and J is the
    FP64 Esirkepov current of their moves within the FP32 result's rounding."""
    dx, dt, n = 0.5, 0.05, max(4000, 40 * nx) + 11
    rp = L.run_params(dt=dt, qm=-1.0, eps0=1.0, c=6.0)
    rp.tile_sort = tile_sort
    rng = np.random.default_rng(nx)
    st = {"x": rng.uniform(0, nx, n).astype(np.float32),
          "y": rng.uniform(0, 1, n).astype(np.float32)}
    st["x"][st["x"] >= nx], st["y"][st["y"] >= 1] = 0, 0
    st["x"][:64] = np.floor(st["x"][:64])
    for k in ("ux", "uy", "uz"):
        st[k] = (rng.uniform(-1, 1, n) * step * dx / dt).astype(np.float32)
    st["uy"] *= 0.5  # half a cell: further, the periodic image on one row is ambiguous
    w = rng.uniform(0.5, 1.5, n).astype(np.float32) * (dx * dx / 16) if per_w else None
    wu = 0.0 if per_w else dx * dx / 16
    sim = MaxwellSimulation(L.grid(nx, 1, nx * dx, dx), rp)
    sim.set_particles(st, w=w, **({} if per_w else {"w_uniform": wu}))
    sim.step()
    sim.synchronize()
    J = sim.mesh_flat()[6 * nx:].reshape(3, 1, nx)
    sim.close()
    og = oracle.grid(nx, 1, dx, dx)
    x1 = st["x"] + (st["ux"].astype(np.float64) * dt / dx).astype(np.float32)
    y1 = st["y"] + (st["uy"].astype(np.float64) * dt / dx).astype(np.float32)
    ref = oracle.esirkepov_f64(og, st["x"], st["y"], x1, y1, st["uz"], -1.0, dt, w=w,
                               w_uniform=wu)
    for q in range(3):
        assert np.linalg.norm(J[q] - ref[q]) < 1e-6 * np.linalg.norm(ref[q]), q


@pytest.mark.parametrize("step", [0.01, 0.4, 0.9])
@pytest.mark.parametrize("nx,ny,tile", [(48, 40, 16), (33, 17, 16), (40, 24, 8), (64, 1, 16)])
def test_darwin_split_deposit_matches_fp64(gpu, oracle, nx, ny, tile, step):
    """The Esirkepov current of the Darwin push, with from a few to nearly all
    of the moves leaving their cell (the queue then drains every iteration),
    against the FP64 restatement of the same moves: quanta of 2^-48 of the
    largest contribution, FP32 result (6e-8), so 1e-6 of the norm."""
    dx, c = 0.5, 6.0
    dt = 0.05
    v = step * dx / dt
    rp = L.run_params(dt=dt, qm=-1.0, eps0=1.0, c=max(c, v), n0=1.0, noisy_load=1, rng_seed=5,
                      B0=(0.1, 0.0, 0.2), wce=0.2, dump_every=100)
    # up to about 0.9 step cells: a move of a cell or more is outside the stencil
    sp = [L.species("a", 0.5, 12, (0.08 * v,) * 3, (0.5 * v, 0.3 * v, 0)),
          L.species("b", 0.5, 12, (0.08 * v,) * 3, (-0.5 * v, 0, 0.2 * v))]
    sim = Simulation(L.grid(nx, ny, nx * dx, ny * dx), rp, sp,
                     SimConfig(field_model=L.AW_MODEL_DARWIN,
                               current_deposit=L.AW_CURRENT_ESIRKEPOV, tile_x=tile, tile_y=tile,
                               sort_every=0, stray_frac=1.0))
    sim.init()
    s0 = sim.particles()
    sim.step(0)
    s1 = sim.particles()
    sim.step(1)
    srcs = sim.sources_all()
    sim.close()
    og = oracle.grid(nx, ny, dx, dx)
    ref = oracle.esirkepov_f64(og, s0["x"], s0["y"], s1["x"], s1["y"], s1["uz"], -1.0, dt,
                               w_uniform=s0["w_uniform"])
    for name, r in zip(("Jx", "Jy", "Jz"), ref):
        assert np.linalg.norm(srcs[name] - r) < 1e-6 * np.linalg.norm(r), name


@pytest.mark.parametrize("tile_x,tile_y", [(30, 48), (41, 35), (25, 57)])
def test_darwin_push_on_the_largest_tiles(gpu, tile_x, tile_y):
    """Tiles whose moments and fields leave LDS for one to six slots of the move
    queue a wavefront, and whose push also keeps 32 bytes for the kinetic energy
    of a diagnostics step: the same bits as on 16x16 tiles."""
    nx, ny, dx = 2 * tile_x, 2 * tile_y, 0.5
    rp = L.run_params(dt=0.05, qm=-1.0, eps0=1.0, c=8.0, n0=1.0, noisy_load=1, rng_seed=3,
                      B0=(0.1, 0.0, 0.2), wce=0.2, dump_every=1)
    sp = [L.species("a", 1.0, 10, (0.5,) * 3, (4.0, -2.0, 0.5))]  # 0.4 cells a step
    out = []
    for tx, ty in ((16, 16), (tile_x, tile_y)):
        sim = Simulation(L.grid(nx, ny, nx * dx, ny * dx), rp, sp,
                         SimConfig(field_model=L.AW_MODEL_DARWIN,
                                   current_deposit=L.AW_CURRENT_ESIRKEPOV, tile_x=tx, tile_y=ty,
                                   sort_every=0, stray_frac=1.0))
        sim.init()
        for n in range(3):
            sim.step(n)
        srcs, P, hist = sim.sources_all(), sim.particles(), sim.history()
        sim.close()
        cols = np.stack([P[k] for k in ("x", "y", "ux", "uy", "uz")])
        out.append((srcs, cols[:, np.lexsort(cols[::-1])], [h["ke"] for h in hist]))
    (s0, p0, k0), (s1, p1, k1) = out
    assert np.array_equal(p0, p1)
    for name in s0:
        assert np.array_equal(s0[name], s1[name]), name
    assert len(k0) == 3 and np.allclose(k0, k1, rtol=1e-12, atol=0)  # FP64 sums, another order
