"""GPU tests of the spectral solves on the library's own transforms (fft.hip):
E of rho, E_L and B of [rho|J], E_T of [dcu|amu] against the same algebra on
numpy's FP64 transforms, over sides of every factor the transforms have a pass
for (5, 4, 3, 2, other primes to 61), odd, prime and one-row grids, the
longest line, and sides of which one kind of solve or both stay with rocFFT.

The library's transforms are FP64 between three FP32 roundings of every value
(the two half spectra and the result), 2^-24 at most and independent: below
3 * 2^-24 = 1.8e-7 of the result's norm, doubled for the fields' own spread.
rocFFT's are FP32 throughout (5e-6)."""
import ctypes as C

import numpy as np
import pytest
import torch

from arcwarden_amd import _lib as L

pytestmark = pytest.mark.gpu

# on the library's own transforms
OWN = [(64, 64), (128, 96), (250, 190), (33, 17), (61, 59), (7, 121), (243, 125), (16, 1),
       (1000, 1), (3125, 1), (2, 2), (3, 5), (1, 24), (512, 96), (40, 600), (625, 625)]
# the electrostatic solve only, and the Darwin ones only
OWN_ES = [(64, 512), (2500, 360), (1200, 360), (3000, 110)]
OWN_EM = [(1024, 64), (512, 128), (1250, 128), (3000, 100)]
# rocFFT: a prime above 61, a line longer than LDS, one that leaves no LDS for
# what else its kernels hold (3150: 163,808 of 163,840 bytes), and the sides where
# rocFFT is ahead
ROCFFT = [(67, 40), (40, 134), (3001, 1), (4096, 1), (3150, 62), (3150, 110), (512, 512),
          (2048, 1), (3599, 1)]


def _kvec(nx, ny, dx, dy):
    i = np.arange(nx // 2 + 1)
    j = np.arange(ny)
    j = np.where(j <= ny // 2, j, j - ny)
    kx = (2 * np.pi / (nx * dx)) * i[None, :] + 0.0 * j[:, None]
    ky = (2 * np.pi / (ny * dy)) * j[:, None] + 0.0 * i[None, :]
    nyq = np.zeros(kx.shape, bool)
    if nx % 2 == 0:
        nyq[:, nx // 2] = True
    if ny % 2 == 0:
        nyq[ny // 2, :] = True
    return kx, ky, nyq, i[None, :], j[:, None]


def _inverse(spec, nx, ny):
    return np.stack([np.fft.irfft2(s, s=(ny, nx)) for s in spec])


def _check(got, ref, tol):
    """Each grid against the largest one's norm: a grid that cancels to nothing
    keeps the rounding of what it cancelled."""
    top = max(np.linalg.norm(r) for r in ref)
    for g, r in zip(got, ref):
        err = np.linalg.norm(g - r) / max(np.linalg.norm(r), 1e-3 * top, 1e-30)
        assert err < tol, err


@pytest.fixture
def solver(gpu):
    made = []

    def make(nx, ny, dx, dy):
        g = L.grid(nx, ny, nx * dx, ny * dy)
        h = C.c_void_p()
        L.call("aw_ctx_create", C.byref(g), 0, 0, C.byref(h))
        made.append(h)
        return h

    yield make
    torch.cuda.synchronize()
    for h in made:
        L.lib().aw_ctx_destroy(h)


@pytest.mark.parametrize("nx,ny", OWN + OWN_ES + OWN_EM + ROCFFT)
def test_solves_match_fp64(solver, nx, ny):
    dx, dy, eps0, c, n0 = 0.5, 0.4, 1.3, 7.0, 0.9
    ctx = solver(nx, ny, dx, dy)
    rng = np.random.default_rng(nx * 7919 + ny)
    src = rng.normal(size=(11, ny, nx)).astype(np.float32)
    d = torch.from_numpy(src).cuda()
    e = torch.zeros(2, ny, nx, device="cuda")
    elb = torch.zeros(5, ny, nx, device="cuda")
    elbs = torch.zeros(5, ny, nx, device="cuda")
    et = torch.zeros(3, ny, nx, device="cuda")
    torch.cuda.synchronize()
    b0 = (C.c_float * 3)(0.3, -0.2, 0.1)
    L.call("aw_solve_es", ctx, d[0].data_ptr(), e[0].data_ptr(), e[1].data_ptr(), eps0, None)
    L.call("aw_solve_darwin_el_b", ctx, d.data_ptr(), elb.data_ptr(), eps0, c, b0, None)
    L.call("aw_solve_darwin_el_b_ex", ctx, d.data_ptr(), elbs.data_ptr(), eps0, c, b0, 1, None)
    L.call("aw_solve_darwin_et", ctx, d[4].data_ptr(), et.data_ptr(), eps0, c, n0, None)
    torch.cuda.synchronize()
    assert np.array_equal(d.cpu().numpy(), src)  # the inputs stay as they are

    tol_es = 3.6e-7 if (nx, ny) in OWN + OWN_ES else 5e-6
    tol = 3.6e-7 if (nx, ny) in OWN + OWN_EM else 5e-6
    kx, ky, nyq, i, j = _kvec(nx, ny, dx, dy)
    k2 = kx ** 2 + ky ** 2
    on = (k2 > 0) & ~nyq
    safe = np.where(on, k2, 1.0)
    s = np.fft.rfft2(src.astype(np.float64))
    E = [np.where(on, -1j * k * s[0] / (eps0 * safe), 0) for k in (kx, ky)]
    _check(e.cpu().numpy(), _inverse(E, nx, ny), tol_es)
    for got, stag in ((elb, False), (elbs, True)):
        jx, jy, jz = s[1], s[2], s[3]
        if stag:
            jx, jy = jx * np.exp(-1j * np.pi * i / nx), jy * np.exp(-1j * np.pi * j / ny)
        G = np.where(on, 1.0 / (eps0 * c * c * safe), 0)
        B = [1j * G * ky * jz, -1j * G * kx * jz, 1j * G * (kx * jy - ky * jx)]
        for q in range(3):
            B[q][0, 0] = float(b0[q]) * nx * ny
        _check(got.cpu().numpy(), _inverse(E + B, nx, ny), tol)
    a0, a1, a2, a3 = s[7:]
    J = [s[4] - 1j * (kx * a0 + ky * a1), s[5] - 1j * (kx * a1 - ky * a0),
         s[6] - 1j * (kx * a2 + ky * a3)]
    kd = (kx * J[0] + ky * J[1]) / safe
    J[0], J[1] = J[0] - kx * kd, J[1] - ky * kd
    G = np.where(on, 1.0 / (eps0 * c * c * safe + n0), 0)
    _check(et.cpu().numpy(), _inverse([-G * v for v in J], nx, ny), tol)


@pytest.mark.parametrize("nx,ny", [(96, 50), (33, 17), (67, 40)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_values_that_are_not_finite_stay_in_their_fields(solver, nx, ny, bad):
    """Two grids share a line of the transforms, but only the fields that depend
    on a grid lose their values with it (the last side is rocFFT's)."""
    ctx = solver(nx, ny, 0.5, 0.4)
    src = np.random.default_rng(nx).normal(size=(11, ny, nx)).astype(np.float32)
    b0 = (C.c_float * 3)(0.3, -0.2, 0.1)

    def fields(at=None):
        d = torch.from_numpy(src).cuda()
        if at is not None:
            d[at, ny // 2, nx // 3] = bad
        elb, et = torch.zeros(5, ny, nx, device="cuda"), torch.zeros(3, ny, nx, device="cuda")
        L.call("aw_solve_darwin_el_b", ctx, d.data_ptr(), elb.data_ptr(), 1.0, 7.0, b0, None)
        L.call("aw_solve_darwin_et", ctx, d[4].data_ptr(), et.data_ptr(), 1.0, 7.0, 0.9, None)
        torch.cuda.synchronize()
        return torch.cat([elb, et]).cpu().numpy()

    clean = fields()
    # grid -> the fields made of it: ELx ELy Bx By Bz ETx ETy ETz
    for at, of in {1: (4,), 2: (4,), 3: (2, 3), 6: (7,), 7: (5, 6), 10: (7,)}.items():
        got = fields(at)
        for q in range(8):
            if q in of:
                assert not np.isfinite(got[q]).any(), (at, q)
            else:
                err = np.linalg.norm(got[q] - clean[q]) / np.linalg.norm(clean[q])
                assert err < 1e-6, (at, q, err)


def test_darwin_solves_captured_after_the_first(solver):
    """Once one Darwin solve has run, a graph captures both (nothing is left to
    allocate); every replay equals the eager result of the same inputs."""
    nx, ny = 96, 50
    ctx = solver(nx, ny, 0.5, 0.4)
    rng = np.random.default_rng(5)
    d = torch.zeros(11, ny, nx, device="cuda")
    elb, et = torch.zeros(5, ny, nx, device="cuda"), torch.zeros(3, ny, nx, device="cuda")
    b0 = (C.c_float * 3)(0.3, -0.2, 0.1)

    def el_b(out):
        L.call("aw_solve_darwin_el_b", ctx, d.data_ptr(), out.data_ptr(), 1.0, 7.0, b0,
               C.c_void_p(torch.cuda.current_stream().cuda_stream))

    def e_t(out):
        L.call("aw_solve_darwin_et", ctx, d[4].data_ptr(), out.data_ptr(), 1.0, 7.0, 0.9,
               C.c_void_p(torch.cuda.current_stream().cuda_stream))

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        el_b(elb)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        el_b(elb)
        e_t(et)
    for _ in range(3):
        d.copy_(torch.from_numpy(rng.normal(size=(11, ny, nx)).astype(np.float32)))
        ref_b, ref_t = torch.zeros_like(elb), torch.zeros_like(et)
        el_b(ref_b)
        e_t(ref_t)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(elb, ref_b) and torch.equal(et, ref_t)
        assert float(et.abs().max()) > 0
